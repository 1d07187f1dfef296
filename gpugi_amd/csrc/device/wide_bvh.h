// Re-packed 8-wide BVH with 8-bit quantized child boxes (host layout + device view).
//
// Node: 80 bytes, read as five 16-byte loads:
//   q0 = {origin.x, origin.y, origin.z, exps}   exps = ex | ey<<8 | ez<<16 | inner<<24,
//                                              scale_a = 2^(e_a - 127)
//   q1 = {firstChild, firstTri, ends[0..7]}     ends: one byte per child
//   q2 = {lo.x[8], lo.y[8]}, q3 = {lo.z[8], hi.x[8]}, q4 = {hi.y[8], hi.z[8]}
// A child sits in one of eight slots.  Bit k of `inner` marks slot k as an inner
// node; the inner children are consecutive nodes from firstChild in slot order.
// Any other slot is a leaf whose triangles are firstTri + [ends[k-1], ends[k])
// (ends[-1] = 0), which is empty for an unused slot; an unused slot also has
// the inverted box lo = 255, hi = 0.  Slots are in the order of the child boxes'
// surface, smallest first.  (Compressed eight-wide nodes: Ylitie, Karras and
// Laine 2017, "Efficient incoherent ray traversal on GPUs through compressed
// wide BVHs".)
// child box along axis a = [origin_a + lo*scale_a, origin_a + hi*scale_a]; the
// host rounds lo down and hi up and checks in extended precision that the
// exact origin + q * scale encloses the child box, so the quantized tree is conservative.
// Triangle: 48 bytes {p0, slot}, {e0 = p1-p0, material}, {e1 = p0-p2, 0}: the
// operands of the reference triangle test, computed once in FP32 (in
// watertight mode the raw vertices {p0, slot}, {p1, material}, {p2, 0}).
#pragma once
#include <stdint.h>

#include <string>
#include <vector>

#include "gpugi_rt.h"

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#endif

namespace gpugi {

constexpr int kWideArity = 8;
constexpr uint32_t kWideNodeBytes = 80;
constexpr uint32_t kWideMaxTris = 1u << 27;
constexpr uint32_t kWideMaxNodes = 1u << 25;  // node offsets stay below 2^32 bytes
constexpr uint32_t kWideMaxLeafTris = 16;     // ends[7] <= 8 * 16 fits its byte

struct WideNodeHost {
  float origin[3];
  uint32_t exps;
  uint32_t firstChild, firstTri;
  uint8_t ends[kWideArity];
  uint8_t lo[3][kWideArity];
  uint8_t hi[3][kWideArity];
};
static_assert(sizeof(WideNodeHost) == kWideNodeBytes, "wide node is 80 bytes");

struct WideTriHost {
  float p0[3];
  int32_t slot;
  float e0[3];
  int32_t material;
  float e1[3];
  int32_t pad;
};
static_assert(sizeof(WideTriHost) == 48, "wide triangle is 48 bytes");

struct WideBVHHost {
  std::vector<WideNodeHost> nodes;
  std::vector<WideTriHost> tris;
  uint32_t maxStack = 0;  // most traversal stack entries of a ray (one holds the waiting children of a node)
  uint32_t depth = 0;
  // Slab distances are computed times this power of two: 1, or less where a node's quantum exceeds 2^36
  // (wide_visit multiplies by up to 2^24 / 1e-20 * quantum, which has to stay finite).
  float tScale = 1.0f;
  // Triangles that a random line through the root's box meets on average: twice their
  // area over the box's (Cauchy), so 2 and more for a closed room, 0.9 for a terrain.
  float crossings = 0.0f;
};
constexpr int kWideQuantumLog2 = 36;

// Re-packs the reference BVH2 (any arity up to 8 written in preorder with escape
// pointers) into the 8-wide quantized layout.  Leaves of up to
// `maxLeafTris` triangles are formed from subtrees that small.  rawVertices:
// triangles store {p0, slot}{p1, mat}{p2, 0} (watertight test) instead of the
// reference test's operands {p0, slot}{p1 - p0, mat}{p0 - p2, 0}.
std::string BuildWideBVH(const gpugi_scene_desc& desc, uint32_t maxLeafTris, WideBVHHost* out,
                         bool rawVertices = false);

// Launch shape of the wide kernel: threads per block and LDS stack entries per thread.
constexpr int kWideBlock = 256;
constexpr int kWideLdsStack = 16;

#if defined(__HIPCC__)
struct WideScene {
  const uint4* __restrict__ nodes;    // 5 x uint4 per node
  const float4* __restrict__ tris;    // 3 x float4 per triangle
  uint2* spill;                       // per-thread overflow stack (global memory)
  uint32_t spillDepth;                // entries per thread in `spill`
  uint32_t numThreads;                // persistent threads the spill buffer is sized for
  uint32_t* errorFlag;                // set to nonzero if a stack would overflow
  uint32_t* queue;                    // kWideQueueWords: the trace kernel's per-XCD batch counters
  float tScale;                       // WideBVHHost::tScale
  float hitScale;                     // tScale * (1 + 2^-20): scales and widens the hit distance
};
inline void SetWideScale(WideScene* s, float tScale) {
  s->tScale = tScale;
  s->hitScale = tScale * 1.00000095f;
}
constexpr int kWideQueueStride = 32;  // counters 128 bytes apart
constexpr int kWideQueueWords = 8 * kWideQueueStride;
#endif

}  // namespace gpugi
