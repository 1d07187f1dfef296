// The wide traversal of gpugi_amd/csrc/device/trace_wide.h run on the CPU, one
// ray at a time (a wave of one lane), over the tree BuildWideBVH makes.  The
// device functions are compiled as they stand; only the few GPU built-ins they
// use are supplied here.  Built and driven by tests/test_wide_walk_cpu.py.
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

static inline uint32_t __float_as_uint(float f) { uint32_t u; std::memcpy(&u, &f, 4); return u; }
static inline float __uint_as_float(uint32_t u) { float f; std::memcpy(&f, &u, 4); return f; }
static inline int __float_as_int(float f) { return (int)__float_as_uint(f); }
static inline float __int_as_float(int i) { return __uint_as_float((uint32_t)i); }
static inline int __popc(uint32_t x) { return __builtin_popcount(x); }
static inline int __popcll(uint64_t x) { return __builtin_popcountll(x); }
static inline uint64_t __ballot(bool b) { return b ? 1u : 0u; }
static inline uint32_t atomicOr(uint32_t* p, uint32_t v) { const uint32_t o = *p; *p |= v; return o; }
static inline float amd_rcp(float x) { return 1.0f / x; }
static uint32_t slots_tested;  // the walk shifts in one bit per child box
static inline uint32_t amd_alignbit(uint32_t hi, uint32_t lo, uint32_t n) {
  ++slots_tested;
  return (uint32_t)((((uint64_t)hi << 32) | lo) >> (n & 31u));
}
// bytes 0-3 of a selector byte are lo's, 4-7 hi's, 0x0c is zero
static inline uint32_t amd_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  const uint64_t w = ((uint64_t)hi << 32) | lo;
  uint32_t r = 0;
  for (int i = 0; i < 4; ++i) {
    const uint32_t c = (sel >> (8 * i)) & 0xffu;
    r |= (c == 0x0cu ? 0u : (uint32_t)(w >> (8 * c)) & 0xffu) << (8 * i);
  }
  return r;
}
#define __builtin_amdgcn_perm amd_perm
#define __builtin_amdgcn_rcpf amd_rcp
#define __builtin_amdgcn_alignbit amd_alignbit
using std::max;
using std::min;

#define __HIPCC__ 1  // wide_bvh.h declares the device view with it
#include "device/trace_wide.h"
#include "device/wide_bvh.h"

using namespace gpugi;

namespace {
constexpr int kLanes = 3;  // LDS stack of three lanes; the ray runs on lane 1

template <bool ANY, int S, bool WT>
void Trace(const WideScene& s, const float* rays, int32_t* hits, size_t n, std::vector<uint2>* lds,
           std::vector<uint2>* spill) {
  for (size_t i = 0; i < n; ++i) {
    const float* r = rays + 8 * i;
    const WideResult w = trace_wide_ray<ANY, kLanes, S, WT>(s, gg::v3(r[0], r[1], r[2]), gg::v3(r[4], r[5], r[6]), r[3],
                                                            lds->data(), 1, spill->data());
    int32_t* h = hits + 4 * i;
    h[0] = ANY ? (w.any ? 1 : 0) : w.slot;
    h[1] = __float_as_int(w.t);
    h[2] = __float_as_int(w.by);
    h[3] = __float_as_int(w.bz);
  }
}

template <int S>
void TraceS(bool any, bool wt, const WideScene& s, const float* rays, int32_t* hits, size_t n, std::vector<uint2>* lds,
            std::vector<uint2>* spill) {
  if (any && wt) Trace<true, S, true>(s, rays, hits, n, lds, spill);
  else if (any) Trace<true, S, false>(s, rays, hits, n, lds, spill);
  else if (wt) Trace<false, S, true>(s, rays, hits, n, lds, spill);
  else Trace<false, S, false>(s, rays, hits, n, lds, spill);
}
}  // namespace

// Traces n rays (8 floats each) into hits (4 words each).  counts: {nodes, triangles,
// max stack entries, entries the deepest ray used, overflow flag, nodes visited}.
// ldsEntries: 1 or 10.  Returns 0, or 1 if the tree could not be built.
extern "C" int wide_walk(const gpugi_scene_desc* d, uint32_t leaf, int any, int wt, int ldsEntries, const float* rays,
                         int32_t* hits, size_t n, uint32_t counts[6]) {
  WideBVHHost b;
  if (!BuildWideBVH(*d, leaf, &b, wt != 0).empty()) return 1;
  uint32_t flag = 0;
  WideScene s{};
  s.nodes = (const uint4*)b.nodes.data();
  s.tris = (const float4*)b.tris.data();
  s.spillDepth = b.maxStack > (uint32_t)ldsEntries ? b.maxStack - (uint32_t)ldsEntries : 0;
  s.errorFlag = &flag;
  SetWideScale(&s, b.tScale);
  std::vector<uint2> lds((size_t)ldsEntries * kLanes, uint2{0xdeadu, 0xdeadu});
  std::vector<uint2> spill(s.spillDepth, uint2{0xdeadu, 0xdeadu});
  slots_tested = 0;
  if (ldsEntries == 1) TraceS<1>(any != 0, wt != 0, s, rays, hits, n, &lds, &spill);
  else TraceS<10>(any != 0, wt != 0, s, rays, hits, n, &lds, &spill);
  counts[0] = (uint32_t)b.nodes.size();
  counts[1] = (uint32_t)b.tris.size();
  counts[2] = b.maxStack;
  counts[3] = 0;
  for (int e = 0; e < ldsEntries; ++e) counts[3] += lds[(size_t)e * kLanes + 1].x != 0xdeadu;
  for (const uint2& e : spill) counts[3] += e.x != 0xdeadu;
  counts[4] = flag;
  counts[5] = slots_tested / kWideArity;
  return 0;
}
