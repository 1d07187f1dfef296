// Ordered traversal of the 8-wide quantized BVH (wide_bvh.h), one ray per lane.
//
// A ray's state holds the next inner node to visit, up to two pending leaf
// groups and a stack.  Work comes in two kinds of wave-wide passes:
//   box pass   every lane with a node visits it: eight child box tests; the
//              nearest hit child, if inner, becomes the next node, the other hit
//              inner children wait together in one stack entry; the hit leaves
//              take a free pending slot, as one group;
//   leaf pass  every lane with pending leaves tests the triangles of one.
// A lane with a pending leaf keeps traversing (speculative traversal,
// Aila and Laine 2009, "Understanding the efficiency of ray traversal on
// GPUs"), so a wave runs a leaf pass only once enough lanes wait for one and
// does not pay a divergent triangle loop on every node visit.  The caller
// chooses the pass from two ballots (wide_choose_leaf_pass).  Lanes left
// without a node pop: entries whose children all lie beyond the current hit are
// dropped, a leaf entry fills a free pending slot, a node entry gives its next
// child and stays until it is empty.
// The result does not depend on the order of the work: the closest hit is the
// minimum distance, ties resolved to the smaller reference slot index (the
// triangle the reference's preorder walk meets first).
//
// A stack entry is 8 bytes:
//   nodes   {firstChild of the parent, waiting | inner << 8 | next << 16 | bound}
//   leaves  {parent | kWideLeafEntry, waiting | bound}
// waiting: one bit per slot; next: the slot of the nearest child that waits (the
// others follow in slot order, smallest box first); bound: the 13 high bits of a
// float, a lower bound of the waiting children's entry distances.  An any-hit
// query takes the largest box first, which is the likeliest to hold an occluder,
// and keeps no distances: next and bound are 0.
// Per lane, the first S entries live in LDS laid out
// [depth][thread], so lanes at different depths touch different banks; deeper
// entries spill to global memory (WideStack), sized by the host from the exact
// worst case of the tree.
//
// Box tests use the quantized boxes the host made conservative, slab distances
// computed with one fma per plane and a slack that covers their rounding (see
// wide_visit), and axis-parallel direction components replaced by +-1e-20 so
// that 0 * inf never occurs: a box that contains the closest hit is never
// rejected.  The triangle test is the reference formula
// (intersectiontests.glsl:63-79) or, in watertight mode, the watertight test.
#pragma once
#include <hip/hip_runtime.h>

#include "../common/gvec.h"
#include "trace_ref.h"
#include "wide_bvh.h"

namespace gpugi {

constexpr uint32_t kWideNoNode = 0xffffffffu;
constexpr uint32_t kWideLeafEntry = 0x80000000u;
constexpr uint32_t kWideBoundMask = 0xfff80000u;

// What the lanes of a wave trace: closest hits, any hits, or either, by WideState::anyHit.
enum WideQuery { kWideClosest = 0, kWideAny = 1, kWideMixed = 2 };

struct WideResult {
  float t;     // final ray length (tmax on a miss)
  int slot;    // reference slot index, -1 on a miss, -2 on stack overflow
  float by, bz;
  bool any;    // any-hit result
};

// A lane's traversal stack: entry i < S at
// LDS lds[i * B + tid], deeper entries at spill[(i - S) * spillStride]
// (spillStride = number of threads sharing the spill buffer when it is laid out
// [depth][thread], so a wave's spills at one depth are contiguous; 1 for a
// per-thread slice).
// The LDS part is typed as LDS memory, so its accesses stay ds_* instructions
// and are never merged with the spill's global accesses into flat ones.
// (The host pass of the compiler sees the device code too and has no LDS.)
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) uint2 LdsEntry;
#else
typedef uint2 LdsEntry;
#endif
__device__ __forceinline__ LdsEntry* as_lds(uint2* p) { return (LdsEntry*)p; }

struct WideStack {
  LdsEntry* lds;
  int tid;
  uint2* spill;
  uint32_t spillStride;
};


struct WideState {
  gg::V3 o, d;
  float ix, iy, iz;  // 1/d times WideScene::tScale, so slab and entry distances are scaled, tbest is not
  float tbest;
  int bestSlot;
  float bu, bv;
  uint32_t node;  // next inner node to visit, kWideNoNode if none
  uint32_t leafNode[2];  // the pending leaf groups' nodes
  uint32_t leafMask;     // their hit leaves' slots, 8 bits each; 0: none, below 256: the first only
  int sp;
  bool found;   // kWideAny only
  bool anyHit;  // kWideMixed only; such a ray has found an occluder once bestSlot >= 0
  WtRay wr;     // watertight mode only
};

// 1/d by v_rcp_f32 (within 1 ulp): a reciprocal with relative error
// below 2^-23 scales every slab distance of a ray by the same factor (1 + δ),
// which the far-distance and hit-distance widening of 1 + 2^-20 covers.
__device__ __forceinline__ float safe_inv(float d) {
  return __builtin_amdgcn_rcpf(copysignf(fmaxf(fabsf(d), 1e-20f), d));  // (NaN: 1e-20)
}

// Two quantized planes as 16-bit integers: bytes i and i + 1 of `lo` or of `hi`,
// i = 0 or 2; which word is in the selector (kPlaneLo, kPlaneHi for i = 0).
constexpr uint32_t kPlaneLo = 0x0c010c00u, kPlaneHi = 0x0c050c04u, kPlaneOther = kPlaneLo ^ kPlaneHi;
constexpr uint32_t kPlaneNextPair = 0x00020002u;
__device__ __forceinline__ uint32_t plane_pair(uint32_t lo, uint32_t hi, uint32_t selector) {
  return __builtin_amdgcn_perm(hi, lo, selector);
}

// q * A + b for the low (half 0) or high plane q of a pair, A24 = A * 2^24: a byte
// read as a binary16 is exactly q * 2^-24 (a subnormal), which the mixed-precision
// fma takes as it is, so no conversion instruction is needed.
__device__ __forceinline__ float plane_fma(uint32_t pair, int half, float A24, float b) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef _Float16 Half2 __attribute__((ext_vector_type(2)));
  return __builtin_fmaf((float)__builtin_bit_cast(Half2, pair)[half], A24, b);
#else
  return __builtin_fmaf((float)((pair >> (16 * half)) & 0xffffu) * 5.9604644775390625e-8f, A24, b);
#endif
}

__device__ __forceinline__ bool finite(float x) { return fabsf(x) < INFINITY; }

template <bool WT = false>
__device__ __forceinline__ void wide_init(const WideScene& s, WideState& st, gg::V3 o, gg::V3 d, float tmax) {
  st.o = o;
  st.d = d;
  st.ix = safe_inv(d.x) * s.tScale;
  st.iy = safe_inv(d.y) * s.tScale;
  st.iz = safe_inv(d.z) * s.tScale;
  st.tbest = tmax;
  st.bestSlot = -1;
  st.bu = st.bv = 0.0f;
  st.node = 0;
  st.leafNode[0] = st.leafNode[1] = 0;
  st.leafMask = 0;
  st.sp = 0;
  st.found = false;
  if (WT) st.wr = wt_setup(d);
  // A ray without a finite origin component, or with a NaN for its length, hits nothing,
  // but minima and maxima drop the NaNs of its slab distances: they would let every box
  // through.  Here the scene lies behind it, so that its walk ends at the root.
  // (Selects: with a branch the compiler computes the box pass's plane selectors after
  // the node's loads have come instead of before, 3 % for small launches.)
  const bool dead = !(finite(o.x) || finite(o.y) || finite(o.z)) || tmax != tmax;
  st.o.x = dead ? 1e38f : o.x;
  st.ix = dead ? s.tScale : st.ix;
}

// The node in slot `slot` of the node whose inner children (mask `inner`) start at `first`.
__device__ __forceinline__ uint32_t wide_child(uint32_t first, uint32_t inner, uint32_t slot) {
  return first + (uint32_t)__popc(inner & ((1u << slot) - 1u));
}

// Which of the waiting slots (not 0) is visited next: the nearest one if it waits
// (if it is not a leaf or gone already), else the first; any hit: the last.
template <int Q>
__device__ __forceinline__ uint32_t wide_next(const WideState& st, uint32_t waiting, uint32_t nearest) {
  const uint32_t last = 31u - (uint32_t)__builtin_clz(waiting);
  if (Q == kWideAny) return last;
  const uint32_t closest = (waiting >> nearest) & 1u ? nearest : (uint32_t)__builtin_ctz(waiting);
  return Q == kWideMixed && st.anyHit ? last : closest;
}

// Puts an entry on the stack; false if it would overflow (impossible when the
// host sized the spill from the tree).
template <int B, int S>
__device__ __forceinline__ bool wide_push(const WideScene& s, WideState& st, const WideStack& stk, uint2 e) {
  if (st.sp < S) stk.lds[st.sp * B + stk.tid] = e;
  else if ((uint32_t)(st.sp - S) < s.spillDepth) stk.spill[(size_t)(st.sp - S) * stk.spillStride] = e;
  else return false;
  ++st.sp;
  return true;
}

// Takes a leaf group (leaves != 0) into a free pending slot; false if both are taken.
__device__ __forceinline__ bool wide_hold(WideState& st, uint32_t node, uint32_t leaves) {
  if (st.leafMask > 0xffu) return false;
  const bool empty = st.leafMask == 0u;
  st.leafNode[0] = empty ? node : st.leafNode[0];
  st.leafNode[1] = empty ? st.leafNode[1] : node;
  st.leafMask |= empty ? leaves : leaves << 8;
  return true;
}

// Box pass for a lane with st.node != kWideNoNode.  Returns false if the stack
// would overflow.
template <int Q, int B, int S>
__device__ __forceinline__ bool wide_visit(const WideScene& s, WideState& st, const WideStack& stk) {
  const gg::V3 o = st.o;
  const uint32_t nodeIndex = st.node;
  // (n << 6) + (n << 4) is 80 n, below 2^32 for kWideMaxNodes
  const uint4* n = (const uint4*)((const char*)s.nodes + ((nodeIndex << 6) + (nodeIndex << 4)));
  const uint4 q0 = n[0], q1 = n[1], q2 = n[2], q3 = n[3], q4 = n[4];
  const float ox = __uint_as_float(q0.x), oy = __uint_as_float(q0.y), oz = __uint_as_float(q0.z);
  const float sx = __uint_as_float((q0.w & 0xffu) << 23);
  const float sy = __uint_as_float(((q0.w >> 8) & 0xffu) << 23);
  const float sz = __uint_as_float(((q0.w >> 16) & 0xffu) << 23);
  // Slab distances straight from the quantized bytes: along axis a,
  //   t(q) = (origin_a + q * s_a - o_a) / d_a ~ q * A_a + B_a,
  //   A_a = s_a * inv_a (exact: s_a is a power of two),  B_a = (origin_a - o_a) * inv_a.
  // With inv_a = (1/d_a)(1 + δ_a), |δ_a| <= 2^-23 (safe_inv), the exact distances
  // along an axis are scaled by 1 + δ_a.  Near distances use B_a - |B_a| * 2^-21,
  // which covers the two roundings of B_a.  Far ones use
  // B_a + |B_a| * 2^-20 + |A_a| * 2^-12: along every ray into a box, t is at most
  // |B_a| + 255 |A_a| for each far plane, so this covers the axes' different δ_a
  // (2^-22 t), the roundings of B_a (2^-23 |B_a|) and those of both fmas (2^-24 t
  // each).  (inv_a, so every distance here, is times s.tScale, a power of two that is 1
  // but for scenes whose A_a * 2^24 could overflow.)  The bytes giving the near planes
  // (lo or hi) are picked per axis by the sign of inv_a.  The host checks in extended
  // precision that origin + q * s encloses every child box, so with the hit distance
  // widened by 1 + 2^-20 a box that holds the closest hit is never rejected (the
  // argument of Ize 2013, "Robust BVH ray traversal").
  const float Ax = sx * st.ix, Ay = sy * st.iy, Az = sz * st.iz;
  const float Bx = (ox - o.x) * st.ix, By = (oy - o.y) * st.iy, Bz = (oz - o.z) * st.iz;
  constexpr float kNearSlack = 4.76837158e-7f, kFarSlack = 9.53674316e-7f, kQuantumSlack = 2.44140625e-4f;
  const float bnx = __builtin_fmaf(-fabsf(Bx), kNearSlack, Bx), bny = __builtin_fmaf(-fabsf(By), kNearSlack, By),
              bnz = __builtin_fmaf(-fabsf(Bz), kNearSlack, Bz);
  const float bfx = __builtin_fmaf(fabsf(Ax), kQuantumSlack, __builtin_fmaf(fabsf(Bx), kFarSlack, Bx)),
              bfy = __builtin_fmaf(fabsf(Ay), kQuantumSlack, __builtin_fmaf(fabsf(By), kFarSlack, By)),
              bfz = __builtin_fmaf(fabsf(Az), kQuantumSlack, __builtin_fmaf(fabsf(Bz), kFarSlack, Bz));
  constexpr float k2p24 = 16777216.0f;
  const float Ax24 = Ax * k2p24, Ay24 = Ay * k2p24, Az24 = Az * k2p24;
  const float tbScaled = st.tbest * s.hitScale;
  const uint32_t selX = st.ix < 0.0f ? kPlaneHi : kPlaneLo, selY = st.iy < 0.0f ? kPlaneHi : kPlaneLo,
                 selZ = st.iz < 0.0f ? kPlaneHi : kPlaneLo;
  // A hit child's key is its entry distance with the three lowest bits replaced
  // by the slot (rounded down, ties in slot order); misses are all ones.
  uint32_t misses = 0;  // bit k: slot k is missed
  uint32_t keys[kWideArity];
#pragma unroll
  for (int pair = kWideArity / 2 - 1; pair >= 0; --pair) {
    const uint32_t next = pair & 1 ? kPlaneNextPair : 0u;
    const bool high = pair >= 2;  // the words of slots 4..7
    const uint32_t nx = plane_pair(high ? q2.y : q2.x, high ? q3.w : q3.z, selX ^ next);
    const uint32_t ny = plane_pair(high ? q2.w : q2.z, high ? q4.y : q4.x, selY ^ next);
    const uint32_t nz = plane_pair(high ? q3.y : q3.x, high ? q4.w : q4.z, selZ ^ next);
    const uint32_t fx = plane_pair(high ? q2.y : q2.x, high ? q3.w : q3.z, selX ^ next ^ kPlaneOther);
    const uint32_t fy = plane_pair(high ? q2.w : q2.z, high ? q4.y : q4.x, selY ^ next ^ kPlaneOther);
    const uint32_t fz = plane_pair(high ? q3.y : q3.x, high ? q4.w : q4.z, selZ ^ next ^ kPlaneOther);
#pragma unroll
    for (int h = 1; h >= 0; --h) {
      const int k = 2 * pair + h;
      const float tnear = fmaxf(fmaxf(fmaxf(plane_fma(nx, h, Ax24, bnx), plane_fma(ny, h, Ay24, bny)),
                                      plane_fma(nz, h, Az24, bnz)), 0.0f);
      const float tfar = fminf(fminf(fminf(plane_fma(fx, h, Ax24, bfx), plane_fma(fy, h, Ay24, bfy)),
                                     plane_fma(fz, h, Az24, bfz)), tbScaled);
      if (Q == kWideAny) {
        misses = __builtin_amdgcn_alignbit(misses, __float_as_uint(tfar - tnear), 31);
      } else {
        keys[k] = tnear <= tfar ? (__float_as_uint(tnear) & ~7u) | (uint32_t)k : 0xffffffffu;
        misses = __builtin_amdgcn_alignbit(misses, keys[k], 31);
      }
    }
  }
  uint32_t first = 0xffffffffu;  // the smallest key
  if (Q != kWideAny) {
#pragma unroll
    for (int k = 0; k < kWideArity; ++k) first = min(first, keys[k]);
  }
  const uint32_t inner = q0.w >> 24, hits = ~misses & 0xffu;
  const uint32_t leaves = hits & ~inner;
  uint32_t waiting = hits & inner;
  bool fits = true;
  st.node = kWideNoNode;
  if (waiting != 0u) {
    const uint32_t next = wide_next<Q>(st, waiting, first & 7u);
    st.node = wide_child(q1.x, inner, next);
    waiting &= ~(1u << next);
    if (waiting != 0u) {
      uint32_t e = waiting | (inner << 8);
      if (Q != kWideAny) {
        // the second smallest key: a distance, since two children or more are hit, and
        // no larger than those of the children that wait
        uint32_t a = keys[0], second = 0xffffffffu;
#pragma unroll
        for (int k = 1; k < kWideArity; ++k) {
          second = min(second, max(a, keys[k]));
          a = min(a, keys[k]);
        }
        e |= ((second & 7u) << 16) | (second & kWideBoundMask);
      }
      fits = wide_push<B, S>(s, st, stk, make_uint2(q1.x, e));
    }
  }
  if (leaves != 0u && !wide_hold(st, nodeIndex, leaves))
    fits = wide_push<B, S>(s, st, stk, make_uint2(nodeIndex | kWideLeafEntry, leaves | (Q == kWideAny ? 0u : first & kWideBoundMask))) &&
           fits;
  if (!fits) {
    atomicOr(s.errorFlag, 1u);
    st.bestSlot = -2;
  }
  return fits;
}

// Leaf pass for a lane with pending leaves: tests the triangles of one leaf of
// the first group.  One leaf a pass: a lane with several does not hold the
// others' next passes (2^24 diffuse rays on the heightfield: with all of a lane's
// leaves in one pass 1.10 times the time).
template <int Q, bool WT>
__device__ __forceinline__ void wide_leaf(const WideScene& s, WideState& st) {
  const gg::V3 o = st.o, d = st.d;
  // {firstChild, firstTri, ends} of the group's node
  const uint4 q1 = ((const uint4*)((const char*)s.nodes + ((st.leafNode[0] << 6) + (st.leafNode[0] << 4))))[1];
  const uint32_t shift = 8u * (uint32_t)__builtin_ctz(st.leafMask);
  uint32_t mask = st.leafMask & (st.leafMask - 1u);
  const bool last = (mask & 0xffu) == 0u;  // the second group moves up
  st.leafNode[0] = last ? st.leafNode[1] : st.leafNode[0];
  st.leafMask = last ? mask >> 8 : mask;
  const uint64_t ends = (uint64_t)q1.z | ((uint64_t)q1.w << 32);
  uint32_t tri = q1.y + ((uint32_t)((ends << 8) >> shift) & 0xffu);
  // empty for an unused slot whose inverted box the slack let through
  const uint32_t end = q1.y + ((uint32_t)(ends >> shift) & 0xffu);
  for (; tri < end; ++tri) {
    const size_t ti = 3 * (size_t)tri;
    const float4 a = s.tris[ti + 0];
    const float4 b = s.tris[ti + 1];
    const float4 c = s.tris[ti + 2];
    const gg::V3 p0 = gg::v3(a.x, a.y, a.z);
    const int slot = __float_as_int(a.w);
    float t, by, bz;
    bool ok;
    if (WT) {
      gg::V3 bary;
      ok = intersect_triangle_wt(o, st.wr, p0, gg::v3(b.x, b.y, b.z), gg::v3(c.x, c.y, c.z), t, bary);
      by = bary.y;
      bz = bary.z;
    } else {
      const gg::V3 e0 = gg::v3(b.x, b.y, b.z);
      const gg::V3 e1 = gg::v3(c.x, c.y, c.z);
      const gg::V3 nn = gg::cross(e1, e0);
      const gg::V3 e2 = (1.0f / gg::dot(nn, d)) * (p0 - o);
      const gg::V3 ii = gg::cross(d, e2);
      by = gg::dot(ii, e1);
      bz = gg::dot(ii, e0);
      const float bx = 1.0f - (bz + by);
      t = gg::dot(nn, e2);
      ok = t > 0.0001f && bx >= 0.0f && by >= 0.0f && bz >= 0.0f;
    }
    if (Q == kWideAny) {
      if (ok && t < st.tbest) {
        st.found = true;
        return;
      }
    } else if (ok && (t < st.tbest || (t == st.tbest && slot < st.bestSlot))) {
      st.tbest = t;
      st.bestSlot = slot;
      st.bu = by;
      st.bv = bz;
    }
  }
}

// For a lane without a next node: pops entries still in front of the closest
// hit until one yields a node, or a leaf group finds both pending slots taken
// (the entry stays), or the stack is empty.
template <int Q, int B, int S>
__device__ __forceinline__ void wide_pop(const WideScene& s, WideState& st, const WideStack& stk) {
  const float tb = st.tbest * s.hitScale;  // entry distances are lower bounds with this slack
  int sp = st.sp;
  uint32_t node = kWideNoNode;
  while (sp > 0) {
    const int top = sp - 1;
    uint2 e;
    if (top < S) e = stk.lds[top * B + stk.tid];
    else e = stk.spill[(size_t)(top - S) * stk.spillStride];
    if (Q != kWideAny && __uint_as_float(e.y & kWideBoundMask) > tb) {
      sp = top;
      continue;
    }
    if (e.x & kWideLeafEntry) {
      if (!wide_hold(st, e.x & ~kWideLeafEntry, e.y & 0xffu)) break;
      sp = top;
      continue;
    }
    const uint32_t next = wide_next<Q>(st, e.y & 0xffu, (e.y >> 16) & 7u);  // a node entry has a waiting child
    node = wide_child(e.x, (e.y >> 8) & 0xffu, next);
    e.y &= ~(1u << next);
    if ((e.y & 0xffu) == 0u) sp = top;
    else if (top < S) stk.lds[top * B + stk.tid].y = e.y;
    else stk.spill[(size_t)(top - S) * stk.spillStride].y = e.y;
    break;
  }
  st.sp = sp;
  st.node = node;
}

// Wave-uniform pass choice for the working lanes (mask `working`, a ballot
// taken by the caller): a leaf pass when no working lane has a node to visit
// or at least `waitLanes` of them have only pending leaves.
__device__ __forceinline__ bool wide_choose_leaf_pass(uint64_t working, const WideState& st, int waitLanes) {
  const uint64_t hasNode = __ballot(st.node != kWideNoNode);
  return (working & hasNode) == 0 || __popcll(working & ~hasNode) >= waitLanes;
}

// One pass for a working lane.  Returns true when the ray is finished.
template <int Q, int B, int S, bool WT>
__device__ __forceinline__ bool wide_pass(const WideScene& s, WideState& st, bool leafPass, const WideStack& stk) {
  if (leafPass) {
    if (st.leafMask == 0u) return false;  // still traversing; unaffected by this pass
    wide_leaf<Q, WT>(s, st);
    if (Q == kWideAny && st.found) return true;
    if (Q == kWideMixed && st.anyHit && st.bestSlot >= 0) return true;
  } else {
    if (st.node == kWideNoNode) return false;  // waiting for a leaf pass
    if (!wide_visit<Q, B, S>(s, st, stk)) return true;  // overflow, slot -2
  }
  if (st.node == kWideNoNode) {
    wide_pop<Q, B, S>(s, st, stk);
    return st.node == kWideNoNode && st.leafMask == 0u;
  }
  return false;
}

// Traces one ray per calling lane to the end; the calling lanes form the wave
// for pass choices.  lds: LDS array of S * B stack entries; tid in [0, B);
// spill: this thread's own slice of s.spillDepth entries.
template <bool ANY, int B, int S, bool WT = false>
__device__ __forceinline__ WideResult trace_wide_ray(const WideScene& s, gg::V3 o, gg::V3 d, float tmax,
                                                     uint2* lds, int tid, uint2* spill) {
  const WideStack stk{as_lds(lds), tid, spill, 1u};
  WideState st;
  wide_init<WT>(s, st, o, d, tmax);
  bool live = true;
  for (;;) {
    const uint64_t act = __ballot(live);
    if (act == 0) break;
    // a quarter of the live lanes: 3 % (room, path tracer) below a half; an eighth is the same
    const bool leafPass = wide_choose_leaf_pass(act, st, (__popcll(act) + 3) / 4);
    if (live && wide_pass<ANY, B, S, WT>(s, st, leafPass, stk)) live = false;
  }
  WideResult r;
  r.t = st.tbest;
  r.slot = st.bestSlot;
  r.by = st.bu;
  r.bz = st.bv;
  r.any = st.found;
  return r;
}

}  // namespace gpugi
