// Traversal kernels and ray generators of the microbenchmark.
// Compiled with -ffp-contract=off: the triangle test must round exactly like
// the reference formula.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "launch.h"

namespace gpugi {

// ---------------------------------------------------------------------------
// Reference layout, one ray per lane, in wave-wide steps: up to kRefBoxSteps box
// steps of every lane without a leaf to test, or, once a quarter of the lanes at
// work have one, a leaf step of those.  A ray waits at its leaf, since its next
// box test needs the leaf's hit distance.  Lanes whose ray has ended take the
// next rays of the wave's batches once kRefRefill are idle; but where every wave has
// several batches and the rays of the one at hand all point into one octant, only
// once all have ended: such rays mostly end together, and a refill stalls the wave
// for the new rays' load (2^23 camera rays, room of 16 spheres: 740 -> 660 us).
// Bound by the dependent 32-byte node loads.  With one thread per ray almost every
// turn of a wave's loop ran the triangle test for a few lanes, and a wave lasted
// as long as its longest ray: 2^20 diffuse rays on a 524,288-triangle
// heightfield 866 -> 472 us, 2^24 on the 2,097,152-triangle one 13.0 -> 6.2 ms
// (2.7 Grays/s).  A leaf step at an eighth of the lanes: 492 us; at 16 lanes: 593 us;
// two box steps a turn: 635 us against 593 with four.  Refills at 8 idle lanes: 2.66
// against 2.50 ms for 2^23 diffuse rays on the 524,288-triangle heightfield.
// Waves are dealt out statically (the walk needs no memory but the caller's): block
// b runs on XCD b % 8, and the waves of an XCD take its batches in turn.  XCD x's
// are the x-th eighth of the ray array, so that neighbouring rays share an L2; from
// four batches a wave on it has every eighth chunk of 2^kRefChunkLog2 batches, since
// the eighths of an image can cost very differently, and the launch waits for the
// dearest (2^21 camera rays, room of 400 spheres: 1230 -> 950 us; the larger the
// chunks, the less so: 2^23 camera rays, 524,288-triangle heightfield, 1.57 ms with
// 2^8 batches, 1.85 with 2^10).
constexpr int kRefBoxSteps = 4;
constexpr uint32_t kRefRefill = 16, kRefXcds = 8, kRefWaves = 256 / 64, kRefChunkLog2 = 8;
constexpr uint32_t kRefTinyNodes = 1024, kRefL2Nodes = (4u << 20) / 32;

template <bool ANY, bool WT, bool OBOX>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8))) void k_trace_ref(
    RefScene s, const float4* __restrict__ rays, int4* __restrict__ hits, uint32_t n,
    const uint32_t* __restrict__ nDev, uint32_t resident) {
  if (nDev) n = min(*nDev, n);  // the ray count as the device holds it
  const int lane = threadIdx.x & 63;
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t batches = (n + 63u) / 64u, perX = (batches + kRefXcds - 1u) / kRefXcds;
  const uint32_t xcd = blockIdx.x % kRefXcds;
  const uint32_t stride = gridDim.x / kRefXcds * kRefWaves;
  const bool several = batches >= 2u * resident;
  const bool inChunks = several && (s.numNodes <= kRefTinyNodes || batches >= 4u * resident);
  constexpr uint32_t mask = (1u << kRefChunkLog2) - 1u;
  // wave-uniform: which of the XCD's batches is next, the batch being handed out, how
  // many of its rays are gone, and the idle lanes to wait for
  uint32_t nextOfXcd = blockIdx.x / kRefXcds * kRefWaves +
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)threadIdx.x / 64);
  uint32_t cur = 0, pos = 64, refill = kRefRefill;
  bool exhausted = false, active = false;
  uint32_t ri = 0;
  RefWalk w;
  for (;;) {
    const uint64_t idle = ~__ballot(active);
    const uint32_t nidle = (uint32_t)__popcll(idle);
    if (!exhausted && nidle >= refill) {
      const uint32_t avail = 64u - pos;
      const uint32_t next = inChunks ? (nextOfXcd & ~mask) * kRefXcds + (xcd << kRefChunkLog2) + (nextOfXcd & mask)
                                     : xcd * perX + nextOfXcd;
      const bool more = avail < nidle && next < batches && (inChunks || nextOfXcd < perX);
      if (!active) {
        const uint32_t rank = (uint32_t)__popcll(idle & below);
        uint32_t r = n;
        if (rank < avail) r = cur * 64u + pos + rank;
        else if (more) r = next * 64u + (rank - avail);
        if (r < n) {
          const float4 r0 = rays[2 * (size_t)r], r1 = rays[2 * (size_t)r + 1];
          ref_walk_init<WT>(w, gg::v3(r0.x, r0.y, r0.z), gg::v3(r1.x, r1.y, r1.z), r0.w);
          ri = r;
          active = true;
        }
      }
      if (avail >= nidle) {
        pos += nidle;
      } else if (more) {
        cur = next;
        pos = nidle - avail;
        nextOfXcd += stride;
      } else {
        exhausted = true;
      }
      if (several && nidle == 64u) {
        const uint64_t all = __ballot(active), x = __ballot(active && w.d.x < 0.0f),
                       y = __ballot(active && w.d.y < 0.0f), z = __ballot(active && w.d.z < 0.0f);
        refill = (x == 0 || x == all) && (y == 0 || y == all) && (z == 0 || z == all) ? 64u : kRefRefill;
      }
    }
    const uint64_t act = __ballot(active);
    if (act == 0) {
      if (exhausted) break;
      continue;
    }
    const uint64_t leaves = __ballot(active && w.leaf >= 0);
    bool ended = false;
    if (4 * __popcll(leaves) >= __popcll(act)) {
      if (active && w.leaf >= 0) ended = ref_walk_leaf<ANY, WT>(s, w);
    } else {
      for (int k = 0; k < kRefBoxSteps; ++k)
        if (active && w.leaf < 0 && !ended) ended = ref_walk_box<OBOX>(s, w);
    }
    if (ended) {
      if (ANY) hits[ri] = make_int4(w.found ? 1 : 0, 0, 0, 0);
      else hits[ri] = make_int4(w.slot, __float_as_int(w.t), __float_as_int(w.by), __float_as_int(w.bz));
      active = false;
    }
  }
}

// TRACERAY_IMPORTANCE_BREAK walk; nodes (optional) get {hit node, node
// importance bits, node size^2 bits, 0} per ray.
template <bool ANY, bool WT>
__global__ __launch_bounds__(256) void k_trace_ref_ib(RefScene s, const float4* __restrict__ rays,
                                                      int4* __restrict__ hits, int4* __restrict__ nodes, uint32_t n,
                                                      ImportanceBreak ib) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float4 r0 = rays[2 * (size_t)i], r1 = rays[2 * (size_t)i + 1];
  gg::V3 o = gg::v3(r0.x, r0.y, r0.z), d = gg::v3(r1.x, r1.y, r1.z);
  float rayLength = r0.w;
  RefHit h;
  uint32_t nb = 0, nt = 0;
  const bool any = trace_ref<ANY, false, WT>(s, o, d, rayLength, h, nb, nt, ib);
  if (ANY) {
    hits[i] = make_int4(any ? 1 : 0, 0, 0, 0);
  } else {
    hits[i] = make_int4(h.slot, __float_as_int(rayLength), __float_as_int(h.slot >= 0 ? h.bary.y : 0.0f),
                        __float_as_int(h.slot >= 0 ? h.bary.z : 0.0f));
    if (nodes) nodes[i] = make_int4(h.node, __float_as_int(h.nodeImportance), __float_as_int(h.nodeSizeSq), 0);
  }
}

template <bool ANY>
__global__ __launch_bounds__(256) void k_trace_ref_counts(RefScene s, const float4* __restrict__ rays,
                                                          uint32_t* __restrict__ nbox,
                                                          uint32_t* __restrict__ ntri, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const float4 r0 = rays[2 * (size_t)i], r1 = rays[2 * (size_t)i + 1];
  gg::V3 o = gg::v3(r0.x, r0.y, r0.z), d = gg::v3(r1.x, r1.y, r1.z);
  float rayLength = r0.w;
  RefHit h;
  uint32_t nb = 0, nt = 0;
  trace_ref<ANY, true>(s, o, d, rayLength, h, nb, nt);
  nbox[i] = nb;
  ntri[i] = nt;
}

hipError_t LaunchTraceRefImportance(const RefScene& s, int query, const gpugi_ray* rays, gpugi_hit* hits,
                                    int4* nodes, size_t n, const ImportanceBreak& ib, bool watertight,
                                    hipStream_t stream) {
  if (n == 0) return hipSuccess;
  dim3 grid((unsigned)((n + 255) / 256));
  const float4* r = (const float4*)rays;
  int4* h = (int4*)hits;
  const uint32_t m = (uint32_t)n;
  if (query == GPUGI_ANY_HIT) {
    if (watertight) hipLaunchKernelGGL((k_trace_ref_ib<true, true>), grid, dim3(256), 0, stream, s, r, h, nodes, m, ib);
    else hipLaunchKernelGGL((k_trace_ref_ib<true, false>), grid, dim3(256), 0, stream, s, r, h, nodes, m, ib);
  } else {
    if (watertight) hipLaunchKernelGGL((k_trace_ref_ib<false, true>), grid, dim3(256), 0, stream, s, r, h, nodes, m, ib);
    else hipLaunchKernelGGL((k_trace_ref_ib<false, false>), grid, dim3(256), 0, stream, s, r, h, nodes, m, ib);
  }
  return hipGetLastError();
}

hipError_t LaunchTraceRef(const RefScene& s, int query, const gpugi_ray* rays, gpugi_hit* hits, size_t n,
                          bool watertight, hipStream_t stream, const uint32_t* nDevice) {
  if (n == 0) return hipSuccess;
  if (n > 0xffffffffull - 255) return hipErrorInvalidValue;  // the kernel indexes rays with 32 bits
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  // A wave for every batch on a tree of some dozen triangles: its rays end after a few
  // steps, and waves that the hardware deals out balance better than refills pay
  // (Cornell room, 2^21 camera / diffuse / shadow rays: 71 / 234 / 127 us; 94 / 239 / 158
  // with resident waves).  Else at most eight blocks per CU, which hide the loads'
  // latency best, or six where each still gets four batches and more and the tree is
  // larger than an XCD's L2 (4 MB): fewer waves share the L1 better (2^23 diffuse rays,
  // 2,097,152-triangle heightfield: 3.3 against 3.5 ms).  Whole blocks per XCD.
  const uint32_t batches = (uint32_t)((n + 63) / 64);
  const uint32_t perX = (batches + kRefXcds - 1) / kRefXcds;
  const uint32_t resident = (uint32_t)cus * 8 * kRefWaves, blocks = (perX + kRefWaves - 1) / kRefWaves;
  const uint32_t perCu = batches >= 4 * resident && s.numNodes > kRefL2Nodes ? 6 : 8;
  const uint32_t most = s.numNodes <= kRefTinyNodes ? blocks : std::max(1u, (uint32_t)cus * perCu / kRefXcds);
  dim3 grid(kRefXcds * std::min(blocks, most));
  typedef void (*Kernel)(RefScene, const float4*, int4*, uint32_t, const uint32_t*, uint32_t);
  static const Kernel kernels[2][2][2] = {
      {{k_trace_ref<false, false, false>, k_trace_ref<false, false, true>},
       {k_trace_ref<false, true, false>, k_trace_ref<false, true, true>}},
      {{k_trace_ref<true, false, false>, k_trace_ref<true, false, true>},
       {k_trace_ref<true, true, false>, k_trace_ref<true, true, true>}}};
  const Kernel fn = kernels[query == GPUGI_ANY_HIT][watertight ? 1 : 0][s.obox ? 1 : 0];
  hipLaunchKernelGGL(fn, grid, dim3(256), 0, stream, s, (const float4*)rays, (int4*)hits, (uint32_t)n, nDevice, resident);
  return hipGetLastError();
}

hipError_t LaunchTraceRefCounts(const RefScene& s, int query, const gpugi_ray* rays, uint32_t* nbox,
                                uint32_t* ntri, size_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  dim3 grid((unsigned)((n + 255) / 256));
  if (query == GPUGI_ANY_HIT)
    hipLaunchKernelGGL(k_trace_ref_counts<true>, grid, dim3(256), 0, stream, s, (const float4*)rays, nbox,
                       ntri, (uint32_t)n);
  else
    hipLaunchKernelGGL(k_trace_ref_counts<false>, grid, dim3(256), 0, stream, s, (const float4*)rays, nbox,
                       ntri, (uint32_t)n);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Ray generators.
__global__ __launch_bounds__(256) void k_raygen_primary(gpugi_camera cam, int width, int height, uint32_t seed,
                                                        float4* __restrict__ rays, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t pix = i % (uint32_t)(width * height);
  const int px = (int)(pix % (uint32_t)width), py = (int)(pix / (uint32_t)width);
  uint32_t rs = gg::init_random_seed(seed, i);
  float j0 = gg::random01(rs);
  float j1 = gg::random01(rs);
  gg::V3 U = gg::v3(cam.u[0], cam.u[1], cam.u[2]);
  gg::V3 V = gg::v3(cam.v[0], cam.v[1], cam.v[2]);
  gg::V3 W = gg::v3(cam.w[0], cam.w[1], cam.w[2]);
  gg::V3 d = gg::primary_direction(j0, j1, px, py, width, height, U, V, W);
  rays[2 * (size_t)i] = make_float4(cam.position[0], cam.position[1], cam.position[2], gg::kRayMax);
  rays[2 * (size_t)i + 1] = make_float4(d.x, d.y, d.z, 0.0f);
}

hipError_t LaunchRaygenPrimary(const gpugi_camera& cam, int width, int height, uint32_t seed, gpugi_ray* rays,
                               size_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_raygen_primary, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, cam, width,
                     height, seed, (float4*)rays, (uint32_t)n);
  return hipGetLastError();
}

// Deterministic stream compaction of the hit indices (index order kept):
// per-block counts, one-block scan of the counts, scatter.
constexpr int kScanBlock = 1024;

__global__ __launch_bounds__(kScanBlock) void k_compact_count(const int4* __restrict__ hits, uint32_t n,
                                                              uint32_t* __restrict__ blockCounts) {
  __shared__ uint32_t warpSums[kScanBlock / 64];
  const uint32_t i = blockIdx.x * kScanBlock + threadIdx.x;
  const bool flag = i < n && hits[i].x >= 0;
  uint64_t mask = __ballot(flag);
  if ((threadIdx.x & 63) == 0) warpSums[threadIdx.x >> 6] = (uint32_t)__popcll(mask);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t s = 0;
    for (int w = 0; w < kScanBlock / 64; ++w) s += warpSums[w];
    blockCounts[blockIdx.x] = s;
  }
}

__global__ __launch_bounds__(kScanBlock) void k_compact_scan(uint32_t* __restrict__ blockCounts, uint32_t numBlocks,
                                                             uint32_t* __restrict__ total) {
  // Single block: each thread scans a contiguous chunk, then a block scan of chunk sums.
  __shared__ uint32_t sums[kScanBlock];
  const uint32_t per = (numBlocks + kScanBlock - 1) / kScanBlock;
  const uint32_t begin = threadIdx.x * per;
  uint32_t local = 0;
  for (uint32_t k = 0; k < per; ++k)
    if (begin + k < numBlocks) local += blockCounts[begin + k];
  sums[threadIdx.x] = local;
  __syncthreads();
  for (int off = 1; off < kScanBlock; off <<= 1) {
    uint32_t v = threadIdx.x >= (uint32_t)off ? sums[threadIdx.x - off] : 0u;
    __syncthreads();
    sums[threadIdx.x] += v;
    __syncthreads();
  }
  uint32_t run = sums[threadIdx.x] - local;  // exclusive prefix of this chunk
  for (uint32_t k = 0; k < per; ++k) {
    if (begin + k < numBlocks) {
      uint32_t c = blockCounts[begin + k];
      blockCounts[begin + k] = run;
      run += c;
    }
  }
  if (threadIdx.x == kScanBlock - 1) *total = sums[kScanBlock - 1];
}

__global__ __launch_bounds__(kScanBlock) void k_compact_scatter(const int4* __restrict__ hits, uint32_t n,
                                                                const uint32_t* __restrict__ blockOffsets,
                                                                uint32_t* __restrict__ list) {
  __shared__ uint32_t warpSums[kScanBlock / 64];
  const uint32_t i = blockIdx.x * kScanBlock + threadIdx.x;
  const bool flag = i < n && hits[i].x >= 0;
  uint64_t mask = __ballot(flag);
  const uint32_t lane = threadIdx.x & 63;
  if (lane == 0) warpSums[threadIdx.x >> 6] = (uint32_t)__popcll(mask);
  __syncthreads();
  uint32_t base = blockOffsets[blockIdx.x];
  for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) base += warpSums[w];
  const uint64_t below = lane ? (mask & (~0ull >> (64 - lane))) : 0ull;
  if (flag) list[base + (uint32_t)__popcll(below)] = i;
}

hipError_t LaunchHitCompaction(const gpugi_hit* hits, size_t n, uint32_t* list, uint32_t* count, void* temp,
                               size_t* tempBytes, hipStream_t stream) {
  const uint32_t numBlocks = (uint32_t)((n + kScanBlock - 1) / kScanBlock);
  const size_t need = (size_t)numBlocks * 4;
  if (!temp) { *tempBytes = need; return hipSuccess; }
  if (*tempBytes < need) return hipErrorInvalidValue;
  uint32_t* bc = (uint32_t*)temp;
  hipLaunchKernelGGL(k_compact_count, dim3(numBlocks), dim3(kScanBlock), 0, stream, (const int4*)hits,
                     (uint32_t)n, bc);
  hipLaunchKernelGGL(k_compact_scan, dim3(1), dim3(kScanBlock), 0, stream, bc, numBlocks, count);
  hipLaunchKernelGGL(k_compact_scatter, dim3(numBlocks), dim3(kScanBlock), 0, stream, (const int4*)hits,
                     (uint32_t)n, bc, list);
  return hipGetLastError();
}

// Hit point and geometric normal of primary ray j, as pathtracer.comp:56-61
// computes them (origin + t * dir; cross(e1, e0) of intersectiontests.glsl:68).
__device__ __forceinline__ void hit_frame(const RefScene& s, const float4* prim, const int4* hits, uint32_t j,
                                          gg::V3& p, gg::V3& din, gg::V3& ng) {
  const float4 r0 = prim[2 * (size_t)j], r1 = prim[2 * (size_t)j + 1];
  const int4 h = hits[j];
  gg::V3 o = gg::v3(r0.x, r0.y, r0.z);
  din = gg::v3(r1.x, r1.y, r1.z);
  p = o + __int_as_float(h.y) * din;
  const int4 tri = s.slots[h.x];
  gg::V3 p0 = load_pos(s.positions, tri.x), p1 = load_pos(s.positions, tri.y), p2 = load_pos(s.positions, tri.z);
  ng = gg::cross(p0 - p2, p1 - p0);
}

__global__ __launch_bounds__(256) void k_raygen_diffuse(RefScene s, const float4* __restrict__ prim,
                                                        const int4* __restrict__ hits,
                                                        const uint32_t* __restrict__ list,
                                                        const uint32_t* __restrict__ count, uint32_t seed,
                                                        float4* __restrict__ rays, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t nh = *count;
  if (nh == 0) {  // nothing was hit: emit an inert ray
    rays[2 * (size_t)i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    rays[2 * (size_t)i + 1] = make_float4(0.0f, 1.0f, 0.0f, 0.0f);
    return;
  }
  const uint32_t j = list[i % nh];
  gg::V3 p, din, ng;
  hit_frame(s, prim, hits, j, p, din, ng);
  gg::V3 N = gg::normalize(ng);
  if (gg::dot(N, din) > 0.0f) N = -N;
  gg::V3 U, V;
  gg::create_onb(N, U, V);
  uint32_t rs = gg::init_random_seed(seed, i);
  float r0 = gg::random01(rs);
  float r1 = gg::random01(rs);
  gg::V3 d = gg::sample_hemisphere_cosine(r0, r1, U, V, N);
  gg::V3 o = p + d * gg::kRayHitEpsilon;
  rays[2 * (size_t)i] = make_float4(o.x, o.y, o.z, gg::kRayMax);
  rays[2 * (size_t)i + 1] = make_float4(d.x, d.y, d.z, 0.0f);
}

__global__ __launch_bounds__(256) void k_raygen_shadow(const float4* __restrict__ prim,
                                                       const int4* __restrict__ hits,
                                                       const uint32_t* __restrict__ list,
                                                       const uint32_t* __restrict__ count,
                                                       const float* __restrict__ lights, uint32_t numLights,
                                                       float4* __restrict__ rays, uint32_t n) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n) return;
  const uint32_t nh = *count;
  if (nh == 0) {
    rays[2 * (size_t)i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    rays[2 * (size_t)i + 1] = make_float4(0.0f, 1.0f, 0.0f, 0.0f);
    return;
  }
  const uint32_t j = list[i % nh];
  const float4 a = prim[2 * (size_t)j], b = prim[2 * (size_t)j + 1];
  gg::V3 p = gg::v3(a.x, a.y, a.z) + __int_as_float(hits[j].y) * gg::v3(b.x, b.y, b.z);
  const uint32_t l = i % numLights;
  gg::V3 L = gg::v3(lights[3 * l], lights[3 * l + 1], lights[3 * l + 2]);
  // EstimateDirectLight's shadow ray (lightsource.glsl:18-21,39-40).
  gg::V3 dir = L - p;
  float lightDistSq = gg::dot(dir, dir) + gg::kDivisorEpsilon;
  float lightDist = sqrtf(lightDistSq);
  dir = dir / lightDist;
  gg::V3 o = gg::kRayHitEpsilon * dir + p;
  rays[2 * (size_t)i] = make_float4(o.x, o.y, o.z, lightDist - gg::kRayHitEpsilon * 2.0f);
  rays[2 * (size_t)i + 1] = make_float4(dir.x, dir.y, dir.z, 0.0f);
}

hipError_t LaunchRaygenDiffuse(const RefScene& s, const gpugi_ray* prim, const gpugi_hit* hits,
                               const uint32_t* list, const uint32_t* count, uint32_t seed, gpugi_ray* rays,
                               size_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_raygen_diffuse, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, s,
                     (const float4*)prim, (const int4*)hits, list, count, seed, (float4*)rays, (uint32_t)n);
  return hipGetLastError();
}

hipError_t LaunchRaygenShadow(const gpugi_ray* prim, const gpugi_hit* hits, const uint32_t* list,
                              const uint32_t* count, const float* lights, uint32_t numLights, gpugi_ray* rays,
                              size_t n, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_raygen_shadow, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream,
                     (const float4*)prim, (const int4*)hits, list, count, lights, numLights, (float4*)rays,
                     (uint32_t)n);
  return hipGetLastError();
}

}  // namespace gpugi
