// Re-pack of the reference BVH2 into the 8-wide quantized layout of wide_bvh.h.
#include "../device/wide_bvh.h"

#include <algorithm>
#include <array>
#include <limits>
#include <cmath>
#include <cstring>

namespace gpugi {
namespace {

struct Bvh2View {
  const gpugi_scene_desc* d;
  uint32_t n;
  const float* box(uint32_t i) const { return d->hierarchy + (size_t)i * 8; }
  uint32_t firstChild(uint32_t i) const { uint32_t u; std::memcpy(&u, box(i) + 3, 4); return u; }
  uint32_t escape(uint32_t i) const { uint32_t u; std::memcpy(&u, box(i) + 7, 4); return u; }
  bool isLeafNode(uint32_t i) const { return (firstChild(i) & 0x80000000u) != 0; }
  float surface(uint32_t i) const {
    const float* b = box(i);
    float x = b[4] - b[0], y = b[5] - b[1], z = b[6] - b[2];
    return 2.0f * (x * y + y * z + z * x);
  }
};

// The exact real origin + q * scale (extended precision: the kernel never rounds a
// decoded bound, it folds q * scale into the slab distance).
long double Decode(float origin, uint32_t q, float scale) {
  return (long double)origin + (long double)q * (long double)scale;
}
float ScaleOf(uint32_t biased) { uint32_t u = biased << 23; float f; std::memcpy(&f, &u, 4); return f; }

}  // namespace

std::string BuildWideBVH(const gpugi_scene_desc& desc, uint32_t maxLeafTris, WideBVHHost* out, bool rawVertices) {
  constexpr int W = kWideArity;
  if (maxLeafTris < 1 || maxLeafTris > kWideMaxLeafTris) return "maxLeafTris must be in [1, 16]";
  Bvh2View v{&desc, desc.num_nodes};
  if (v.n == 0) return "empty hierarchy";
  const uint32_t tpl = desc.triangles_per_leaf;
  // Children of every inner node: firstChild, then escapes until the chain leaves
  // the parent (the last child escapes to the parent's escape); node i's are
  // kids[kidsAt[i]..kidsAt[i + 1]).
  std::vector<uint32_t> kids, kidsAt(v.n + 1, 0);
  kids.reserve(v.n);
  for (uint32_t i = 0; i < v.n; ++i) {
    kidsAt[i] = (uint32_t)kids.size();
    if (v.isLeafNode(i)) continue;
    uint32_t c = v.firstChild(i);
    const uint32_t stop = v.escape(i);
    for (int guard = 0;; ++guard) {
      if (guard == 64) return "node " + std::to_string(i) + " has more than 64 children";
      if (c <= i || c >= v.n) return "malformed hierarchy below node " + std::to_string(i);
      kids.push_back(c);
      const uint32_t e = v.escape(c);
      if (e == stop) break;
      if (e <= c) return "malformed escape chain below node " + std::to_string(i);
      c = e;
    }
  }
  kidsAt[v.n] = (uint32_t)kids.size();
  // Subtree valid-triangle counts, bottom-up (children follow parents in preorder).
  std::vector<uint32_t> count(v.n, 0);
  double area = 0.0;  // twice the triangles'
  for (uint32_t ii = v.n; ii-- > 0;) {
    uint32_t c = 0;
    if (v.isLeafNode(ii)) {
      uint32_t leaf = v.firstChild(ii) & 0x7fffffffu;
      if (leaf >= desc.num_leaves) return "leaf index out of range";
      for (uint32_t k = 0; k < tpl; ++k) {
        const int32_t* t = desc.triangles + ((size_t)leaf * tpl + k) * 4;
        if (t[0] == t[1]) break;
        ++c;
        double e0[3], e1[3], n2 = 0.0;
        for (int a = 0; a < 3; ++a) {
          const double p0 = desc.positions[(size_t)t[0] * 3 + a];
          e0[a] = desc.positions[(size_t)t[1] * 3 + a] - p0;
          e1[a] = desc.positions[(size_t)t[2] * 3 + a] - p0;
        }
        for (int a = 0; a < 3; ++a) {
          const int b = (a + 1) % 3, d = (a + 2) % 3;
          const double x = e0[b] * e1[d] - e0[d] * e1[b];
          n2 += x * x;
        }
        area += std::sqrt(n2);
      }
    } else {
      for (uint32_t k = kidsAt[ii]; k < kidsAt[ii + 1]; ++k) c += count[kids[k]];
    }
    count[ii] = c;
  }
  out->crossings = v.surface(0) > 0.0f ? (float)(area / (double)v.surface(0)) : 0.0f;
  out->nodes.clear();
  out->tris.clear();
  out->tris.reserve(count[0]);

  std::vector<uint32_t> walk;
  auto appendTris = [&](uint32_t sub) {
    // All valid slots of a BVH2 subtree in slot order of a preorder walk.
    walk.assign(1, sub);
    while (!walk.empty()) {
      uint32_t i = walk.back();
      walk.pop_back();
      if (v.isLeafNode(i)) {
        uint32_t leaf = v.firstChild(i) & 0x7fffffffu;
        for (uint32_t k = 0; k < tpl; ++k) {
          size_t slot = (size_t)leaf * tpl + k;
          const int32_t* t = desc.triangles + slot * 4;
          if (t[0] == t[1]) break;
          const float* p0 = desc.positions + (size_t)t[0] * 3;
          const float* p1 = desc.positions + (size_t)t[1] * 3;
          const float* p2 = desc.positions + (size_t)t[2] * 3;
          WideTriHost w;
          for (int a = 0; a < 3; ++a) {
            w.p0[a] = p0[a];
            // reference test operands e0 = p1 - p0, e1 = p0 - p2, or the raw vertices
            w.e0[a] = rawVertices ? p1[a] : p1[a] - p0[a];
            w.e1[a] = rawVertices ? p2[a] : p0[a] - p2[a];
          }
          w.slot = (int32_t)slot;
          w.material = t[3];
          w.pad = 0;
          out->tris.push_back(w);
        }
      } else {
        for (uint32_t k = kidsAt[i + 1]; k-- > kidsAt[i];) walk.push_back(kids[k]);
      }
    }
  };

  // SAH-optimal collapse of the BVH2 into 8-wide nodes (the dynamic program of
  // Ylitie, Karras and Laine 2017).  dist[n][j] is the least expected cost of
  // covering n's subtree with at most j children of one wide node; a child is a
  // leaf (a reference leaf, or a subtree of at most maxLeafTris valid triangles)
  // or a wide node of its own.  A wide node costs kNodeCost * area per visit, a
  // leaf kTriCost * area * triangles; the ratio is the measured cost of a box
  // pass (the slab tests, ordering, stack) to that of one triangle test.  The
  // topology stays the reference's: only which BVH2 nodes become wide nodes or
  // leaves is chosen.
  constexpr float kNodeCost = 1.0f, kTriCost = 0.4f;
  constexpr float kInf = std::numeric_limits<float>::infinity();
  struct Dp {
    float dist[W + 1];
    uint8_t pick[W + 1];  // 0: no child (empty subtree), 1: n as one child, 2: n's children share j
    bool leaf;            // n as one child: a leaf (else a wide node)
    bool open;            // n's own children fit one wide node
  };
  std::vector<Dp> dp(v.n);
  // split[kidsAt[i] + k][j]: children given to kid k when kids 0..k of node i
  // share j (knapsack back-pointers)
  typedef std::array<uint8_t, W + 1> Split;
  std::vector<Split> split(kids.size(), Split{});
  for (uint32_t n = v.n; n-- > 0;) {
    Dp& d = dp[n];
    if (count[n] == 0) {
      for (int j = 0; j <= W; ++j) { d.dist[j] = 0.0f; d.pick[j] = 0; }
      d.leaf = d.open = true;
      continue;
    }
    const float area = v.surface(n);
    const bool leafOk = v.isLeafNode(n) || count[n] <= maxLeafTris;
    const float leafCost = leafOk ? kTriCost * area * (float)count[n] : kInf;
    std::array<float, W + 1> comb;
    comb.fill(kInf);
    if (!v.isLeafNode(n)) {
      comb[0] = 0.0f;
      for (uint32_t k = kidsAt[n]; k < kidsAt[n + 1]; ++k) {
        const Dp& c = dp[kids[k]];
        std::array<float, W + 1> next;
        next.fill(kInf);
        for (int j = 0; j <= W; ++j)
          for (int a = 0; a <= j; ++a) {
            const float cost = comb[j - a] + c.dist[a];
            if (cost < next[j]) { next[j] = cost; split[k][j] = (uint8_t)a; }
          }
        comb = next;
      }
    }
    const float nodeCost = v.isLeafNode(n) ? kInf : kNodeCost * area + comb[W];
    const float single = std::min(leafCost, nodeCost);
    d.leaf = leafCost <= nodeCost;
    d.open = v.isLeafNode(n) || comb[W] < kInf;
    d.dist[0] = kInf;
    d.pick[0] = 0;
    for (int j = 1; j <= W; ++j) {
      if (single <= comb[j]) { d.dist[j] = single; d.pick[j] = 1; }
      else { d.dist[j] = comb[j]; d.pick[j] = 2; }
    }
  }
  // The children of the wide node for BVH2 node n: n's own children sharing W.
  struct Item {
    uint32_t bvh2;
    bool leaf;
  };
  std::vector<Item> items;
  std::vector<std::pair<uint32_t, int>> work;  // (BVH2 node, children it may use), last first
  auto openKids = [&](uint32_t n, int j) {  // knapsack back-tracking over n's kids
    for (uint32_t k = kidsAt[n + 1]; k-- > kidsAt[n];) {
      const int a = split[k][j];
      work.push_back({kids[k], a});
      j -= a;
    }
  };
  auto wideChildren = [&](uint32_t n) {
    items.clear();
    if (v.isLeafNode(n)) {  // a one-leaf scene
      if (count[n] > 0) items.push_back({n, true});
      return;
    }
    work.clear();
    openKids(n, W);
    while (!work.empty()) {  // in the reference's child order
      const auto [c, j] = work.back();
      work.pop_back();
      const Dp& d = dp[c];
      if (j == 0 || d.pick[j] == 0) continue;
      if (d.pick[j] == 1) items.push_back({c, d.leaf});
      else openKids(c, j);
    }
  };

  struct Pending {
    uint32_t bvh2;       // BVH2 node whose subtree this wide node covers
    uint32_t wideIndex;  // index of the wide node to fill
  };
  std::vector<Pending> todo;
  uint32_t largest = 0;  // biased exponent of the largest quantum
  out->nodes.push_back(WideNodeHost());
  todo.push_back({0, 0});
  while (!todo.empty()) {
    Pending p = todo.back();
    todo.pop_back();
    // Subtrees without a valid triangle never produce a hit and are left out.
    wideChildren(p.bvh2);
    std::stable_sort(items.begin(), items.end(),
                     [&](const Item& a, const Item& b) { return v.surface(a.bvh2) < v.surface(b.bvh2); });
    if (!dp[p.bvh2].open) return "BVH node with more than 8 children cannot be packed";
    WideNodeHost node;
    std::memset(&node, 0, sizeof(node));
    std::memset(node.lo, 255, sizeof(node.lo));  // unused slots: inverted boxes, no triangles
    node.firstTri = (uint32_t)out->tris.size();
    if (items.empty()) {  // a scene without any valid triangle
      node.exps = 1u | (1u << 8) | (1u << 16);
      out->nodes[p.wideIndex] = node;
      continue;
    }
    // Quantization frame.
    float origin[3], top[3];
    for (int a = 0; a < 3; ++a) {
      origin[a] = v.box(items[0].bvh2)[a];
      top[a] = v.box(items[0].bvh2)[4 + a];
      for (const Item& it : items) {
        origin[a] = std::min(origin[a], v.box(it.bvh2)[a]);
        top[a] = std::max(top[a], v.box(it.bvh2)[4 + a]);
      }
      node.origin[a] = origin[a];
    }
    uint32_t biased[3];
    for (int a = 0; a < 3; ++a) {
      double ext = (double)top[a] - (double)origin[a];
      int b = 1;
      if (ext > 0.0) b = std::max(1, std::min(254, (int)std::ceil(std::log2(ext / 255.0)) + 127));
      for (;; ++b) {
        if (b > 254) return "cannot quantize a node box";
        const float scale = ScaleOf((uint32_t)b);
        bool ok = true;
        for (size_t k = 0; k < items.size() && ok; ++k) {
          const float lo = v.box(items[k].bvh2)[a], hi = v.box(items[k].bvh2)[4 + a];
          double ql = std::floor(((double)lo - (double)origin[a]) / (double)scale);
          double qh = std::ceil(((double)hi - (double)origin[a]) / (double)scale);
          if (ql < 0) ql = 0;
          if (qh > 255.0) { ok = false; break; }
          uint32_t qlo = (uint32_t)ql, qhi = (uint32_t)std::max(0.0, qh);
          while (qlo > 0 && Decode(origin[a], qlo, scale) > lo) --qlo;
          while (qhi <= 255 && Decode(origin[a], qhi, scale) < hi) ++qhi;
          if (qhi > 255 || Decode(origin[a], qlo, scale) > lo) { ok = false; break; }
          node.lo[a][k] = (uint8_t)qlo;
          node.hi[a][k] = (uint8_t)qhi;
        }
        if (ok) break;
      }
      biased[a] = (uint32_t)b;
      largest = std::max(largest, biased[a]);
    }
    uint32_t inner = 0, numInner = 0;
    for (size_t s = 0; s < (size_t)W; ++s) {
      if (s < items.size() && items[s].leaf) appendTris(items[s].bvh2);
      else if (s < items.size()) { inner |= 1u << s; ++numInner; }
      node.ends[s] = (uint8_t)(out->tris.size() - node.firstTri);
    }
    if (out->tris.size() > kWideMaxTris) return "too many triangles for the wide layout";
    node.firstChild = (uint32_t)out->nodes.size();
    if (node.firstChild + numInner > kWideMaxNodes) return "too many nodes for the wide layout";
    out->nodes.resize(out->nodes.size() + numInner);
    for (int s = W, i = (int)numInner; s-- > 0;)
      if ((inner >> s) & 1) todo.push_back({items[s].bvh2, node.firstChild + (uint32_t)--i});
    node.exps = biased[0] | (biased[1] << 8) | (biased[2] << 16) | (inner << 24);
    out->nodes[p.wideIndex] = node;
  }
  out->tScale = std::ldexp(1.0f, std::min(0, 127 + kWideQuantumLog2 - (int)largest));
  // Worst-case stack.  A visit goes on with one hit inner child; the other hit
  // inner children wait in one entry, and the hit leaves in another when both
  // pending-leaf slots of the lane are taken.  An unused slot counts as a leaf: from
  // about 10^6 of the node's extents away the slack of the slab test lets its
  // inverted box through.  So
  //   stack(n) = [n has two inner children] + [a slot of n is no inner child] + max stack(inner child).
  // An entry that waits keeps its place while children of it are visited, which
  // the sum covers.  Children are numbered after their parents.
  std::vector<uint32_t> stack(out->nodes.size(), 0), depth(out->nodes.size(), 1);
  for (size_t i = out->nodes.size(); i-- > 0;) {
    const WideNodeHost& n = out->nodes[i];
    const uint32_t numInner = (uint32_t)__builtin_popcount(n.exps >> 24);
    for (uint32_t c = n.firstChild; c < n.firstChild + numInner; ++c) {
      stack[i] = std::max(stack[i], stack[c]);
      depth[i] = std::max(depth[i], depth[c] + 1);
    }
    stack[i] += (numInner > 1 ? 1 : 0) + (numInner < (uint32_t)W ? 1 : 0);
  }
  out->maxStack = stack[0];
  out->depth = depth[0];
  return std::string();
}

}  // namespace gpugi
