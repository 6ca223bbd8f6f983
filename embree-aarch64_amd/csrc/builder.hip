// GPU BVH8 builder (see builder.h for the pipeline).
//
// Reference anchors for what each phase computes:
//   primitive references and validity: kernels/common/scene_triangle_mesh.h:127-147,220-231,
//     kernels/builders/primrefgen.cpp:36-56 (invalid triangles are skipped);
//   Morton codes on 2x centroids, 10 bits per axis: kernels/builders/bvh_builder_morton.h:70-101;
//   radix sort: common/algorithms/parallel_sort.h:437-456 (semantics only);
//   leaf/inner decision by SAH cost and the 8-wide collapse that repeatedly
//     opens the child with the largest half area: kernels/builders/bvh_builder_sah.h:222-330;
//   leaf fill e1 = v0-v1, e2 = v2-v0: kernels/geometry/triangle.h:40-41,98-120.
#include <algorithm>
#include <chrono>
#include <cstring>
#include <string>

#include "builder.h"

namespace rtg {

struct BuildCounters {
  uint32_t glo[3], ghi[3];
  uint32_t clo[3], chi[3];
  uint32_t maxabs;
  uint32_t valid;
  uint32_t node_count;
  uint32_t tri_count;
  uint32_t top_nodes;  // nodes that k_walk_top numbered
  uint32_t subtrees;   // subtrees that it left to k_walk_rest
  uint32_t max_depth;
  uint32_t error;  // bit 0: refit walk too long, bit 1: collapse index out of range, bit 2: bad tree,
                   // bit 8: the binary tree's build failed
  uint32_t max_stack;  // most traversal stack entries any root-to-node path can need
  uint32_t roots_seen; // tree roots met by the tree check
  double sah_nodes, sah_leaves, sah_leaves_tri;
};

constexpr uint32_t COUNTER_WORDS = sizeof(BuildCounters) / 4;
static_assert(COUNTER_WORDS <= 63, "the counters are posted by one wave");

constexpr uint32_t NONE = 0xffffffffu;
constexpr int BT = 256;

// A node of the 8-wide tree to come.
struct WideNode {
  uint32_t bref;   // binary ref: REF_LEAF | sorted prim index, or inner node index
  uint32_t tri;    // first of its subtree's leaf records (as many as it has primitives)
  uint32_t level;  // depth << 16 | stack entries the traversal may hold on reaching it
  uint32_t link;   // while it waits: its own number; when walked: the number of its first inner child
};

// ------------------------------------------------------------ reductions --

__device__ inline float wave_min(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ inline float wave_max(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
  return v;
}
__device__ inline uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
__device__ inline uint32_t wave_umax(uint32_t v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = max(v, (uint32_t)__shfl_xor(v, d, 64));
  return v;
}
__device__ inline double wave_sum(double v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}

// Per-scene reductions of a batched build.
struct SceneAcc {
  uint32_t glo[3], ghi[3], clo[3], chi[3];
  uint32_t valid;
  uint32_t pad[3];
};

__global__ void k_init_sacc(SceneAcc* a, uint32_t n) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (i >= n) return;
  for (int k = 0; k < 3; k++) {
    a[i].glo[k] = a[i].clo[k] = f2o(INFINITY);
    a[i].ghi[k] = a[i].chi[k] = f2o(-INFINITY);
  }
  a[i].valid = 0;
}

__global__ void k_fill_none(uint32_t* v, uint32_t n) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (i < n) v[i] = 0xffffffffu;
}

__global__ void k_iota(uint32_t* v, uint32_t n) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (i < n) v[i] = i;
}

// The counters of a new build, and its geometries from pinned memory.
__global__ __launch_bounds__(BT) void k_init_build(BuildCounters* c, uint32_t nscenes,
                                                   const uint32_t* __restrict__ stage, uint32_t* __restrict__ geoms,
                                                   uint32_t words) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (i < words) geoms[i] = stage[i];
  if (i != 0) return;
  for (int k = 0; k < 3; k++) {
    c->glo[k] = f2o(INFINITY);
    c->ghi[k] = f2o(-INFINITY);
    c->clo[k] = f2o(INFINITY);
    c->chi[k] = f2o(-INFINITY);
  }
  c->maxabs = f2o(0.0f);
  c->valid = 0;
  c->node_count = nscenes;
  c->roots_seen = 0;
  c->tri_count = 0;
  c->top_nodes = 0;
  c->subtrees = 0;
  c->max_depth = 0;
  c->max_stack = 0;
  c->error = 0;
  c->sah_nodes = c->sah_leaves = c->sah_leaves_tri = 0.0;
}

// ------------------------------------------------------------ primrefs --

__device__ inline bool finite_v(float x) { return (x > -FLT_LARGE_) & (x < FLT_LARGE_); }

// Primitive references of PR_PER * BT consecutive primitives per block
// (PR_PER per thread, BT apart), with the scene bounds and valid count
// reduced over the block before one set of global atomics: one set per
// BT primitives would serialise on those few addresses.
constexpr int PR_PER = 4;

__global__ __launch_bounds__(BT) void k_primrefs(const GeomDesc* __restrict__ geoms, uint32_t ngeoms,
                                                 uint32_t total, float4* __restrict__ lo4,
                                                 float4* __restrict__ hi4, uint32_t* __restrict__ keys,
                                                 BuildCounters* __restrict__ cnt, SceneAcc* __restrict__ sacc) {
  float b[13];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    b[k] = INFINITY;        // geom lo
    b[3 + k] = -INFINITY;   // geom hi
    b[6 + k] = INFINITY;    // cent lo
    b[9 + k] = -INFINITY;   // cent hi
  }
  b[12] = 0.0f;
  uint32_t valid = 0, smin = 0xffffffffu, smax = 0u;
  const uint32_t base = blockIdx.x * (BT * PR_PER) + threadIdx.x;
#pragma unroll
  for (int j = 0; j < PR_PER; j++) {
    const uint32_t i = base + (uint32_t)j * BT;
    if (i >= total) break;
    uint32_t lo = 0, hi = ngeoms - 1;
    while (lo < hi) {  // last geometry with prim_offset <= i
      uint32_t mid = (lo + hi + 1) >> 1;
      if (geoms[mid].prim_offset <= i) lo = mid; else hi = mid - 1;
    }
    const GeomDesc g = geoms[lo];
    const uint32_t prim = i - g.prim_offset;
    bool ok;
    float l[3], h[3];
    if (g.kind == GEOM_INSTANCES) {  // a precomputed world box per instance record
      const float* bx = (const float*)(g.vertices + (uint64_t)prim * g.vstride);
      ok = true;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        l[k] = bx[k];
        h[k] = bx[3 + k];
        ok = ok && finite_v(l[k]) && finite_v(h[k]) && (l[k] <= h[k]);
      }
    } else {
      const uint32_t* ix = (const uint32_t*)(g.indices + (uint64_t)prim * g.istride);
      const uint32_t i0 = ix[0], i1 = ix[1], i2 = ix[2];
      ok = (i0 < g.num_vertices) & (i1 < g.num_vertices) & (i2 < g.num_vertices);
      float v[9];
      if (ok) {
        const float* p0 = (const float*)(g.vertices + (uint64_t)i0 * g.vstride);
        const float* p1 = (const float*)(g.vertices + (uint64_t)i1 * g.vstride);
        const float* p2 = (const float*)(g.vertices + (uint64_t)i2 * g.vstride);
        v[0] = p0[0]; v[1] = p0[1]; v[2] = p0[2];
        v[3] = p1[0]; v[4] = p1[1]; v[5] = p1[2];
        v[6] = p2[0]; v[7] = p2[1]; v[8] = p2[2];
#pragma unroll
        for (int k = 0; k < 9; k++) ok &= finite_v(v[k]);
      }
#pragma unroll
      for (int k = 0; k < 3; k++) {
        l[k] = ok ? fminf(v[k], fminf(v[3 + k], v[6 + k])) : 0.0f;
        h[k] = ok ? fmaxf(v[k], fmaxf(v[3 + k], v[6 + k])) : 0.0f;
      }
    }
    if (ok) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const float c2 = l[k] + h[k];
        b[k] = fminf(b[k], l[k]);
        b[3 + k] = fmaxf(b[3 + k], h[k]);
        b[6 + k] = fminf(b[6 + k], c2);
        b[9 + k] = fmaxf(b[9 + k], c2);
        b[12] = fmaxf(b[12], fmaxf(fabsf(l[k]), fabsf(h[k])));
      }
      lo4[i] = make_float4(l[0], l[1], l[2], __uint_as_float(lo));
      hi4[i] = make_float4(h[0], h[1], h[2], __uint_as_float(prim));
      keys[i] = g.scene;
      smin = min(smin, g.scene);
      smax = max(smax, g.scene);
      valid++;
    } else {
      keys[i] = 0xffffffffu;
    }
  }
  // block reduction
  __shared__ float red[BT / 64][13];
  __shared__ uint32_t redc[BT / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < 13; k++) {
    const bool mx = (k >= 3 && k < 6) || (k >= 9);
    float x = mx ? wave_max(b[k]) : wave_min(b[k]);
    if (lane == 0) red[wave][k] = x;
  }
  uint32_t vc = wave_sum(valid);
  if (lane == 0) redc[wave] = vc;
  __shared__ uint32_t s_min, s_max;
  if (threadIdx.x == 0) {
    s_min = 0xffffffffu;
    s_max = 0u;
  }
  __syncthreads();
  if (sacc && valid) {
    atomicMin(&s_min, smin);
    atomicMax(&s_max, smax);
  }
  if (threadIdx.x < 13) {
    const int k = threadIdx.x;
    const bool mx = (k >= 3 && k < 6) || (k >= 9);
    float x = red[0][k];
    for (int w = 1; w < BT / 64; w++) x = mx ? fmaxf(x, red[w][k]) : fminf(x, red[w][k]);
    uint32_t* dst = (k < 3) ? &cnt->glo[k] : (k < 6) ? &cnt->ghi[k - 3] : (k < 9) ? &cnt->clo[k - 6]
                    : (k < 12) ? &cnt->chi[k - 9] : &cnt->maxabs;
    if (!__builtin_isinf(x) && !(k == 12 && x == 0.0f)) {
      if (mx) atomicMax(dst, f2o(x)); else atomicMin(dst, f2o(x));
    }
  }
  if (threadIdx.x == 0) {
    uint32_t sum = 0;
    for (int w = 0; w < BT / 64; w++) sum += redc[w];
    if (sum) atomicAdd(&cnt->valid, sum);
  }
  if (!sacc) return;
  // per-scene bounds: the block's reduction when all its valid primitives
  // belong to one scene, else one set of atomics per primitive
  __syncthreads();
  if (s_min == 0xffffffffu) return;
  if (s_min == s_max) {
    SceneAcc* a = sacc + s_min;
    if (threadIdx.x < 12) {
      const int k = threadIdx.x;
      const bool mx = (k >= 3 && k < 6) || (k >= 9);
      float x = red[0][k];
      for (int w = 1; w < BT / 64; w++) x = mx ? fmaxf(x, red[w][k]) : fminf(x, red[w][k]);
      uint32_t* dst = (k < 3) ? &a->glo[k] : (k < 6) ? &a->ghi[k - 3] : (k < 9) ? &a->clo[k - 6] : &a->chi[k - 9];
      if (mx) atomicMax(dst, f2o(x)); else atomicMin(dst, f2o(x));
    }
    if (threadIdx.x == 0) {
      uint32_t sum = 0;
      for (int w = 0; w < BT / 64; w++) sum += redc[w];
      atomicAdd(&a->valid, sum);
    }
  } else {
    for (int j = 0; j < PR_PER; j++) {
      const uint32_t i = base + (uint32_t)j * BT;
      if (i >= total) break;
      const uint32_t sc = keys[i];
      if (sc == 0xffffffffu) continue;
      SceneAcc* a = sacc + sc;
      const float4 l = lo4[i], h = hi4[i];
      const float lv[3] = {l.x, l.y, l.z}, hv[3] = {h.x, h.y, h.z};
      for (int k = 0; k < 3; k++) {
        atomicMin(&a->glo[k], f2o(lv[k]));
        atomicMax(&a->ghi[k], f2o(hv[k]));
        atomicMin(&a->clo[k], f2o(lv[k] + hv[k]));
        atomicMax(&a->chi[k], f2o(lv[k] + hv[k]));
      }
      atomicAdd(&a->valid, 1u);
    }
  }
}

// ---------------------------------------------------------------- morton --

// bitInterleave (reference common/math/math.h:390-409)
__device__ inline uint32_t interleave3(uint32_t x) {
  x = (x | (x << 16)) & 0x030000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

__global__ __launch_bounds__(BT) void k_morton(const float4* __restrict__ lo4, const float4* __restrict__ hi4,
                                               uint32_t total, uint32_t* __restrict__ keys,
                                               uint32_t* __restrict__ vals, const BuildCounters* __restrict__ cnt,
                                               uint32_t* post, uint32_t seq) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (i < 64) post_words(post, seq, reinterpret_cast<const uint32_t*>(cnt), COUNTER_WORDS);
  if (i >= total) return;
  vals[i] = i;
  if (keys[i] == 0xffffffffu) return;
  const float4 l = lo4[i], h = hi4[i];
  const float c[3] = {l.x + h.x, l.y + h.y, l.z + h.z};
  uint32_t q[3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const float base = o2f(cnt->clo[k]);
    const float diag = o2f(cnt->chi[k]) - base;
    const float scale = diag > 1e-19f ? (1024.0f * 0.99f) / diag : 0.0f;
    float x = (c[k] - base) * scale;
    x = fminf(fmaxf(x, 0.0f), 1023.0f);
    q[k] = (uint32_t)x;
  }
  keys[i] = interleave3(q[0]) | (interleave3(q[1]) << 1) | (interleave3(q[2]) << 2);
}

// Where the scenes' roots come from: `stage` (pinned) holds their first
// positions, their primitive counts and the index of their tree.
struct RootArgs {
  uint32_t nscenes;           // 0: the roots are not placed yet
  const uint32_t* stage;
  const uint32_t* tree_root;  // null: the radix tree's root, node 0
  const uint32_t* tree_error;
  uint32_t* roots;            // binary references, first positions, primitive counts
  uint32_t* error;
};

// The boxes in position order; also no node visited yet, and the scenes' roots.
__global__ __launch_bounds__(BT) void k_gather_sorted(const uint32_t* __restrict__ vals,
                                                      const float4* __restrict__ lo4,
                                                      const float4* __restrict__ hi4, uint32_t n,
                                                      float4* __restrict__ slo, float4* __restrict__ shi,
                                                      uint32_t* __restrict__ visit, RootArgs ra) {
  const uint32_t j = blockIdx.x * BT + threadIdx.x;
  if (j < ra.nscenes) {
    const uint32_t f = ra.stage[j], c = ra.stage[ra.nscenes + j];
    uint32_t ref = c == 0u ? REF_EMPTY : f | REF_LEAF;
    if (c >= 2u) {
      ref = ra.tree_root ? ra.tree_root[ra.stage[2 * ra.nscenes + j]] : 0u;
      if (ref + 1u >= n || ref == REF_EMPTY) {
        atomicOr(ra.error, 256u);
        ref = 0u;
      }
    }
    ra.roots[j] = ref;
    ra.roots[ra.nscenes + j] = f;
    ra.roots[2 * ra.nscenes + j] = c;
    if (j == 0u && ra.tree_error && *ra.tree_error) atomicOr(ra.error, 256u);
  }
  if (j >= n) return;
  if (j + 1u < n || n == 1u) visit[j] = 0u;
  const uint32_t o = vals[j];
  slo[j] = lo4[o];
  shi[j] = hi4[o];
}

// ------------------------------------------------------- radix tree (LBVH) --

__device__ inline int delta(const uint32_t* __restrict__ keys, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  const uint32_t a = keys[i], b = keys[j];
  if (a != b) return __clz(a ^ b);
  return 32 + __clz((uint32_t)i ^ (uint32_t)j);
}

// Binary radix tree over sorted keys (Karras, HPG 2012): inner node i covers
// a contiguous range of sorted primitives and splits it where the highest
// differing key bit changes.
__global__ __launch_bounds__(BT) void k_radix_tree(const uint32_t* __restrict__ keys, int n,
                                                   uint32_t* __restrict__ child, uint32_t* __restrict__ parent_int,
                                                   uint32_t* __restrict__ parent_leaf, uint2* __restrict__ range) {
  const int i = blockIdx.x * BT + threadIdx.x;
  if (i >= n - 1) return;
  const int d = (delta(keys, n, i, i + 1) - delta(keys, n, i, i - 1)) >= 0 ? 1 : -1;
  const int dmin = delta(keys, n, i, i - d);
  int lmax = 2;
  while (delta(keys, n, i, i + lmax * d) > dmin) lmax <<= 1;
  int l = 0;
  for (int t = lmax >> 1; t >= 1; t >>= 1)
    if (delta(keys, n, i, i + (l + t) * d) > dmin) l += t;
  const int j = i + l * d;
  const int dnode = delta(keys, n, i, j);
  int s = 0, t = l;
  while (true) {
    t = (t + 1) >> 1;
    if (delta(keys, n, i, i + (s + t) * d) > dnode) s += t;
    if (t <= 1) break;
  }
  const int gamma = i + s * d + (d < 0 ? -1 : 0);
  if (gamma < 0 || gamma + 1 >= n) return;  // impossible for sorted keys; keeps writes in bounds
  const int first = i < j ? i : j, last = i < j ? j : i;
  const uint32_t left = (first == gamma) ? ((uint32_t)gamma | REF_LEAF) : (uint32_t)gamma;
  const uint32_t right = (last == gamma + 1) ? ((uint32_t)(gamma + 1) | REF_LEAF) : (uint32_t)(gamma + 1);
  child[2 * i] = left;
  child[2 * i + 1] = right;
  if (left & REF_LEAF) parent_leaf[left & ~REF_LEAF] = i; else parent_int[left] = i;
  if (right & REF_LEAF) parent_leaf[right & ~REF_LEAF] = i; else parent_int[right] = i;
  range[i] = make_uint2((uint32_t)first, (uint32_t)last);
  if (i == 0) parent_int[0] = NONE;
}

__device__ inline float box_half_area(float4 l, float4 h) { return half_area(h.x - l.x, h.y - l.y, h.z - l.z); }


// Bottom-up bounds and the SAH-optimal 8-wide collapse table, each node after
// its two children.
// For every binary node n and slot budget s = 1..8, cost8 holds
// the least SAH cost of covering n's subtree with at most s subtrees:
//   c(n,1) = min(leaf: cost_tri*count*A(n), node: cost_node*A(n) + d(n,8))
//   d(n,s) = min_j c(left,j) + c(right,s-j)      (s >= 2)
//   c(n,s) = min(c(n,s-1), d(n,s))
// split8 records, per s, the best j (low 3 bits) and whether fewer slots win
// (bit 7). A binary leaf costs cost_tri*A(prim) whatever the budget.
// (Collapse formulation after Ylitie, Karras, Laine: "Efficient Incoherent
// Ray Traversal on GPUs Through Compressed Wide BVHs", HPG 2017.)
// A node's width is capped at `width` children (d(n, width) in the inner cost).
// Bottom-up step of one inner node: box of its two children, and the
// SAH-optimal way to spend 1..8 child slots below it (the 8-wide collapse
// DP): cost8[s-1] = least cost of covering the subtree with s slots,
// split8[s-1] = how many of them go left (0x80: fewer slots do as well),
// isleaf = a leaf beats an inner node. Returns false on a broken link.
struct RefitArgs {
  uint32_t n;
  const uint32_t* child;
  const uint2* range;
  const float4* slo;
  const float4* shi;
  float4* nlo;
  float4* nhi;
  float* cost8;
  uint8_t* split8;
  uint8_t* isleaf;
  float cost_node, cost_tri;
  uint32_t max_leaf, width, min_leaf, block;
  uint32_t* err;
};

// `inner(c, slot, lo, hi, cost)` reads finished inner child number `slot` (0 or 1),
// and `keep(lo, hi, cost)` gets the node's own box and costs.
template <class Inner, class Keep>
__device__ inline bool refit_node(const RefitArgs& a, uint32_t node, uint2 ch, uint32_t count, Inner inner_child,
                                  Keep keep) {
  const uint32_t n = a.n;
  const float cost_node = a.cost_node, cost_tri = a.cost_tri;
  const uint32_t max_leaf = a.max_leaf, width = a.width, min_leaf = a.min_leaf, block = a.block;
  float4 bl[2], bh[2];
  float cc[2][8];
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const uint32_t c = k ? ch.y : ch.x;
    if ((c & REF_LEAF) ? (c & ~REF_LEAF) >= n : c + 1 >= n) {
      atomicOr(a.err, 1u);
      return false;
    }
    if (c & REF_LEAF) {
      bl[k] = a.slo[c & ~REF_LEAF];
      bh[k] = a.shi[c & ~REF_LEAF];
      const float ct = cost_tri * box_half_area(bl[k], bh[k]);
#pragma unroll
      for (int s = 0; s < 8; s++) cc[k][s] = ct;
    } else {
      inner_child(c, k, bl[k], bh[k], cc[k]);
    }
  }
  const float4 l = make_float4(fminf(bl[0].x, bl[1].x), fminf(bl[0].y, bl[1].y), fminf(bl[0].z, bl[1].z), 0.0f);
  const float4 h = make_float4(fmaxf(bh[0].x, bh[1].x), fmaxf(bh[0].y, bh[1].y), fmaxf(bh[0].z, bh[1].z), 0.0f);
  const float A = box_half_area(l, h);
  float d[9];
  uint32_t dj[9];
#pragma unroll
  for (int s = 2; s <= 8; s++) {
    float best = INFINITY;
    uint32_t bj = 1;
#pragma unroll
    for (int jj = 1; jj < s; jj++) {
      const float v = cc[0][jj - 1] + cc[1][s - jj - 1];
      if (v < best) { best = v; bj = (uint32_t)jj; }
    }
    d[s] = best;
    dj[s] = bj;
  }
  // a leaf pays per block of `block` primitives (the reference's
  // sahBlockSize); subtrees of at most min_leaf primitives are leaves
  const float leafc = count <= max_leaf ? cost_tri * (float)((count + block - 1) / block) * A : INFINITY;
  const float inner = count <= min_leaf ? INFINITY : cost_node * A + d[width];  // at most `width` children
  float c[8];
  uint32_t sp[8];
  c[0] = fminf(leafc, inner);
  sp[0] = 0;
#pragma unroll
  for (int s = 2; s <= 8; s++) {
    if (d[s] < c[s - 2]) { c[s - 1] = d[s]; sp[s - 1] = dj[s]; }
    else { c[s - 1] = c[s - 2]; sp[s - 1] = 0x80u | dj[s]; }
  }
  a.nlo[node] = l;
  a.nhi[node] = h;
  keep(l, h, c);
  uint2* sp8 = reinterpret_cast<uint2*>(a.split8 + 8 * (size_t)node);
  *sp8 = make_uint2(sp[0] | (sp[1] << 8) | (sp[2] << 16) | (sp[3] << 24),
                    sp[4] | (sp[5] << 8) | (sp[6] << 16) | (sp[7] << 24));
  a.isleaf[node] = leafc <= inner ? 1 : 0;
  return true;
}

// A node's costs in HBM, for a parent that another workgroup finishes.
__device__ inline void put_cost(const RefitArgs& a, uint32_t node, const float c[8]) {
  float4* t = reinterpret_cast<float4*>(a.cost8 + 8 * (size_t)node);
  t[0] = make_float4(c[0], c[1], c[2], c[3]);
  t[1] = make_float4(c[4], c[5], c[6], c[7]);
}
__device__ inline void get_node(const RefitArgs& a, uint32_t node, float4& l, float4& h, float c[8]) {
  l = a.nlo[node];
  h = a.nhi[node];
  const float4* t = reinterpret_cast<const float4*>(a.cost8 + 8 * (size_t)node);
  const float4 t0 = t[0], t1 = t[1];
  c[0] = t0.x; c[1] = t0.y; c[2] = t0.z; c[3] = t0.w;
  c[4] = t1.x; c[5] = t1.y; c[6] = t1.z; c[7] = t1.w;
}

// What a workgroup keeps of its nodes in LDS, so that a parent's step waits
// neither for its links nor for its children's results from HBM, and only the
// costs that another workgroup reads are written there (56 B a node kept, 76 KB
// a workgroup, two of them on a CU; Morton builds of 2^20 triangles 0.815 ->
// 0.744 ms, of 20,000 0.226 -> 0.217).
template <uint32_t N>
struct RefitKept {
  float v[14][N];  // box lo, hi, costs of 1..8 slots
  uint2 child[N];
  uint16_t parent[N];
  __device__ inline void put(uint32_t i, float4 l, float4 h, const float c[8]) {
    v[0][i] = l.x; v[1][i] = l.y; v[2][i] = l.z;
    v[3][i] = h.x; v[4][i] = h.y; v[5][i] = h.z;
#pragma unroll
    for (int k = 0; k < 8; k++) v[6 + k][i] = c[k];
  }
  __device__ inline void get(uint32_t i, float4& l, float4& h, float c[8]) const {
    l = make_float4(v[0][i], v[1][i], v[2][i], 0.0f);
    h = make_float4(v[3][i], v[4][i], v[5][i], 0.0f);
#pragma unroll
    for (int k = 0; k < 8; k++) c[k] = v[6 + k][i];
  }
};

// Bottom-up order without a launch per depth: an inner node's id lies in its
// range of positions, in the radix tree as in the binned-SAH tree, so the nodes
// whose range stays within one chunk of REFIT_CHUNK positions form subtrees
// that one workgroup can finish alone, each node once both of its children are
// done. The nodes that span chunks (a boundary is crossed by one path, fewer
// than 70 nodes) go to lists, and the next launch does the same for REFIT_FAN
// chunks at a time. No workgroup waits on another. A tree of 2^20 primitives
// takes three launches, one of 20,000 two, where a launch per depth level took
// 25, with the nodes sorted by depth and a read-back of the level sizes before
// (Morton builds of 20,000 triangles: 0.56 -> 0.48 ms, of 4.2 M: 3.00 -> 2.82).
// What bounds the pass on small trees is the chain of levels, 0.7 us each.
constexpr uint32_t REFIT_CHUNK = 1024, REFIT_FAN = 32;
constexpr uint32_t SPAN_KEPT = 1024;   // and those of them that it keeps in LDS
constexpr uint32_t REFIT_SPAN = 4608;  // listed nodes a workgroup takes (32 chunks of at most 2 x 70)

// Nodes that became ready in round r are in list r % 2, their count in r % 3
// (the third is cleared meanwhile), so a round needs one barrier.
struct RefitReady {
  uint32_t count[3];
};

__global__ __launch_bounds__(BT) void k_refit_chunk(RefitArgs a, const uint32_t* __restrict__ parent_int,
                                                    uint32_t* visit, uint32_t* __restrict__ list,
                                                    uint32_t* __restrict__ list_count) {
  __shared__ uint32_t need[REFIT_CHUNK];  // inner children still to come
  __shared__ uint16_t ready[2][REFIT_CHUNK];
  __shared__ RefitReady rd;
  __shared__ uint32_t nlist;
  __shared__ RefitKept<REFIT_CHUNK> kept;
  __shared__ uint16_t count[REFIT_CHUNK];
  const uint32_t base = blockIdx.x * REFIT_CHUNK, m = a.n - 1u;
  if (threadIdx.x < 3) rd.count[threadIdx.x] = 0u;
  if (threadIdx.x == 0) nlist = 0u;
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < REFIT_CHUNK; k += BT) {
    const uint32_t id = base + k;
    need[k] = 3u;  // never reaches 0: no node, or one of the list
    const uint32_t parent = id < m ? parent_int[id] : REF_EMPTY;
    if (parent == REF_EMPTY) continue;
    const uint2 r = a.range[id];
    if (r.x >= base && r.y - base < REFIT_CHUNK) {
      const uint2 ch = *reinterpret_cast<const uint2*>(a.child + 2 * (size_t)id);
      const uint32_t inner = (ch.x & REF_LEAF ? 0u : 1u) + (ch.y & REF_LEAF ? 0u : 1u);
      need[k] = inner;
      kept.child[k] = ch;
      kept.parent[k] = (uint16_t)min(parent - base, REFIT_CHUNK);  // (REFIT_CHUNK: not in the chunk)
      count[k] = (uint16_t)(r.y - r.x + 1u);
      if (inner == 0u) ready[0][atomicAdd(&rd.count[0], 1u)] = (uint16_t)k;
    } else {
      list[base + atomicAdd(&nlist, 1u)] = id;
    }
  }
  for (uint32_t round = 0;; round++) {
    __syncthreads();
    const uint32_t cnt = rd.count[round % 3u];
    if (cnt == 0u) break;
    if (threadIdx.x == 0) rd.count[(round + 2u) % 3u] = 0u;
    for (uint32_t t = threadIdx.x; t < cnt; t += BT) {
      const uint32_t k = ready[round & 1u][t], id = base + k;
      const uint32_t p = kept.parent[k];
      // (need is 3 where the parent is left to a later launch: only those children's costs are read from HBM)
      const bool local = p < REFIT_CHUNK && need[p] != 3u;
      const bool ok = refit_node(
          a, id, kept.child[k], count[k],
          [&](uint32_t c, int, float4& l, float4& h, float* cost) { kept.get(min(c - base, REFIT_CHUNK - 1u), l, h, cost); },
          [&](float4 l, float4 h, const float* cost) {
            if (local) kept.put(k, l, h, cost);
            else put_cost(a, id, cost);
          });
      if (!ok) continue;
      visit[id] = 2u;  // what the tree check expects of a refitted node
      if (local && atomicSub(&need[p], 1u) == 1u)
        ready[(round + 1u) & 1u][atomicAdd(&rd.count[(round + 1u) % 3u], 1u)] = (uint16_t)p;
    }
  }
  if (threadIdx.x == 0) list_count[blockIdx.x] = nlist;
}

// The listed nodes of REFIT_FAN lists (of `cap` positions each, nlists in all);
// those that span further go to this workgroup's list. While a node waits,
// visit holds 4 + its slot, so that a finished child finds it.
__global__ __launch_bounds__(BT) void k_refit_span(RefitArgs a, const uint32_t* __restrict__ parent_int,
                                                   uint32_t* visit, const uint32_t* __restrict__ in,
                                                   const uint32_t* __restrict__ in_count, uint32_t cap,
                                                   uint32_t nlists, uint32_t* __restrict__ out,
                                                   uint32_t* __restrict__ out_count) {
  __shared__ uint32_t ids[REFIT_SPAN], need[REFIT_SPAN];
  __shared__ uint16_t ready[2][REFIT_SPAN];
  __shared__ RefitReady rd;
  __shared__ uint32_t nids, nout;
  __shared__ RefitKept<SPAN_KEPT> kept;
  __shared__ uint16_t cslot[2][SPAN_KEPT];  // slots of the children that are in this workgroup
  __shared__ uint32_t count[SPAN_KEPT];
  const uint64_t base = (uint64_t)blockIdx.x * REFIT_FAN * cap, end = base + (uint64_t)REFIT_FAN * cap;
  const uint32_t m = a.n - 1u;
  if (threadIdx.x < 3) rd.count[threadIdx.x] = 0u;
  if (threadIdx.x == 0) nids = nout = 0u;
  __syncthreads();
  // eight threads a list
  {
    const uint32_t l = blockIdx.x * REFIT_FAN + threadIdx.x / (BT / REFIT_FAN);
    const uint32_t cnt = l < nlists ? min(in_count[l], cap) : 0u;
    for (uint32_t e = threadIdx.x % (BT / REFIT_FAN); e < cnt; e += BT / REFIT_FAN) {
      const uint32_t id = in[(uint64_t)l * cap + e];
      if (id >= m) continue;
      const uint2 r = a.range[id];
      uint32_t slot = REFIT_SPAN;
      if (r.x >= base && r.y < end) slot = atomicAdd(&nids, 1u);
      if (slot < REFIT_SPAN) {
        ids[slot] = id;
        visit[id] = 4u + slot;
      } else {
        out[base + atomicAdd(&nout, 1u)] = id;
        visit[id] = 0u;
      }
    }
  }
  __syncthreads();
  const uint32_t n = min(nids, REFIT_SPAN);
  // the slot of an inner node, REFIT_SPAN if it is not one of this workgroup's
  auto slot_of = [&](uint32_t id) {
    const uint32_t at = id < m ? visit[id] - 4u : REFIT_SPAN;
    return at < n && ids[at] == id ? at : REFIT_SPAN;
  };
  for (uint32_t k = threadIdx.x; k < n; k += BT) {
    const uint32_t id = ids[k];
    const uint2 ch = *reinterpret_cast<const uint2*>(a.child + 2 * (size_t)id);
    uint32_t wait = 0u;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const uint32_t c = j ? ch.y : ch.x;
      uint32_t at = SPAN_KEPT;
      if (!(c & REF_LEAF)) {
        const uint32_t v = c < m ? visit[c] : 0u;
        if (v != 2u) wait++;
        if (v >= 4u && v - 4u < n && ids[v - 4u] == c) at = min(v - 4u, SPAN_KEPT);
      }
      if (k < SPAN_KEPT) cslot[j][k] = (uint16_t)at;
    }
    if (k < SPAN_KEPT) {
      const uint2 r = a.range[id];
      kept.child[k] = ch;
      kept.parent[k] = (uint16_t)slot_of(parent_int[id]);
      count[k] = r.y - r.x + 1u;
    }
    need[k] = wait;
    if (wait == 0u) ready[0][atomicAdd(&rd.count[0], 1u)] = (uint16_t)k;
  }
  for (uint32_t round = 0;; round++) {
    __syncthreads();
    const uint32_t cnt = rd.count[round % 3u];
    if (cnt == 0u) break;
    if (threadIdx.x == 0) rd.count[(round + 2u) % 3u] = 0u;
    for (uint32_t t = threadIdx.x; t < cnt; t += BT) {
      const uint32_t k = ready[round & 1u][t], id = ids[k];
      uint2 ch;
      uint32_t p, cnt, at[2] = {SPAN_KEPT, SPAN_KEPT};
      if (k < SPAN_KEPT) {
        ch = kept.child[k];
        p = kept.parent[k];
        cnt = count[k];
        at[0] = cslot[0][k];
        at[1] = cslot[1][k];
      } else {
        const uint2 r = a.range[id];
        ch = *reinterpret_cast<const uint2*>(a.child + 2 * (size_t)id);
        p = slot_of(parent_int[id]);
        cnt = r.y - r.x + 1u;
      }
      const bool ok = refit_node(
          a, id, ch, cnt,
          [&](uint32_t c, int j, float4& l, float4& h, float* cost) {
            if (at[j] < SPAN_KEPT) kept.get(at[j], l, h, cost);
            else get_node(a, c, l, h, cost);
          },
          [&](float4 l, float4 h, const float* cost) {
            if (k < SPAN_KEPT) kept.put(k, l, h, cost);
            put_cost(a, id, cost);
          });
      if (!ok) continue;
      visit[id] = 2u;
      if (p < n && atomicSub(&need[p], 1u) == 1u)
        ready[(round + 1u) & 1u][atomicAdd(&rd.count[(round + 1u) % 3u], 1u)] = (uint16_t)p;
    }
  }
  if (threadIdx.x == 0) out_count[blockIdx.x] = nout;
}

// Integrity check of the sorted keys and the radix tree (cheap, one pass):
// bit 3 keys out of order, bit 4 inner node not finished by the refit,
// bit 5 parent/child links disagree.
__global__ __launch_bounds__(BT) void k_check_tree(const uint32_t* __restrict__ keys, uint32_t n, uint32_t* roots_seen,
                                                   const uint32_t* __restrict__ child,
                                                   const uint32_t* __restrict__ parent_int,
                                                   const uint32_t* __restrict__ parent_leaf,
                                                   const uint32_t* __restrict__ visit, uint32_t* err) {
  const uint32_t i = blockIdx.x * BT + threadIdx.x;
  if (keys && i + 1 < n && keys[i] > keys[i + 1]) atomicOr(err, 8u);
  if (i < n) {
    const uint32_t p = parent_leaf[i];
    if (p == NONE) atomicAdd(roots_seen, 1u);  // a scene of one primitive
    else if (p >= n - 1 || (child[2 * p] != (i | REF_LEAF) && child[2 * p + 1] != (i | REF_LEAF))) atomicOr(err, 32u);
  }
  if (i + 1 < n && parent_int[i] != REF_EMPTY) {
    if (visit[i] != 2u) atomicOr(err, 16u);
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const uint32_t c = child[2 * i + k];
      const bool ok = (c & REF_LEAF) ? ((c & ~REF_LEAF) < n && parent_leaf[c & ~REF_LEAF] == i)
                                     : (c + 1 < n && parent_int[c] == i);
      if (!ok) atomicOr(err, 32u);
    }
    if (parent_int[i] == NONE) {
      atomicAdd(roots_seen, 1u);
    } else {
      const uint32_t p = parent_int[i];
      if (p >= n - 1 || (child[2 * p] != i && child[2 * p + 1] != i)) atomicOr(err, 32u);
    }
  }
}

// ---------------------------------------------------------------- collapse --

// The binary tree and its collapse table as the walk and the emission read them.
struct CollapseArgs {
  const uint32_t* child;
  const uint2* range;
  const float4* nlo;
  const float4* nhi;
  const uint8_t* isleaf;
  const uint8_t* split8;
  const float4* slo;
  const float4* shi;
  BuildCounters* cnt;
  uint32_t nscenes;
  uint32_t n;         // primitives
  uint32_t width;     // children per node (2..8)
  uint32_t max_sub;   // subtrees that the arrays below hold
  WideNode* top;      // top node i
  WideNode* sub;      // roots of the subtrees, waiting
  WideNode* rest;     // node i of subtree f at sub[f].tri + i
  uint32_t* count;    // nodes of each subtree without its root, and (prefix) their exclusive sums
  const uint32_t* prefix;
  QNode8* nodes;
  uint32_t* leaf_src; // position of each leaf record's primitive, bit 31: last of its leaf
  NodeInfo* info;
  uint32_t cap;       // capacity of nodes
  struct CollapseStats* stats;  // of each workgroup of the emission
};

constexpr uint32_t LEAF_SRC_LAST = 0x80000000u;  // positions are below 2^31 (REF_LEAF marks them likewise)

__device__ inline bool is_inner(uint32_t ref, const uint8_t* isleaf) {
  return !(ref & REF_LEAF) && !isleaf[ref];
}

// Quantises one axis: returns the biased exponent byte of the grid step.
__device__ inline uint32_t grid_exponent(float p, float hi) {
  const float ext = hi - p;
  int eb = (int)((__float_as_uint(ext) >> 23) & 0xff) - 7;
  if (eb < 1) eb = 1;
  for (int it = 0; it < 64 && eb < 254; it++) {
    const float s = __uint_as_float((uint32_t)eb << 23);
    if (__builtin_fmaf(s, 254.0f, p) >= hi) break;
    eb++;
  }
  return (uint32_t)eb;
}

__device__ inline uint32_t quant_lo(float v, float p, float s) {
  float q = floorf((v - p) / s);
  q = fminf(fmaxf(q, 0.0f), 255.0f);
  uint32_t qi = (uint32_t)q;
  while (qi > 0 && __builtin_fmaf(s, (float)qi, p) > v) qi--;
  return qi;
}
__device__ inline uint32_t quant_hi(float v, float p, float s) {
  float q = ceilf((v - p) / s);
  q = fminf(fmaxf(q, 0.0f), 255.0f);
  uint32_t qi = (uint32_t)q;
  while (qi < 255 && __builtin_fmaf(s, (float)qi, p) < v) qi++;
  return qi;
}

// Byte k of a node's eight split bytes loaded as one uint2.
__device__ inline uint32_t split_byte(uint2 s8, uint32_t k) { return ((k < 4 ? s8.x : s8.y) >> (8 * (k & 3))) & 0xffu; }

// A wide node takes a group of CG lanes: they find its children together, lane k
// keeps child k.
constexpr uint32_t CG = 8;

template <class T>
__device__ inline T group_sum(T v) {
#pragma unroll
  for (int d = 1; d < (int)CG; d <<= 1) v += __shfl_xor(v, d, CG);
  return v;
}
__device__ inline float group_min(float v) {
#pragma unroll
  for (int d = 1; d < (int)CG; d <<= 1) v = fminf(v, __shfl_xor(v, d, CG));
  return v;
}
__device__ inline float group_max(float v) {
#pragma unroll
  for (int d = 1; d < (int)CG; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, CG));
  return v;
}
// exclusive prefix over the group's lanes
__device__ inline uint32_t group_prefix(uint32_t v, uint32_t k) {
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < (int)CG; d <<= 1) {
    const uint32_t y = __shfl_up(x, d, CG);
    if (k >= (uint32_t)d) x += y;
  }
  return x - v;
}

// The children of a wide node: the optimal distribution of `width` slots below
// inner node b. Lane k of the group gets child k in `mine`; returns their
// number, 0 on a corrupt table. A lane that holds a reference has the slots from
// its own place up to the next such lane's; in each round every reference with
// more than one slot is split, the right part going to the lane at the left
// part's end. So the chain of loads is as long as the deepest child, not as the
// number of splits (up to 7, each about 0.8 us): with one lane a node that did
// them in turn, Morton builds of 20,000 triangles took 0.29 ms, now 0.23, of
// 2^20 0.88, now 0.81.
__device__ inline int wide_children(const CollapseArgs& a, uint32_t b, uint32_t k, uint32_t& mine) {
  const uint32_t shift = (threadIdx.x & 63u) & ~(CG - 1u);
  auto group = [&](bool x) { return (uint32_t)(__ballot(x) >> shift) & 0xffu; };
  const uint32_t j8 = a.split8[8 * (size_t)b + a.width - 1] & 7u;
  const uint2 bc = *reinterpret_cast<const uint2*>(a.child + 2 * (size_t)b);
  uint32_t ref = k ? bc.y : bc.x;
  uint32_t slots = k == 0u ? j8 : (k == j8 ? a.width - j8 : 0u);
  bool bad = j8 == 0u || j8 >= a.width;
  bool open = slots > 1u && !(ref & REF_LEAF);
  while (group(open)) {
    uint32_t left = 0u, right = 0u, rref = 0u;  // slots of the parts
    if (open) {
      // the node's eight split bytes and its child pair: two 8 B loads
      const uint2 s8 = *reinterpret_cast<const uint2*>(a.split8 + 8 * (size_t)ref);
      const uint2 cp = *reinterpret_cast<const uint2*>(a.child + 2 * (size_t)ref);
      while (slots > 1u && (split_byte(s8, slots - 1) & 0x80u)) slots--;
      if (slots > 1u) {
        left = split_byte(s8, slots - 1) & 7u;
        bad = bad || left == 0u || left >= slots;
        right = slots - left;
        rref = cp.y;
        ref = cp.x;
        slots = left;
      }
    }
    // the lane whose slots include this one: the last at or before it
    const uint32_t held = group(slots > 0u) & ((2u << k) - 1u);
    const uint32_t from = held ? 31u - (uint32_t)__builtin_clz(held) : 0u;
    const uint32_t fl = (uint32_t)__shfl((int)left, (int)from, CG), fr = (uint32_t)__shfl((int)right, (int)from, CG);
    const uint32_t fref = (uint32_t)__shfl((int)rref, (int)from, CG);
    if (slots == 0u && fr != 0u && from + fl == k) {
      ref = fref;
      slots = fr;
      open = true;
    }
    open = open && slots > 1u && !(ref & REF_LEAF);
    if (group(bad)) break;
  }
  if (group(bad)) {
    if (k == 0) atomicOr(&a.cnt->error, 128u);
    return 0;
  }
  // child k: the k-th lane that holds a reference
  uint32_t held = group(slots > 0u);
  const int n = __builtin_popcount(held);
  for (uint32_t i = 0; i < k && (held & (held - 1u)); i++) held &= held - 1u;
  mine = (uint32_t)__shfl((int)ref, __builtin_ctz(held), CG);
  return n;
}

// The collapse numbers the wide nodes first (the walk: only links, counts and
// leaf flags are read) and then writes them all at once (the emission: boxes
// and quantisation). A wide node owns as many leaf records as it has
// primitives: its leaves take the first, its inner children the rest in turn.
// Node numbers need a counter, which lives in LDS: one workgroup walks the top
// of the tree, then each subtree has a workgroup, and the subtrees' node counts
// are summed before the emission. (A launch for each level with its slots from
// counters in HBM took 28 us a level on small trees, and on large ones the
// atomics of all workgroups on those counters passed one at a time, about
// 40 ns each: 2^20 triangles 1.20 -> 0.95 ms for a Morton build, 3.20 -> 2.96
// for binned SAH; 131,000 triangles 0.68 -> 0.50 and 1.46 -> 1.33 ms.)
// The top is every node with more than 1/256 of the primitives, so fewer than
// 256 on a level (eight lanes each), and the subtrees take about the same time.
constexpr uint32_t TOP_SHARE = 256, TOP_LEVELS = 256;
// Primitives that are always one subtree (Morton builds of 131,000 terrain
// triangles 0.347 ms, at 512 0.388, at 4096 0.356; of 20,000 0.225, 0.229, 0.228).
constexpr uint32_t TOP_MIN = 2048;
constexpr uint32_t SUB_MAX = 2047;  // subtrees beside the scenes (their sums are one scan launch)
// Top nodes: fewer than TOP_SHARE on each level, the subtrees' roots, the scenes.
__host__ __device__ inline uint32_t top_cap(uint32_t max_sub) { return max_sub + TOP_SHARE * TOP_LEVELS; }

// Walks one wide node with a group: `take` gives lane 0 the first of ni numbers
// for its inner children, `put` gets each of those (in its own lane) with its
// primitive count, and `record` (in lane 0) the first number, for the node's own
// record.
template <class Take, class Put, class Record>
__device__ inline void walk_node(const CollapseArgs& a, const WideNode& w, uint32_t k, Take take, Put put,
                                 Record record) {
  uint32_t ref = REF_EMPTY;
  int n = 0;
  if (w.bref != REF_EMPTY && is_inner(w.bref, a.isleaf)) n = wide_children(a, w.bref, k, ref);
  uint32_t cnt = 0u;
  bool in = false;
  if (k < (uint32_t)n) {
    cnt = 1u;
    if (!(ref & REF_LEAF)) {
      const uint2 r = a.range[ref];
      cnt = r.y - r.x + 1u;
      in = !a.isleaf[ref];
    }
  }
  const uint32_t nt = group_sum(in ? 0u : cnt), ni = group_sum(in ? 1u : 0u);
  const uint32_t tri = w.tri + nt + group_prefix(in ? cnt : 0u, k), rank = group_prefix(in ? 1u : 0u, k);
  uint32_t first = 0u;
  if (k == 0u && ni) first = take(ni);
  first = (uint32_t)__shfl((int)first, 0, CG);
  const uint32_t level = w.level + (1u << 16) + (n ? (uint32_t)n - 1u : 0u);  // a node pushes at most n-1 of its n children
  if (in) put(cnt, WideNode{ref, tri, level, first + rank});
  if (k == 0u) record(first);
}

constexpr int WT = 1024;  // lanes of a workgroup that walks: 128 nodes at a time

__global__ __launch_bounds__(WT) void k_walk_top(CollapseArgs a, const uint32_t* __restrict__ roots,
                                                 const uint32_t* __restrict__ first,
                                                 const uint32_t* __restrict__ prims) {
  __shared__ WideNode level[2][TOP_SHARE];
  __shared__ uint32_t nlevel[2], nodes, nsub, run;
  if (threadIdx.x == 0) {
    run = a.cnt->error ? 0u : 1u;  // a tree that failed its check is not followed
    nodes = a.nscenes;
    nsub = nlevel[0] = nlevel[1] = 0u;
  }
  __syncthreads();
  if (!run) return;
  uint32_t in = 0;
  const uint32_t share = max(a.n / TOP_SHARE, TOP_MIN);
  // a wide node joins the next level's list or the subtrees
  auto place = [&](uint32_t to, uint32_t cnt, const WideNode& w) {
    if (cnt > share) {
      const uint32_t at = atomicAdd(&nlevel[to], 1u);
      if (at < TOP_SHARE) level[to][at] = w;
      else atomicOr(&a.cnt->error, 2u);
    } else {
      const uint32_t at = atomicAdd(&nsub, 1u);
      if (at < a.max_sub) a.sub[at] = w;
      else atomicOr(&a.cnt->error, 2u);
    }
  };
  for (uint32_t i = threadIdx.x; i < a.nscenes; i += WT) place(0, prims[i], WideNode{roots[i], first[i], 1u << 16, i});
  __syncthreads();
  while (true) {
    // (each walked node may add 8 subtrees; every wave decides before any adds one)
    const uint32_t count = min(nlevel[in], TOP_SHARE);
    const bool last = count == 0u || nsub + 8u * count > a.max_sub;
    __syncthreads();
    if (last) break;
    for (uint32_t i = threadIdx.x / CG; i < count; i += WT / CG) {
      const WideNode w = level[in][i];
      walk_node(
          a, w, threadIdx.x % CG, [&](uint32_t ni) { return atomicAdd(&nodes, ni); },
          [&](uint32_t cnt, const WideNode& c) { place(in ^ 1u, cnt, c); },
          [&](uint32_t f) {
            if (w.link < top_cap(a.max_sub)) a.top[w.link] = WideNode{w.bref, w.tri, w.level, f};
            else atomicOr(&a.cnt->error, 2u);
          });
    }
    __syncthreads();
    if (threadIdx.x == 0) nlevel[in] = 0u;
    in ^= 1u;
    __syncthreads();
  }
  // (of unusually narrow trees) the level that was not walked
  const uint32_t count = min(nlevel[in], TOP_SHARE);
  if (threadIdx.x < count && nsub + threadIdx.x < a.max_sub) a.sub[nsub + threadIdx.x] = level[in][threadIdx.x];
  if (threadIdx.x == 0) {
    a.cnt->top_nodes = nodes;
    a.cnt->subtrees = min(nsub + count, a.max_sub);
  }
}

// The subtrees, a workgroup each: up to 128 waiting nodes are walked at a time,
// last first, from a stack in LDS. Where the stack could fill up, fewer are
// taken, down to one, which needs 7 entries a level.
constexpr uint32_t REST_STACK = 3072, REST_SPARE = 7 * 128;

__global__ __launch_bounds__(WT) void k_walk_rest(CollapseArgs a) {
  __shared__ WideNode stack[REST_STACK];
  __shared__ uint32_t count, nodes, run;
  if (threadIdx.x == 0) run = a.cnt->error ? 0u : 1u;
  __syncthreads();
  const uint32_t nsub = run ? a.cnt->subtrees : 0u;
  for (uint32_t f = blockIdx.x; f <= a.max_sub; f += gridDim.x) {
    if (f >= nsub) {  // (the sums run over all of the array)
      if (threadIdx.x == 0) a.count[f] = 0u;
      continue;
    }
    const WideNode root = a.sub[f];
    if (threadIdx.x == 0) {
      stack[0] = root;
      count = 1u;
      nodes = 0u;
    }
    __syncthreads();
    for (bool top = true;; top = false) {
      const uint32_t c = count;
      if (c == 0u) break;
      const uint32_t room = REST_STACK - REST_SPARE > c ? (REST_STACK - REST_SPARE - c) / 7u : 0u;
      const uint32_t m = min(min(c, WT / CG), max(room, 1u));
      const uint32_t g = threadIdx.x / CG;
      WideNode w{};
      if (g < m) w = stack[c - 1u - g];
      __syncthreads();
      if (threadIdx.x == 0) count = c - m;
      __syncthreads();
      if (g < m) {
        walk_node(
            a, w, threadIdx.x % CG, [&](uint32_t ni) { return atomicAdd(&nodes, ni); },
            [&](uint32_t, const WideNode& ch) {
              const uint32_t at = atomicAdd(&count, 1u);
              if (at < REST_STACK) stack[at] = ch;
              else atomicOr(&a.cnt->error, 2u);
            },
            [&](uint32_t i) {
              if (top && root.link < top_cap(a.max_sub)) a.top[root.link] = WideNode{w.bref, w.tri, w.level, REF_LEAF | f};
              else if (!top && root.tri + w.link < a.n) a.rest[root.tri + w.link] = WideNode{w.bref, w.tri, w.level, i};
              else atomicOr(&a.cnt->error, 2u);
            });
      }
      __syncthreads();
      if (threadIdx.x == 0 && count > REST_STACK) count = 0u;  // (reported above)
      __syncthreads();
    }
    if (threadIdx.x == 0) a.count[f] = nodes;
    __syncthreads();
  }
}

// Statistics of the nodes that a thread, then a workgroup, wrote.
struct CollapseStats {
  uint32_t max_depth = 0, max_stack = 0, records = 0;
  double sah_nodes = 0.0, sah_leaves = 0.0, sah_leaves_tri = 0.0;
  __device__ void add(const CollapseStats& o) {
    max_depth = max(max_depth, o.max_depth);
    max_stack = max(max_stack, o.max_stack);
    records += o.records;
    sah_nodes += o.sah_nodes;
    sah_leaves += o.sah_leaves;
    sah_leaves_tri += o.sah_leaves_tri;
  }
};

// The workgroup's statistics, in thread 0.
__device__ inline void block_stats(CollapseStats& st) {
  __shared__ __align__(8) char mem[BT / 64 * sizeof(CollapseStats)];
  CollapseStats* w = reinterpret_cast<CollapseStats*>(mem);
  st.max_depth = wave_umax(st.max_depth);
  st.max_stack = wave_umax(st.max_stack);
  st.records = wave_sum(st.records);
  st.sah_nodes = wave_sum(st.sah_nodes);
  st.sah_leaves = wave_sum(st.sah_leaves);
  st.sah_leaves_tri = wave_sum(st.sah_leaves_tri);
  if ((threadIdx.x & 63u) == 0u) w[threadIdx.x >> 6] = st;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = 1; i < BT / 64; i++) st.add(w[i]);
}

// Writes node number `number` (w.link: the number of its first inner child).
__device__ inline void emit_node(const CollapseArgs& a, const WideNode& w, uint32_t number, uint32_t k, CollapseStats& st) {
  const float eps = o2f(a.cnt->maxabs) * BOX_EPS_REL;
  const uint32_t depth = w.level >> 16;
  if (number >= a.cap) {
    if (k == 0) atomicOr(&a.cnt->error, 2u);
    return;
  }
  if (w.bref == REF_EMPTY) {  // root of a scene without primitives: a node with no children
    if (k == 0) {
      QNode8 q;
      q.px = q.py = q.pz = 0.0f;
      q.ex = q.ey = q.ez = 127;
      q.imask = 0;
      q.child_base = q.tri_base = 0;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        q.meta[j] = 0;
        q.qlox[j] = q.qloy[j] = q.qloz[j] = 255;
        q.qhix[j] = q.qhiy[j] = q.qhiz[j] = 0;
      }
      a.nodes[number] = q;
      NodeInfo inf;
      inf.lo[0] = inf.lo[1] = inf.lo[2] = 0.0f;
      inf.hi[0] = inf.hi[1] = inf.hi[2] = 0.0f;
      inf.count = 0;
      inf.depth = depth;
      a.info[number] = inf;
    }
    return;
  }

  // children; lane k keeps child k
  uint32_t mine = 0u;
  int n = 1;
  if (!is_inner(w.bref, a.isleaf)) {
    mine = w.bref;  // whole (small) scene as one leaf
  } else {
    n = wide_children(a, w.bref, k, mine);
  }

  // this lane's child: box, primitive range and kind
  const bool has = k < (uint32_t)n;
  const uint32_t* rng32 = reinterpret_cast<const uint32_t*>(a.range);
  float4 l = make_float4(INFINITY, INFINITY, INFINITY, 0.0f), h = make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
  uint32_t f = 0u, cnt = 0u;
  bool inner = false;
  if (has) {
    if (mine & REF_LEAF) {
      l = a.slo[mine & ~REF_LEAF];
      h = a.shi[mine & ~REF_LEAF];
      f = mine & ~REF_LEAF;
      cnt = 1u;
    } else {
      l = a.nlo[mine];
      h = a.nhi[mine];
      f = rng32[2 * mine];
      cnt = rng32[2 * mine + 1] - f + 1u;
    }
    inner = is_inner(mine, a.isleaf);
  }
  const float ul[3] = {group_min(l.x), group_min(l.y), group_min(l.z)};
  const float uh[3] = {group_max(h.x), group_max(h.y), group_max(h.z)};
  const uint32_t ci = inner ? 1u : 0u, ct = (has && !inner) ? cnt : 0u;
  const uint32_t ni = group_sum(ci), nt = group_sum(ct);
  const uint32_t ninner_prims = group_sum(inner ? cnt : 0u);
  const uint32_t rank_i = group_prefix(ci, k), off_t = group_prefix(ct, k);
  double sah_leaf = 0.0, sah_leaf_tri = 0.0;
  if (has && !inner) {
    const float A = box_half_area(l, h);
    sah_leaf = (double)A * (double)((cnt + 3) / 4);
    sah_leaf_tri = (double)A * (double)cnt;
  }
  sah_leaf = group_sum(sah_leaf);
  sah_leaf_tri = group_sum(sah_leaf_tri);
  // the children partition the parent's range: a second count of the leaf primitives
  if (k == 0) {
    const uint32_t b = w.bref;
    const uint32_t total_prims = (b & REF_LEAF) ? 1u : (rng32[2 * b + 1] - rng32[2 * b] + 1u);
    if (total_prims - ninner_prims != nt) atomicOr(&a.cnt->error, 64u);
  }
  const uint32_t child_base = w.link, tri_base = w.tri;
  if ((uint64_t)child_base + ni > a.cap || (uint64_t)tri_base + nt + ninner_prims > a.n) {
    if (k == 0) atomicOr(&a.cnt->error, 2u);
    return;
  }
  if (k == 0) {
    st.records += nt;
    st.max_depth = max(st.max_depth, depth);
    st.max_stack = max(st.max_stack, (w.level & 0xffffu) + (uint32_t)n - 1u);  // a node pushes at most n-1 of its n children
    st.sah_nodes += (double)half_area(uh[0] - ul[0], uh[1] - ul[1], uh[2] - ul[2]);
    if (nt) {
      st.sah_leaves += sah_leaf;
      st.sah_leaves_tri += sah_leaf_tri;
    }
  }

  // quantisation grid over the widened union box (every lane the same)
  float p[3], sc[3];
  uint32_t e[3];
#pragma unroll
  for (int d = 0; d < 3; d++) {
    p[d] = ul[d] - eps;
    e[d] = grid_exponent(p[d], uh[d] + eps);
    sc[d] = __uint_as_float(e[d] << 23);
  }
  uint8_t* node = reinterpret_cast<uint8_t*>(a.nodes + number);
  uint32_t meta = 0u, qlx = 255u, qhx = 0u, qly = 255u, qhy = 0u, qlz = 255u, qhz = 0u;
  if (has) {
    qlx = quant_lo(l.x - eps, p[0], sc[0]);
    qhx = quant_hi(h.x + eps, p[0], sc[0]);
    qly = quant_lo(l.y - eps, p[1], sc[1]);
    qhy = quant_hi(h.y + eps, p[1], sc[1]);
    qlz = quant_lo(l.z - eps, p[2], sc[2]);
    qhz = quant_hi(h.z + eps, p[2], sc[2]);
    if (inner) {
      meta = 0x80u | rank_i;
    } else {
      meta = 1u + off_t;
      // leaf records are written afterwards, one thread each (k_write_leaves)
      for (uint32_t j = 0; j < cnt; j++)
        a.leaf_src[tri_base + off_t + j] = (f + j) | ((j + 1 == cnt) ? LEAF_SRC_LAST : 0u);
    }
  }
  node[offsetof(QNode8, meta) + k] = (uint8_t)meta;
  node[offsetof(QNode8, qlox) + k] = (uint8_t)qlx;
  node[offsetof(QNode8, qhix) + k] = (uint8_t)qhx;
  node[offsetof(QNode8, qloy) + k] = (uint8_t)qly;
  node[offsetof(QNode8, qhiy) + k] = (uint8_t)qhy;
  node[offsetof(QNode8, qloz) + k] = (uint8_t)qlz;
  node[offsetof(QNode8, qhiz) + k] = (uint8_t)qhz;
  const uint32_t imask = (uint32_t)group_sum(inner ? (1u << k) : 0u);
  if (k == 0) {
    uint32_t* hdr = reinterpret_cast<uint32_t*>(node);
    hdr[0] = __float_as_uint(p[0]);
    hdr[1] = __float_as_uint(p[1]);
    hdr[2] = __float_as_uint(p[2]);
    hdr[3] = e[0] | (e[1] << 8) | (e[2] << 16) | (imask << 24);
    hdr[4] = child_base;
    hdr[5] = tri_base;
    NodeInfo inf;
    inf.lo[0] = ul[0]; inf.lo[1] = ul[1]; inf.lo[2] = ul[2];
    inf.hi[0] = uh[0]; inf.hi[1] = uh[1]; inf.hi[2] = uh[2];
    inf.count = ninner_prims + nt;
    inf.depth = depth;
    a.info[number] = inf;
  }
}

// Leaf record r: the primitive at position leaf_src[r] (primref vals[pos],
// whose .w fields hold its geometry and primitive index) as a TriRec
// (v0, v0 - v1, v2 - v0; the three vertices for the robust test) or as the
// instance's InstRec, with TRI_LAST on the last record of each leaf.
__global__ __launch_bounds__(BT) void k_write_leaves(const uint32_t* __restrict__ leaf_src,
                                                     const uint32_t* __restrict__ vals, const float4* __restrict__ lo4,
                                                     const float4* __restrict__ hi4, const GeomDesc* __restrict__ geoms,
                                                     const BuildCounters* cnt, TriRec* __restrict__ tris,
                                                     InstRec* __restrict__ insts, uint32_t robust, uint32_t n) {
  const uint32_t r = blockIdx.x * BT + threadIdx.x;
  if (cnt->error || cnt->tri_count != n || r >= n) return;
  const uint32_t e = leaf_src[r];
  const uint32_t o = vals[e & ~LEAF_SRC_LAST];
  const uint32_t last = (e & LEAF_SRC_LAST) ? TRI_LAST : 0u;
  const uint32_t gi = __float_as_uint(lo4[o].w);
  const uint32_t prim = __float_as_uint(hi4[o].w);
  const GeomDesc g = geoms[gi];
  if (g.kind == GEOM_INSTANCES) {
    InstRec ir = *(const InstRec*)(g.indices + (uint64_t)prim * g.istride);
    ir.flags = (ir.flags & ~TRI_LAST) | last;
    insts[r] = ir;
    return;
  }
  const uint32_t* ix = (const uint32_t*)(g.indices + (uint64_t)prim * g.istride);
  const float* p0 = (const float*)(g.vertices + (uint64_t)ix[0] * g.vstride);
  const float* p1 = (const float*)(g.vertices + (uint64_t)ix[1] * g.vstride);
  const float* p2 = (const float*)(g.vertices + (uint64_t)ix[2] * g.vstride);
  TriRec tr;
  tr.v0x = p0[0]; tr.v0y = p0[1]; tr.v0z = p0[2];
  if (robust) {
    tr.e1x = p1[0]; tr.e1y = p1[1]; tr.e1z = p1[2];
    tr.e2x = p2[0]; tr.e2y = p2[1]; tr.e2z = p2[2];
  } else {
    tr.e1x = p0[0] - p1[0]; tr.e1y = p0[1] - p1[1]; tr.e1z = p0[2] - p1[2];
    tr.e2x = p2[0] - p0[0]; tr.e2y = p2[1] - p0[1]; tr.e2z = p2[2] - p0[2];
  }
  tr.primID = prim;
  tr.geomID = g.geomID;
  tr.flags = last;
  tris[r] = tr;
}

// Every node, in the order of their numbers: the top nodes, then the subtrees'
// nodes. A tree that failed its check (error bits set) is not written.
__global__ __launch_bounds__(BT) void k_emit_nodes(CollapseArgs a) {
  __shared__ uint32_t s_run;
  if (threadIdx.x == 0) s_run = a.cnt->error ? 0u : 1u;
  __syncthreads();
  if (!s_run) return;
  const uint32_t top = a.cnt->top_nodes, nsub = a.cnt->subtrees;
  const uint32_t total = top + a.prefix[a.max_sub];
  if (blockIdx.x == 0 && threadIdx.x == 0) a.cnt->node_count = total;
  CollapseStats st;
  for (uint32_t i = (blockIdx.x * BT + threadIdx.x) / CG; i < total; i += gridDim.x * (BT / CG)) {
    WideNode w;
    if (i < top) {
      w = a.top[i];
      if (w.link & REF_LEAF) w.link = top + a.prefix[w.link & ~REF_LEAF];
    } else {
      const uint32_t j = i - top;
      uint32_t lo = 0, hi = nsub - 1u;  // the subtree: the last whose first node is at most j
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) >> 1;
        if (a.prefix[mid] <= j) lo = mid; else hi = mid - 1u;
      }
      const uint32_t p = a.prefix[lo];
      w = a.rest[a.sub[lo].tri + (j - p)];
      w.link += top + p;
    }
    emit_node(a, w, i, threadIdx.x % CG, st);
  }
  block_stats(st);
  if (threadIdx.x == 0) a.stats[blockIdx.x] = st;
}

// The sum of the emission's statistics (atomics of every workgroup on a few
// counters took longer than the emission; this order of summation is fixed).
// The counters then go to the host.
__global__ __launch_bounds__(BT) void k_sum_stats(const CollapseStats* __restrict__ part, uint32_t n, BuildCounters* cnt,
                                                  uint32_t* post, uint32_t seq) {
  CollapseStats st;
  if (cnt->error) n = 0;  // (nothing was emitted)
  for (uint32_t i = threadIdx.x; i < n; i += BT) st.add(part[i]);
  block_stats(st);
  if (threadIdx.x == 0) {
    cnt->max_depth = st.max_depth;
    cnt->max_stack = st.max_stack;
    cnt->tri_count = st.records;
    cnt->sah_nodes = st.sah_nodes;
    cnt->sah_leaves = st.sah_leaves;
    cnt->sah_leaves_tri = st.sah_leaves_tri;
  }
  __syncthreads();
  if (threadIdx.x < 64) post_words(post, seq, reinterpret_cast<const uint32_t*>(cnt), COUNTER_WORDS);
}

// ------------------------------------------------------------------ host --

namespace {
// Leaves the stream idle however the build ends: the scratch and the staging
// memory are the next build's, which may be another thread's on another stream.
struct IdleAtEnd {
  hipStream_t s;
  bool idle = false;
  ~IdleAtEnd() {
    if (!idle) (void)hipStreamSynchronize(s);
  }
};
}  // namespace

void build_bvh(const std::vector<GeomDesc>& geoms, const BuildParams& prm, BuildScratch& S, DeviceBVH& out,
               hipStream_t s, uint32_t nscenes, UserTree* user, const std::function<void()>& before_write) {
  auto t0 = std::chrono::steady_clock::now();
  out.generation++;
  out.stats = BuildStats();
  out.robust = prm.robust ? 1u : 0u;
  uint64_t total64 = 0;
  for (const auto& g : geoms) total64 += g.num_tris;
  // positions and primitive references carry a flag in bit 31
  if (total64 >= REF_LEAF) throw hip_error(hipErrorInvalidValue, "a build holds fewer than 2^31 primitives");
  const uint32_t total = (uint32_t)total64;
  out.slots.assign(nscenes, SceneSlot());
  if (user) *user = UserTree();
  if (geoms.empty() || total == 0) {
    out.stats.num_prims = 0;
    out.stats.num_nodes = 0;
    return;
  }
  if (user && nscenes != 1) throw hip_error(hipErrorInvalidValue, "a user tree is one scene");
  // a QNode8 leaf slot addresses at most 15 records; a user tree's leaves
  // are handed to the caller and may hold up to 32
  const uint32_t leaf_cap = user ? 32u : 15u;
  const uint32_t max_leaf = prm.max_leaf < 1 ? 1 : (prm.max_leaf > leaf_cap ? leaf_cap : prm.max_leaf);
  const uint32_t width = prm.width < 2 ? 2 : (prm.width > 8 ? 8 : prm.width);
  const uint32_t min_leaf = prm.min_leaf < 1 ? 1 : (prm.min_leaf > max_leaf ? max_leaf : prm.min_leaf);
  const uint32_t block = prm.block < 1 ? 1 : prm.block;

  IdleAtEnd at_end{s};
  if (nscenes == 0 || nscenes > 65535) throw hip_error(hipErrorInvalidValue, "scene count out of range");
  S.geoms.reserve(geoms.size() * sizeof(GeomDesc));
  const uint32_t geom_words = (uint32_t)(geoms.size() * sizeof(GeomDesc) / 4);
  S.stage.reserve(((size_t)geom_words + 3 * (size_t)nscenes) * 4);
  memcpy(S.stage.ptr, geoms.data(), (size_t)geom_words * 4);
  S.counters.reserve(sizeof(BuildCounters));
  S.lo4.reserve((size_t)total * 16);
  S.hi4.reserve((size_t)total * 16);
  S.keys.reserve((size_t)total * 4);
  S.vals.reserve((size_t)total * 4);
  BuildCounters* cnt = S.counters.as<BuildCounters>();

  const bool batched = nscenes > 1;
  SceneAcc* sacc = nullptr;
  if (batched) {
    S.sacc.reserve((size_t)nscenes * sizeof(SceneAcc));
    sacc = S.sacc.as<SceneAcc>();
    hipLaunchKernelGGL(k_init_sacc, dim3(div_up(nscenes, BT)), dim3(BT), 0, s, sacc, nscenes);
  }
  hipLaunchKernelGGL(k_init_build, dim3(div_up(geom_words, BT)), dim3(BT), 0, s, cnt, nscenes,
                     S.stage.as<uint32_t>(), S.geoms.as<uint32_t>(), geom_words);
  hipLaunchKernelGGL(k_primrefs, dim3(div_up(total, (size_t)BT * PR_PER)), dim3(BT), 0, s, S.geoms.as<GeomDesc>(),
                     (uint32_t)geoms.size(), total, S.lo4.as<float4>(), S.hi4.as<float4>(), S.keys.as<uint32_t>(), cnt,
                     sacc);
  BuildCounters hc;
  std::vector<SceneAcc> hs(batched ? nscenes : 0);
  if (batched) {
    // group the references by scene (stable, so each scene keeps primref order); invalid ones sort last
    hipLaunchKernelGGL(k_iota, dim3(div_up(total, BT)), dim3(BT), 0, s, S.vals.as<uint32_t>(), total);
    RTG_HIP(hipGetLastError());
    S.sorter.sort_pairs(S.keys.as<uint32_t>(), S.vals.as<uint32_t>(), total, 0, 16, s);
    RTG_HIP(hipMemcpyAsync(&hc, cnt, sizeof(hc), hipMemcpyDeviceToHost, s));
    RTG_HIP(hipMemcpyAsync(hs.data(), sacc, nscenes * sizeof(SceneAcc), hipMemcpyDeviceToHost, s));
    RTG_HIP(hipStreamSynchronize(s));
  } else {
    // (the counts and bounds are final here: the host gets them while the sort runs)
    uint32_t* post = S.post.arm();
    hipLaunchKernelGGL(k_morton, dim3(div_up(total, BT)), dim3(BT), 0, s, S.lo4.as<float4>(), S.hi4.as<float4>(),
                       total, S.keys.as<uint32_t>(), S.vals.as<uint32_t>(), cnt, post, S.post.seq);
    RTG_HIP(hipGetLastError());
    S.sorter.sort_pairs(S.keys.as<uint32_t>(), S.vals.as<uint32_t>(), total, 0, 32, s);
    S.post.wait(s);
    memcpy(&hc, S.post.words(), sizeof(hc));
  }
  uint32_t n = hc.valid;
  out.stats.num_prims = n;
  for (int k = 0; k < 3; k++) {
    out.stats.bounds_lo[k] = o2f(hc.glo[k]);
    out.stats.bounds_hi[k] = o2f(hc.ghi[k]);
  }
  // scenes: position ranges, bounds, and the binary-tree reference of each root
  out.slots.assign(nscenes, SceneSlot());
  std::vector<uint32_t> first(nscenes, 0), count(nscenes, 0);
  std::vector<SahRoot> trees;
  std::vector<uint32_t> tree_of(nscenes, 0);
  {
    uint32_t pos = 0;
    for (uint32_t sI = 0; sI < nscenes; sI++) {
      SceneSlot& sl = out.slots[sI];
      sl.root = sI;
      count[sI] = batched ? hs[sI].valid : n;
      first[sI] = pos;
      pos += count[sI];
      sl.num_prims = count[sI];
      for (int k = 0; k < 3; k++) {
        sl.bounds_lo[k] = o2f(batched ? hs[sI].glo[k] : hc.glo[k]);
        sl.bounds_hi[k] = o2f(batched ? hs[sI].ghi[k] : hc.ghi[k]);
      }
      if (count[sI] >= 2) {
        SahRoot r;
        r.first = first[sI];
        r.count = count[sI];
        for (int k = 0; k < 3; k++) {
          r.clo[k] = o2f(batched ? hs[sI].clo[k] : hc.clo[k]);
          r.chi[k] = o2f(batched ? hs[sI].chi[k] : hc.chi[k]);
        }
        tree_of[sI] = (uint32_t)trees.size();
        trees.push_back(r);
      }
    }
    if (pos != n) throw hip_error(hipErrorUnknown, "per-scene primitive counts disagree with the total");
  }
  if (n == 0) {
    out.stats.num_nodes = 0;
    return;
  }
  // spatial splits (one scene of triangles, binned-SAH tree): the tree is
  // built over the pieces, whose centroids may lie anywhere in the scene box
  if (prm.split_budget > 0.0f && !batched && !user && geoms[0].kind == GEOM_TRIANGLES && trees.size() == 1 &&
      (prm.builder == BUILDER_SAH || prm.learned)) {
    const uint32_t nr = spatial_presplit(n, prm.split_budget, S.geoms.as<GeomDesc>(), out.stats.bounds_lo,
                                         out.stats.bounds_hi, S.vals, S.lo4, S.hi4, S.spatial, s);
    if (nr != n) {
      out.stats.num_split = nr - n;
      n = nr;
      out.stats.num_prims = n;
      out.slots[0].num_prims = n;
      count[0] = n;
      trees[0].count = n;
      for (int k = 0; k < 3; k++) {
        trees[0].clo[k] = 2.0f * out.stats.bounds_lo[k];
        trees[0].chi[k] = 2.0f * out.stats.bounds_hi[k];
      }
    }
  }
  if (user) user->n = n;

  S.slo.reserve((size_t)n * 16);
  S.shi.reserve((size_t)n * 16);
  const uint32_t ninner = n > 1 ? n - 1 : 1;
  S.child.reserve((size_t)ninner * 8);
  S.parent_int.reserve((size_t)ninner * 4);
  S.parent_leaf.reserve((size_t)n * 4);
  S.range.reserve((size_t)ninner * 8);
  S.nlo.reserve((size_t)ninner * 16);
  S.nhi.reserve((size_t)ninner * 16);
  S.cost.reserve((size_t)ninner * 32);
  S.split8.reserve((size_t)ninner * 8);
  S.isleaf.reserve((size_t)ninner);
  S.visit.reserve((size_t)ninner * 4);
  S.roots.reserve((size_t)nscenes * 12);
  uint32_t* sstage = S.stage.as<uint32_t>() + geom_words;
  std::copy(first.begin(), first.end(), sstage);
  std::copy(count.begin(), count.end(), sstage + nscenes);
  std::copy(tree_of.begin(), tree_of.end(), sstage + 2 * (size_t)nscenes);
  RootArgs ra_none{}, ra_place{nscenes, sstage, nullptr, nullptr, S.roots.as<uint32_t>(), &cnt->error};
  auto gather = [&](const RootArgs& r) {
    hipLaunchKernelGGL(k_gather_sorted, dim3(div_up(std::max(n, r.nscenes), BT)), dim3(BT), 0, s,
                       S.vals.as<uint32_t>(), S.lo4.as<float4>(), S.hi4.as<float4>(), n, S.slo.as<float4>(),
                       S.shi.as<float4>(), S.visit.as<uint32_t>(), r);
  };
  const bool use_sah = batched || prm.builder == BUILDER_SAH || prm.learned;
  gather(use_sah && !trees.empty() ? ra_none : ra_place);
  if (!trees.empty()) {
    if (batched)
      hipLaunchKernelGGL(k_fill_none, dim3(div_up(n, BT)), dim3(BT), 0, s, S.parent_leaf.as<uint32_t>(), n);
    if (use_sah) {
      SahRoots so;
      build_sah_tree(n, S.vals.as<uint32_t>(), S.slo.as<float4>(), S.shi.as<float4>(), trees, S.child.as<uint32_t>(),
                     S.parent_int.as<uint32_t>(), S.parent_leaf.as<uint32_t>(), S.range.as<uint2>(),
                     prm.learned, prm.median_below, S.sah, so, s);
      // boxes in the final primitive order
      ra_place.tree_root = so.roots;
      ra_place.tree_error = so.error;
      gather(ra_place);
    } else {
      hipLaunchKernelGGL(k_radix_tree, dim3(div_up(n - 1, BT)), dim3(BT), 0, s, S.keys.as<uint32_t>(), (int)n,
                         S.child.as<uint32_t>(), S.parent_int.as<uint32_t>(), S.parent_leaf.as<uint32_t>(),
                         S.range.as<uint2>());
    }
    RefitArgs ra{n, S.child.as<uint32_t>(), S.range.as<uint2>(), S.slo.as<float4>(), S.shi.as<float4>(),
                 S.nlo.as<float4>(), S.nhi.as<float4>(), S.cost.as<float>(), S.split8.as<uint8_t>(),
                 S.isleaf.as<uint8_t>(), prm.cost_node, prm.cost_tri, max_leaf, width, min_leaf, block, &cnt->error};
    uint32_t nlists = div_up(n, REFIT_CHUNK), cap = REFIT_CHUNK;
    S.refit_list[0].reserve((size_t)n * 4);
    S.refit_list[1].reserve((size_t)n * 4);
    S.refit_count.reserve((size_t)2 * nlists * 4);
    uint32_t* lcount = S.refit_count.as<uint32_t>();
    hipLaunchKernelGGL(k_refit_chunk, dim3(nlists), dim3(BT), 0, s, ra, S.parent_int.as<uint32_t>(),
                       S.visit.as<uint32_t>(), S.refit_list[0].as<uint32_t>(), lcount);
    for (int k = 0; nlists > 1; k ^= 1) {
      const uint32_t blocks = div_up(nlists, REFIT_FAN);
      hipLaunchKernelGGL(k_refit_span, dim3(blocks), dim3(BT), 0, s, ra, S.parent_int.as<uint32_t>(),
                         S.visit.as<uint32_t>(), S.refit_list[k].as<uint32_t>(), lcount, cap, nlists,
                         S.refit_list[k ^ 1].as<uint32_t>(), lcount + nlists);
      lcount += nlists;
      nlists = blocks;
      cap *= REFIT_FAN;  // (at most 2^30 where another launch follows)
    }
    hipLaunchKernelGGL(k_check_tree, dim3(div_up(n, BT)), dim3(BT), 0, s,
                       use_sah ? nullptr : S.keys.as<uint32_t>(), n, &cnt->roots_seen,
                       S.child.as<uint32_t>(), S.parent_int.as<uint32_t>(), S.parent_leaf.as<uint32_t>(),
                       S.visit.as<uint32_t>(), &cnt->error);
    RTG_HIP(hipGetLastError());
  }
  // tree roots the check must meet (its error bits stop the collapse on the
  // device; both are read back with the collapse's results)
  uint32_t roots_expected = (uint32_t)trees.size();
  for (uint32_t sI = 0; sI < nscenes; sI++) roots_expected += count[sI] == 1 ? 1u : 0u;
  if (user) {
    RTG_HIP(hipMemcpyAsync(&hc, cnt, sizeof(hc), hipMemcpyDeviceToHost, s));
    RTG_HIP(hipStreamSynchronize(s));
    if (!trees.empty() && (hc.error || hc.roots_seen != roots_expected))
      throw hip_error(hipErrorUnknown, "binary tree check failed: error bits " + std::to_string(hc.error) +
                                           ", roots " + std::to_string(hc.roots_seen) + " of " +
                                           std::to_string(roots_expected));
  }

  if (user) {  // the binary tree with its collapse decisions, for the caller's own nodes
    const uint32_t ni = n > 1 ? n - 1 : 0;
    RTG_HIP(hipMemcpyAsync(&user->root, S.roots.ptr, 4, hipMemcpyDeviceToHost, s));
    user->child.resize(2 * (size_t)ni);
    user->range.resize(2 * (size_t)ni);
    user->split8.resize(8 * (size_t)ni);
    user->isleaf.resize(ni);
    user->nbox.resize(8 * (size_t)ni);
    user->pbox.resize(8 * (size_t)n);
    if (ni) {
      RTG_HIP(hipMemcpyAsync(user->child.data(), S.child.ptr, 8 * (size_t)ni, hipMemcpyDeviceToHost, s));
      RTG_HIP(hipMemcpyAsync(user->range.data(), S.range.ptr, 8 * (size_t)ni, hipMemcpyDeviceToHost, s));
      RTG_HIP(hipMemcpyAsync(user->split8.data(), S.split8.ptr, 8 * (size_t)ni, hipMemcpyDeviceToHost, s));
      RTG_HIP(hipMemcpyAsync(user->isleaf.data(), S.isleaf.ptr, ni, hipMemcpyDeviceToHost, s));
      RTG_HIP(hipMemcpy2DAsync(user->nbox.data(), 32, S.nlo.ptr, 16, 16, ni, hipMemcpyDeviceToHost, s));
      RTG_HIP(hipMemcpy2DAsync(user->nbox.data() + 4, 32, S.nhi.ptr, 16, 16, ni, hipMemcpyDeviceToHost, s));
    }
    RTG_HIP(hipMemcpy2DAsync(user->pbox.data(), 32, S.slo.ptr, 16, 16, n, hipMemcpyDeviceToHost, s));
    RTG_HIP(hipMemcpy2DAsync(user->pbox.data() + 4, 32, S.shi.ptr, 16, 16, n, hipMemcpyDeviceToHost, s));
    RTG_HIP(hipStreamSynchronize(s));
    at_end.idle = true;
    user->width = width;
    out.stats.num_prims = n;
    out.stats.ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
    return;
  }

  // outputs: at most n + nscenes nodes, exactly n triangle records
  const uint32_t cap = n + nscenes;
  if (before_write) before_write();
  out.nodes.reserve((size_t)cap * sizeof(QNode8));
  const bool inst_build = geoms[0].kind == GEOM_INSTANCES;
  for (const auto& g : geoms)
    if ((g.kind == GEOM_INSTANCES) != inst_build)
      throw hip_error(hipErrorInvalidValue, "a build holds either triangles or instance records");
  out.instances = inst_build;
  if (inst_build) out.insts.reserve((size_t)n * sizeof(InstRec));
  else out.tris.reserve((size_t)n * sizeof(TriRec));
  out.info.reserve((size_t)cap * sizeof(NodeInfo));
  const uint32_t max_sub = nscenes > 1 ? nscenes + SUB_MAX : SUB_MAX;
  S.walk_top.reserve((size_t)top_cap(max_sub) * sizeof(WideNode));
  S.walk_sub.reserve((size_t)max_sub * sizeof(WideNode));
  S.walk_rest.reserve((size_t)n * sizeof(WideNode));
  S.walk_count.reserve(((size_t)max_sub + 1) * 8);

  CollapseArgs ca;
  ca.child = S.child.as<uint32_t>();
  ca.range = S.range.as<uint2>();
  ca.nlo = S.nlo.as<float4>();
  ca.nhi = S.nhi.as<float4>();
  ca.isleaf = S.isleaf.as<uint8_t>();
  ca.split8 = S.split8.as<uint8_t>();
  ca.slo = S.slo.as<float4>();
  ca.shi = S.shi.as<float4>();
  ca.cnt = cnt;
  ca.nscenes = nscenes;
  ca.n = n;
  ca.width = width;
  ca.max_sub = max_sub;
  ca.top = S.walk_top.as<WideNode>();
  ca.sub = S.walk_sub.as<WideNode>();
  ca.rest = S.walk_rest.as<WideNode>();
  ca.count = S.walk_count.as<uint32_t>();
  ca.prefix = ca.count + max_sub + 1;
  ca.nodes = out.nodes.as<QNode8>();
  S.leaf_src.reserve((size_t)n * 4);
  ca.leaf_src = S.leaf_src.as<uint32_t>();
  ca.info = out.info.as<NodeInfo>();
  ca.cap = cap;
  hipLaunchKernelGGL(k_walk_top, dim3(1), dim3(WT), 0, s, ca, S.roots.as<uint32_t>(), S.roots.as<uint32_t>() + nscenes,
                     S.roots.as<uint32_t>() + 2 * (size_t)nscenes);
  hipLaunchKernelGGL(k_walk_rest, dim3(std::min(max_sub + 1u, 512u)), dim3(WT), 0, s, ca);
  S.scanner.exclusive(ca.count, S.walk_count.as<uint32_t>() + max_sub + 1, (size_t)max_sub + 1, s);
  const uint32_t egrid = std::min(div_up(cap, BT / CG), 4096u);
  S.walk_stats.reserve((size_t)egrid * sizeof(CollapseStats));
  ca.stats = S.walk_stats.as<CollapseStats>();
  hipLaunchKernelGGL(k_emit_nodes, dim3(egrid), dim3(BT), 0, s, ca);
  uint32_t* post = S.post.arm();
  hipLaunchKernelGGL(k_sum_stats, dim3(1), dim3(BT), 0, s, ca.stats, egrid, cnt, post, S.post.seq);
  hipLaunchKernelGGL(k_write_leaves, dim3(div_up(n, BT)), dim3(BT), 0, s, S.leaf_src.as<uint32_t>(),
                     S.vals.as<uint32_t>(), S.lo4.as<float4>(), S.hi4.as<float4>(), S.geoms.as<GeomDesc>(), cnt,
                     inst_build ? nullptr : out.tris.as<TriRec>(), inst_build ? out.insts.as<InstRec>() : nullptr,
                     prm.robust ? 1u : 0u, n);
  RTG_HIP(hipGetLastError());
  RTG_HIP(hipStreamSynchronize(s));
  at_end.idle = true;
  S.post.wait(s);
  memcpy(&hc, S.post.words(), sizeof(hc));
  if (!trees.empty() && (hc.roots_seen != roots_expected || (hc.error & 5u)))
    throw hip_error(hipErrorUnknown, "binary tree check failed: error bits " + std::to_string(hc.error) + ", roots " +
                                         std::to_string(hc.roots_seen) + " of " + std::to_string(roots_expected));
  if (hc.error || hc.tri_count != n)
    throw hip_error(hipErrorUnknown, "BVH build consistency check failed: error bits " + std::to_string(hc.error) +
                                         ", primitives " + std::to_string(n) + ", triangle records " +
                                         std::to_string(hc.tri_count) + ", nodes " + std::to_string(hc.node_count));
  if (hc.max_stack + 1 > TRACE_STACK)
    throw hip_error(hipErrorUnknown, "BVH too deep for the traversal stack: " + std::to_string(hc.max_stack + 1) +
                                         " entries needed, " + std::to_string(TRACE_STACK) + " available");
  out.stats.num_nodes = hc.node_count;
  out.stats.max_depth = hc.max_depth;
  out.stats.max_stack = hc.max_stack + 1;
  const double root_area = half_area(out.stats.bounds_hi[0] - out.stats.bounds_lo[0],
                                     out.stats.bounds_hi[1] - out.stats.bounds_lo[1],
                                     out.stats.bounds_hi[2] - out.stats.bounds_lo[2]);
  if (root_area > 0) {
    out.stats.sah = (hc.sah_nodes + hc.sah_leaves) / root_area;
    out.stats.sah_tri = (hc.sah_nodes + hc.sah_leaves_tri) / root_area;
  }
  if (hc.error) throw hip_error(hipErrorUnknown, "BVH build consistency check failed (" + std::to_string(hc.error) + ")");
  if (hc.tri_count != n) throw hip_error(hipErrorUnknown, "BVH build lost triangles");
  out.stats.ms_total = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace rtg
