// Ray traversal kernels: one ray per lane over the quantised BVH8.
//
// Reference anchors:
//   stream entry rules (rays with !(tnear <= tfar) are skipped, occluded rays
//     get tfar = -inf): kernels/common/rtcore.cpp:595-623, :848-874,
//     kernels/bvh/bvh_intersector_stream_filters.cpp:135-151, bvh_intersector1.cpp:191-193;
//   per-ray stack traversal, nearest child first, far siblings pushed with
//     their entry distance and skipped on pop once beyond the current hit:
//     kernels/bvh/bvh_intersector1.cpp:31-119, bvh_traverser1.h:519-643;
//   robust slab test (rdir scaled by 1 -/+ 3 ulp, zero_fix):
//     kernels/bvh/node_intersector1.h:122-190, common/math/vec3fa.h:172-176;
//   Moeller-Trumbore triangle test, same FP32/FMA sequence:
//     kernels/geometry/triangle_intersector_moeller.h:62-114, common/math/vec3.h:204,209,
//     common/math/math.h:367-372;
//   hit write-back: kernels/geometry/intersector_epilog.h:280-292.
// This file is compiled with -ffp-contract=off: every FMA is explicit.
//
// Differences from the reference, shared with the CPU oracle so results are
// traversal-order independent: t/u/v use IEEE division; the closest hit is
// the lexicographic minimum of (t, geomID, primID) over all valid hits of
// the original [tnear, tfar]; culling is conservative (robust slab test on
// boxes that contain the widened triangle boxes, interval ends widened by
// 2^-12 relative).
#include "trace.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

// Scratch of the no-allocation queries (ray counters, with the error bits
// in word 1), one copy per GPU. In host code this name is a host-side stand-in,
// not a device address: kernels get the address noalloc_setup() looked up.
static __device__ __align__(256) uint32_t scratch[rtg::NOALLOC_SCRATCH_WORDS];

namespace rtg {

constexpr int TB = 256;
constexpr int STACK = (int)TRACE_STACK;  // entries per ray (the builder checks its trees against it)
// A node step pushes up to 7 entries after checking only that the stack
// holds at most STACK (fits()), so the arrays have room for 7 more.
constexpr int STACK_CAP = STACK + 8;

// Sets error bits. The word may be in host memory, which has no atomic OR over
// PCIe: of bits that two lanes set at once, one may be lost, never both.
__device__ inline void raise_error(uint32_t* err, uint32_t bits) {
  const uint32_t old = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  __hip_atomic_store(err, old | bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Per-lane traversal stack: the top LDS_SLOTS entries live in LDS (slot-major,
// so lanes touching the same slot hit distinct banks), older entries spill
// to a private array only when the ring is full. Entry = (ref, entry distance).
// The spill array is a separate local of the kernel: were it a member here,
// a dynamically indexed store into it could alias sp and lo, and the
// compiler would keep the whole struct in scratch memory.
// The LDS pointer is typed in the local address space so that the ring is
// reached with ds_* instructions (a generic pointer makes every access a flat
// access through the vector memory pipeline).
typedef __attribute__((address_space(3))) uint64_t lds_u64;
__device__ inline uint64_t pack_entry(uint2 e) { return (uint64_t)e.x | ((uint64_t)e.y << 32); }
__device__ inline uint2 unpack_entry(uint64_t v) { return make_uint2((uint32_t)v, (uint32_t)(v >> 32)); }

// Second word of a closest-hit stack entry: in the high half the entry
// distance's bits, rounded down, and in the low half the least such of the
// entries below it, so that a pop can tell when every entry left is farther
// than the closest hit. Distances compare as signed integers: positive ones
// order like the floats, and a negative one (tnear < 0) is below all of them.
__device__ inline uint32_t pack_dist(int key, int& smin) {
  const uint32_t y = __builtin_amdgcn_perm((uint32_t)key, (uint32_t)smin, 0x07060302u);
  smin = min(smin, key);
  return y;
}
__device__ inline int below_dist(uint32_t y) { return (int)(y << 16); }
// A word above this belongs to an entry beyond `lim` (which no key of a
// negative distance is, whatever lim).
__device__ inline int dist_limit(float lim) { return max((int)__float_as_uint(lim), 0) | 0xffff; }
constexpr int DIST_NONE = 0x7f800000;         // of an empty stack
constexpr int DIST_ALWAYS = (int)0xff800000;  // of an entry that is never skipped

template <int LDS_SLOTS>
struct RingStack {
  // A power-of-two ring finds entry i's slot as i & (LDS_SLOTS - 1); any
  // other size keeps the byte offset of entry sp's slot in `top`. When the
  // ring is full, the oldest ring entry (lo = sp - LDS_SLOTS) sits in entry
  // sp's slot.
  static constexpr bool POW2 = (LDS_SLOTS & (LDS_SLOTS - 1)) == 0;
  static constexpr uint32_t STEP = TB * 8, RING = LDS_SLOTS * STEP;  // bytes between a lane's slots, and of the ring
  typedef __attribute__((address_space(3))) char lds_char;
  lds_char* lds;
  uint64_t* spill;  // STACK_CAP entries, private
  int sp, lo;       // [0, lo) spilled, [lo, sp) in the ring
  uint32_t top;     // (other sizes than powers of two)
  __device__ inline lds_u64& slot() const {
    if constexpr (POW2) return *(lds_u64*)(lds + (uint32_t)(sp & (LDS_SLOTS - 1)) * STEP);
    else return *(lds_u64*)(lds + top);
  }
  // (the one of x and x -/+ RING that is in the ring is the smaller as unsigned)
  __device__ inline void up() {
    sp++;
    if constexpr (!POW2) top = min(top + STEP, top + STEP - RING);
  }
  __device__ inline void down() {
    sp--;
    if constexpr (!POW2) top = min(top - STEP, top - STEP + RING);
  }
  __device__ inline void init(uint64_t* ring, uint64_t* spill_mem) {
    lds = (lds_char*)(POW2 ? ring + threadIdx.x : ring);
    spill = spill_mem;
    clear();
  }
  // Whether a node's entries (at most 7) may be put(): true while the stack
  // holds at most STACK entries, which a tree the builder accepted never
  // exceeds; past it the arrays' 7 spare entries keep a corrupt tree's
  // pushes in bounds until the error stops the ray.
  __device__ inline bool fits() const { return sp <= STACK; }
  __device__ inline void put(uint2 e) {
    if (sp - lo == LDS_SLOTS) {
      spill[lo] = slot();
      lo++;
    }
    slot() = pack_entry(e);
    up();
  }
  __device__ inline bool push(uint2 e) {
    if (sp >= STACK) return false;
    put(e);
    return true;
  }
  __device__ inline uint2 pop() {
    down();
    // an entry below the ring comes back through its ring slot, so that the
    // read below is always an LDS read
    if (sp < lo) {
      lo = sp;
      slot() = spill[sp];
    }
    return unpack_entry(slot());
  }
  __device__ inline bool empty() const { return sp == 0; }
  __device__ inline void clear() {
    sp = lo = 0;
    top = threadIdx.x * 8;
  }
};

// LDS_SLOTS == 0: the whole stack is a private array.
template <>
struct RingStack<0> {
  uint64_t* spill;
  int sp;
  __device__ inline void init(uint64_t*, uint64_t* spill_mem) {
    spill = spill_mem;
    sp = 0;
  }
  __device__ inline bool push(uint2 e) {
    if (sp >= STACK) return false;
    spill[sp++] = pack_entry(e);
    return true;
  }
  __device__ inline bool fits() const { return sp <= STACK; }
  __device__ inline void put(uint2 e) { spill[sp++] = pack_entry(e); }
  __device__ inline uint2 pop() { return unpack_entry(spill[--sp]); }
  __device__ inline bool empty() const { return sp == 0; }
  __device__ inline void clear() { sp = 0; }
};

// How a persistent launch shares out its M rays: in `count` runs of RAY_RUN
// consecutive slots, dealt in groups of 1 << qs to as many queues (one for each
// XCD: blocks are dealt to the XCDs in turn). Run j of queue q is run
// (j << qs) + ((q + j) & ((1 << qs) - 1)): the turn keeps a queue from getting
// one column of an image.
struct RayRuns {
  uint32_t count, qs;
};

// Slots of a run: one refill of a whole wave. Longer runs need fewer atomics
// but leave more to the last waves: with one counter for all, 256 gave 573 us
// and 64 gave 616 us for 2 M camera rays on a 2.1 M triangle terrain (the
// atomics on one address pass one at a time), with a counter for each XCD 64
// gives 430 us (128: 473, 32: 451, 16: 517). 2^24 incoherent rays in the
// 2^20-triangle soup take 7.22 ms at 64 and 7.43 at 256, two million rays
// through 10,000 instances and their shadow rays 3.56 ms against 4.07.
constexpr uint32_t RAY_RUN = 64;

// A persistent wave's rays. Its first run is its own (the wave's place in its
// queue), the next ones come from its queue's counter, so a refill costs a
// global atomic only once every RAY_RUN rays (its latency stalls the whole
// wave), and a stream that the first runs cover needs no counter. Every lane
// computes the same values (all inputs are wave-uniform), so the state needs
// no broadcast.
struct WavePool {
  uint32_t lb, le;  // unassigned slots [lb, le) of the current run
  bool gdone;       // the wave's queue has no more runs
  __device__ inline void run(const RayRuns& rr, uint32_t M, uint32_t j, uint32_t& nb, uint32_t& ne) {
    const uint32_t k = (j << rr.qs) + ((blockIdx.x + j) & ((1u << rr.qs) - 1u));
    gdone = ((j + 1u) << rr.qs) >= rr.count;
    nb = k < rr.count ? k * RAY_RUN : M;
    ne = M - nb < RAY_RUN ? M : nb + RAY_RUN;
  }
  __device__ inline void init(const RayRuns& rr, uint32_t M) {
    run(rr, M, (blockIdx.x >> rr.qs) * (TB / 64) + (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lb, le);
    gdone = gdone || ((gridDim.x * (TB / 64)) >= rr.count);
  }
  // Hands out nidle slots (idle lane `rank` gets the rank-th); returns this
  // lane's slot or 0xffffffff when the rays have run out.
  __device__ inline uint32_t take(const RayRuns& rr, uint32_t* next, uint32_t M, int nidle, uint32_t rank, int lane) {
    const uint32_t have = le - lb;
    uint32_t nb = 0, ne = 0;
    if (have < (uint32_t)nidle && !gdone) {
      uint32_t g = 0;
      if (lane == 0) g = atomicAdd(next + (blockIdx.x & ((1u << rr.qs) - 1u)) * COUNTER_STRIDE, 1u);
      g = (uint32_t)__builtin_amdgcn_readfirstlane((int)g);
      run(rr, M, (gridDim.x >> rr.qs) * (TB / 64) + g, nb, ne);
    }
    uint32_t slot = 0xffffffffu;
    if (rank < have) slot = lb + rank;
    else if (nb + (rank - have) < ne) slot = nb + (rank - have);
    if (have >= (uint32_t)nidle) {
      lb += (uint32_t)nidle;
    } else {
      const uint32_t need = (uint32_t)nidle - have;
      lb = nb + (need < ne - nb ? need : ne - nb);
      le = ne;
    }
    return slot;
  }
  __device__ inline bool empty() const { return gdone && lb >= le; }
};

__device__ inline float widen_up(float x) { return __builtin_isinf(x) ? x : x + fabsf(x) * CULL_MARGIN; }
__device__ inline float widen_down(float x) { return __builtin_isinf(x) ? x : x - fabsf(x) * CULL_MARGIN; }

struct TRay {
  float ox, oy, oz, dx, dy, dz;
  float rnx, rny, rnz, rfx, rfy, rfz;
  bool negx, negy, negz;
  float tnear, tfar, tlo;
};

__device__ inline float zero_fix(float d) { return fabsf(d) < MIN_RCP_INPUT ? MIN_RCP_INPUT : d; }

__device__ inline void setup_ray(TRay& r, float4 a, float4 b, float tfar) {
  const float round_down = 1.0f - 3.0f * 1.1920928955078125e-7f;
  const float round_up = 1.0f + 3.0f * 1.1920928955078125e-7f;
  r.ox = a.x; r.oy = a.y; r.oz = a.z; r.tnear = a.w;
  r.dx = b.x; r.dy = b.y; r.dz = b.z;
  r.tfar = tfar;
  const float rx = 1.0f / zero_fix(b.x), ry = 1.0f / zero_fix(b.y), rz = 1.0f / zero_fix(b.z);
  r.rnx = round_down * rx; r.rny = round_down * ry; r.rnz = round_down * rz;
  r.rfx = round_up * rx; r.rfy = round_up * ry; r.rfz = round_up * rz;
  r.negx = !(r.rnx >= 0.0f);
  r.negy = !(r.rny >= 0.0f);
  r.negz = !(r.rnz >= 0.0f);
  r.tlo = widen_down(a.w);
}

__device__ inline uint32_t spread3(uint32_t x) {
  x = (x | (x << 16)) & 0x030000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

__device__ inline float byte_f(uint32_t w, int k) { return (float)((w >> (8 * k)) & 0xffu); }

// A lane without a ray (REF_EMPTY: one that has to pop its next reference).
// That state lives in the reference itself, and branches set it instead of
// leaving the step: a bool that several branches set, or a `continue`, costs a
// lane mask in scalar registers and scalar instructions at every merge. (The
// two-level kernel spilled 43 to 55 scalar registers to vector lanes: 3.52 ms
// for two million rays through 10,000 instances and their shadow rays, 2.82
// without any; the one-level kernels gained 1.5 to 4.5 %.) REF_DONE: the ray
// has ended and its hit is still to be written, with those of the wave's other
// ended rays at the next refill.
constexpr uint32_t REF_IDLE = 0xffffffffu, REF_DONE = 0xfffffffdu;

struct NodeHit {
  uint32_t mask;
  uint32_t imask;
  uint32_t cb, tb;  // reference bases of meta_ref()
  uint32_t meta_lo, meta_hi;
  float tn[8];
  bool hit[8];
};

// Slab test of the 8 children on planes that decode as fmaf(2^(e-127), q, p)
// (the expression the builder verified against every widened child box),
// with rdir rounded down for near and up for far planes as the reference's
// robust TravRay does (kernels/bvh/node_intersector1.h:122-190).
template <bool OCCLUDED>
__device__ inline void intersect_node(const QNode8* __restrict__ nodes, uint32_t i, const TRay& r, float thi,
                                      NodeHit& h) {
  const uint4* np = reinterpret_cast<const uint4*>(nodes + i);
  const uint4 w0 = np[0], w1 = np[1], w2 = np[2], w3 = np[3], w4 = np[4];
  const float px = __uint_as_float(w0.x), py = __uint_as_float(w0.y), pz = __uint_as_float(w0.z);
  const float sx = __uint_as_float((w0.w & 0xffu) << 23);
  const float sy = __uint_as_float(((w0.w >> 8) & 0xffu) << 23);
  const float sz = __uint_as_float(((w0.w >> 16) & 0xffu) << 23);
  h.imask = w0.w >> 24;
  h.cb = w1.x - 0x80u;
  h.tb = (w1.y | REF_LEAF) - 1u;
  // Defined here, so that the compiler keeps the node's 16 B loads whole
  // instead of loading these two words again where the pushes use them.
  asm volatile("" : "+v"(h.cb), "+v"(h.tb));
  h.meta_lo = w1.z;
  h.meta_hi = w1.w;
  // near / far plane bytes per axis (lo plane is near for a positive direction)
  const uint32_t nx0 = r.negx ? w2.z : w2.x, nx1 = r.negx ? w2.w : w2.y;
  const uint32_t fx0 = r.negx ? w2.x : w2.z, fx1 = r.negx ? w2.y : w2.w;
  const uint32_t ny0 = r.negy ? w3.z : w3.x, ny1 = r.negy ? w3.w : w3.y;
  const uint32_t fy0 = r.negy ? w3.x : w3.z, fy1 = r.negy ? w3.y : w3.w;
  const uint32_t nz0 = r.negz ? w4.z : w4.x, nz1 = r.negz ? w4.w : w4.y;
  const uint32_t fz0 = r.negz ? w4.x : w4.z, fz1 = r.negz ? w4.y : w4.w;
  // Plane distance (p + s q - o) rdir as one FMA per plane, q a + b with
  // a = s rdir (exact: s is a power of two) and b = (p - o) rdir (two
  // roundings) formed once per node. Against the decode-then-subtract form
  // the error moves from |plane - o| to |p - o|: at most u|b| + u/2 |t|
  // (u = 2^-23). Where |b| is close to |t| (origin away from the node) the
  // 3-ulp scaling of rdir covers it; where it cancels (origin near or in the
  // node), |p - o| is within the node's extent, below 2 max|coord|, and the
  // builder's box widening by max|coord| 2^-20 = 8u max|coord| covers it. So
  // no box holding a hit is culled (the hits of this form equal the
  // oracle's on every parity test), and each plane costs a byte conversion
  // and one FMA instead of an FMA, a subtraction and a product.
  const float anx = sx * r.rnx, afx = sx * r.rfx, any = sy * r.rny, afy = sy * r.rfy, anz = sz * r.rnz, afz = sz * r.rfz;
  const float bnx = (px - r.ox) * r.rnx, bfx = (px - r.ox) * r.rfx;
  const float bny = (py - r.oy) * r.rny, bfy = (py - r.oy) * r.rfy;
  const float bnz = (pz - r.oz) * r.rnz, bfz = (pz - r.oz) * r.rfz;
  uint32_t mask = 0;
#pragma unroll
  for (int c = 0; c < 8; c++) {
    const int k = c & 3;
    const uint32_t mb = ((c < 4 ? h.meta_lo : h.meta_hi) >> (8 * k)) & 0xffu;
    const float qnx = byte_f(c < 4 ? nx0 : nx1, k), qfx = byte_f(c < 4 ? fx0 : fx1, k);
    const float qny = byte_f(c < 4 ? ny0 : ny1, k), qfy = byte_f(c < 4 ? fy0 : fy1, k);
    const float qnz = byte_f(c < 4 ? nz0 : nz1, k), qfz = byte_f(c < 4 ? fz0 : fz1, k);
    const float tnx = __builtin_fmaf(qnx, anx, bnx), tfx = __builtin_fmaf(qfx, afx, bfx);
    const float tny = __builtin_fmaf(qny, any, bny), tfy = __builtin_fmaf(qfy, afy, bfy);
    const float tnz = __builtin_fmaf(qnz, anz, bnz), tfz = __builtin_fmaf(qfz, afz, bfz);
    const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, r.tlo));
    // (closest hit: push_near_to_far compares the entry distances with the limit)
    const float tf = OCCLUDED ? fminf(fminf(tfx, tfy), fminf(tfz, thi)) : fminf(fminf(tfx, tfy), tfz);
    h.tn[c] = tn;
    h.hit[c] = (tn <= tf) && (mb != 0u);
    mask |= h.hit[c] ? (1u << c) : 0u;
  }
  h.mask = mask;
}

// A child's reference from its meta byte m (internal children 0x80 | rank,
// leaves 1 + offset of the first record): m plus a base chosen by bit 7,
// cb = child_base - 0x80 or tb = (tri_base | REF_LEAF) - 1.
__device__ inline uint32_t meta_ref(uint32_t m, uint32_t cb, uint32_t tb) { return m + ((m & 0x80u) ? cb : tb); }

__device__ inline uint32_t child_ref(const NodeHit& h, int c) {
  const uint32_t mb = ((c < 4 ? h.meta_lo : h.meta_hi) >> (8 * (c & 3))) & 0xffu;
  return meta_ref(mb, h.cb, h.tb);
}

// Occlusion: pushes the hit children except the first in slot order, sets
// `next` to that one and returns whether any child was hit.
template <class Stack>
__device__ inline bool push_any_order(const NodeHit& h, Stack& stack, uint32_t* err, uint32_t& next) {
  if (!h.mask) return false;
  const uint32_t cb = h.cb, tb = h.tb;
  const uint64_t meta = (uint64_t)h.meta_lo | ((uint64_t)h.meta_hi << 32);
  const int c0 = __builtin_ctz(h.mask);
  uint32_t rem = h.mask & (h.mask - 1u);
  if (stack.fits()) {
    while (rem) {
      const int c = __builtin_ctz(rem);
      rem &= rem - 1u;
      stack.put(make_uint2(meta_ref((uint32_t)(meta >> (8 * c)) & 0xffu, cb, tb), 0u));
    }
  } else {
    raise_error(err, 1u);
  }
  next = meta_ref((uint32_t)(meta >> (8 * c0)) & 0xffu, cb, tb);
  return true;
}

// Closest hit: pushes the hit children except the nearest, farthest first,
// each with its entry distance, sets `next` to the nearest child and returns
// whether any child was hit within the limit.
// A key is the entry distance's bit pattern with the child's meta byte in the
// low 8 bits (distinct among a node's children), or NO_HIT for a child that is
// not hit; keys compare as signed integers (see pack_dist). The perturbation of
// the low 8 bits changes only the order among nearly equal children. A
// 19-comparator network (Batcher's odd-even merge sort) orders the keys
// decreasingly without branches: children not hit and those beyond the limit
// first, the nearest hit child last. The stored distance is the key's high half
// (rounded down), never above a positive entry distance, so the pop test stays
// conservative. The limit is compared with the sorted keys (which a push tests
// anyway) instead of taking part in every child's slab test. (With integer
// distances and this, 274 VALU instructions a ray instead of 290 on the
// 2^20-triangle soup, 7.00 ms instead of 7.14 for 2^24 rays; with the lanes'
// state in their references 229 and 6.72 ms.)
template <class Stack>
__device__ inline bool push_near_to_far(const NodeHit& h, Stack& stack, int& smin, float lim, uint32_t* err,
                                        uint32_t& next) {
  constexpr int NO_HIT = 0x7fffffff;
  int k[8];
  // v_perm_b32 selector: byte 0 from the meta word (byte c & 3), bytes 1-3
  // from the distance
#pragma unroll
  for (int c = 0; c < 8; c++)
    k[c] = h.hit[c] ? (int)__builtin_amdgcn_perm(__float_as_uint(h.tn[c]), c < 4 ? h.meta_lo : h.meta_hi,
                                                 0x07060500u | (uint32_t)(c & 3))
                    : NO_HIT;
  auto ce = [&](int i, int j) {
    const int hi = max(k[i], k[j]), lo = min(k[i], k[j]);
    k[i] = hi;
    k[j] = lo;
  };
  ce(0, 1); ce(2, 3); ce(4, 5); ce(6, 7);
  ce(0, 2); ce(1, 3); ce(4, 6); ce(5, 7);
  ce(1, 2); ce(5, 6);
  ce(0, 4); ce(1, 5); ce(2, 6); ce(3, 7);
  ce(2, 4); ce(3, 5);
  ce(1, 2); ce(3, 4); ce(5, 6);
  // at most the pattern of +inf with a full low byte, below NO_HIT
  const int klim = max((int)__float_as_uint(lim), 0) | 0xff;
  if (k[7] > klim) return false;
  const uint32_t cb = h.cb, tb = h.tb;
  if (stack.fits()) {
#pragma unroll
    for (int j = 0; j < 7; j++) {
      if (k[j] <= klim) {
        const uint32_t y = pack_dist(k[j], smin);
        stack.put(make_uint2(meta_ref((uint32_t)k[j] & 0xffu, cb, tb), y));
      }
    }
  } else {
    raise_error(err, 1u);
  }
  next = meta_ref((uint32_t)k[7] & 0xffu, cb, tb);
  return true;
}

// A ray's best hit: none while geom is the invalid ID. (The first one is taken
// whatever its distance, which is NaN where T and |den| both overflow.) u = un / dn
// and v = vn / dn are divided when the hit is written: nearly every step of a wave
// improves some lane's hit, and would run the two divisions for it.
struct Hit {
  float t, un, vn, dn, ngx, ngy, ngz;
  uint32_t prim, geom;
};

__device__ inline float prod_diff(float a, float b, float c, float d) { return __builtin_fmaf(a, b, -(c * d)); }
__device__ inline float dot3(float ax, float ay, float az, float bx, float by, float bz) {
  return __builtin_fmaf(ax, bx, __builtin_fmaf(ay, by, az * bz));
}

// One triangle test. t is final; the hit's barycentrics are un/dn and vn/dn
// (divided only when the hit improves the current best).
struct TriTest {
  float t, un, vn, dn, ngx, ngy, ngz;
  uint32_t prim, geom, flags;
};

__device__ inline float sse_min(float a, float b) { return a < b ? a : b; }
__device__ inline float sse_max(float a, float b) { return a > b ? a : b; }

// PL = false: Moeller-Trumbore on the record (v0, e1 = v0-v1, e2 = v2-v0).
// PL = true: Pluecker (robust scenes) on the record (v0, v1, v2),
//   kernels/geometry/triangle_intersector_pluecker.h:55-110 and finalize
//   :29-36: edge functions of the origin-shifted vertices, eps = ulp*|U+V+W|,
//   stable_triangle_normal (common/math/vec3.h:210-222), den and T doubled,
//   t = T/den, u = U/UVW (U*0 when |UVW| < min_rcp_input), min/max of three
//   with SSE semantics; valid for tnear <= t <= tfar.
template <bool PL>
__device__ inline bool tri_test(const TRay& r, const TriRec* __restrict__ tp, TriTest& o) {
  const float4* p4 = reinterpret_cast<const float4*>(tp);
  const float4 a = p4[0], b = p4[1], c = p4[2];
  o.prim = __float_as_uint(a.w);
  o.geom = __float_as_uint(b.w);
  o.flags = __float_as_uint(c.w);
  if (!PL) {
    const float Cx = a.x - r.ox, Cy = a.y - r.oy, Cz = a.z - r.oz;
    // R = cross(C, D)
    const float Rx = prod_diff(Cy, r.dz, Cz, r.dy);
    const float Ry = prod_diff(Cz, r.dx, Cx, r.dz);
    const float Rz = prod_diff(Cx, r.dy, Cy, r.dx);
    // Ng = cross(e2, e1)
    o.ngx = prod_diff(c.y, b.z, c.z, b.y);
    o.ngy = prod_diff(c.z, b.x, c.x, b.z);
    o.ngz = prod_diff(c.x, b.y, c.y, b.x);
    const float den = dot3(o.ngx, o.ngy, o.ngz, r.dx, r.dy, r.dz);
    const float absDen = fabsf(den);
    const uint32_t sgn = __float_as_uint(den) & 0x80000000u;
    const float U = __uint_as_float(__float_as_uint(dot3(Rx, Ry, Rz, c.x, c.y, c.z)) ^ sgn);
    const float V = __uint_as_float(__float_as_uint(dot3(Rx, Ry, Rz, b.x, b.y, b.z)) ^ sgn);
    bool valid = (den != 0.0f) & (U >= 0.0f) & (V >= 0.0f) & (U + V <= absDen);
    const float T = __uint_as_float(__float_as_uint(dot3(o.ngx, o.ngy, o.ngz, Cx, Cy, Cz)) ^ sgn);
    valid &= (absDen * r.tnear < T) & (T <= absDen * r.tfar);
    if (valid) o.t = T / absDen;
    o.un = U;
    o.vn = V;
    o.dn = absDen;
    return valid;
  } else {
    const float v0x = a.x - r.ox, v0y = a.y - r.oy, v0z = a.z - r.oz;
    const float v1x = b.x - r.ox, v1y = b.y - r.oy, v1z = b.z - r.oz;
    const float v2x = c.x - r.ox, v2y = c.y - r.oy, v2z = c.z - r.oz;
    const float e0x = v2x - v0x, e0y = v2y - v0y, e0z = v2z - v0z;
    const float e1x = v0x - v1x, e1y = v0y - v1y, e1z = v0z - v1z;
    const float e2x = v1x - v2x, e2y = v1y - v2y, e2z = v1z - v2z;
    float sx = v2x + v0x, sy = v2y + v0y, sz = v2z + v0z;
    const float U = dot3(prod_diff(e0y, sz, e0z, sy), prod_diff(e0z, sx, e0x, sz), prod_diff(e0x, sy, e0y, sx),
                         r.dx, r.dy, r.dz);
    sx = v0x + v1x; sy = v0y + v1y; sz = v0z + v1z;
    const float V = dot3(prod_diff(e1y, sz, e1z, sy), prod_diff(e1z, sx, e1x, sz), prod_diff(e1x, sy, e1y, sx),
                         r.dx, r.dy, r.dz);
    sx = v1x + v2x; sy = v1y + v2y; sz = v1z + v2z;
    const float W = dot3(prod_diff(e2y, sz, e2z, sy), prod_diff(e2z, sx, e2x, sz), prod_diff(e2x, sy, e2y, sx),
                         r.dx, r.dy, r.dz);
    const float UVW = U + V + W;
    const float eps = 1.1920928955078125e-7f * fabsf(UVW);
    bool valid = (sse_min(sse_min(U, V), W) >= -eps) || (sse_max(sse_max(U, V), W) <= eps);
    // stable_triangle_normal(e0, e1, e2)
    const float ab_x = e0z * e1y, ab_y = e0x * e1z, ab_z = e0y * e1x;
    const float bc_x = e1z * e2y, bc_y = e1x * e2z, bc_z = e1y * e2x;
    o.ngx = fabsf(ab_x) < fabsf(bc_x) ? __builtin_fmaf(e0y, e1z, -ab_x) : __builtin_fmaf(e1y, e2z, -bc_x);
    o.ngy = fabsf(ab_y) < fabsf(bc_y) ? __builtin_fmaf(e0z, e1x, -ab_y) : __builtin_fmaf(e1z, e2x, -bc_y);
    o.ngz = fabsf(ab_z) < fabsf(bc_z) ? __builtin_fmaf(e0x, e1y, -ab_z) : __builtin_fmaf(e1x, e2y, -bc_z);
    const float d = dot3(o.ngx, o.ngy, o.ngz, r.dx, r.dy, r.dz);
    const float den = d + d;
    const float tt = dot3(v0x, v0y, v0z, o.ngx, o.ngy, o.ngz);
    const float T = tt + tt;
    o.t = T / den;
    valid &= (r.tnear <= o.t) & (o.t <= r.tfar) & (den != 0.0f);
    const bool tiny = fabsf(UVW) < MIN_RCP_INPUT;
    o.un = tiny ? U * 0.0f : U;
    o.vn = tiny ? V * 0.0f : V;
    o.dn = tiny ? 1.0f : UVW;
    return valid;
  }
}

template <bool ALIGNED>
__device__ inline void load_ray(const char* rp, float4& a, float4& b, float& tfar) {
  if (ALIGNED) {
    a = *reinterpret_cast<const float4*>(rp);
    b = *reinterpret_cast<const float4*>(rp + 16);
  } else {
    const float* f = reinterpret_cast<const float*>(rp);
    a = make_float4(f[0], f[1], f[2], f[3]);
    b = make_float4(f[4], f[5], f[6], f[7]);
  }
  tfar = *reinterpret_cast<const float*>(rp + 32);
}

template <bool OCCLUDED, bool ALIGNED, bool COUNT, int LDS_SLOTS, bool PL>
__global__ __launch_bounds__(TB) void k_trace(DevScene sc, char* __restrict__ rays, uint32_t M, uint64_t stride,
                                              uint32_t inst_id, uint32_t* __restrict__ cnt_nodes,
                                              uint32_t* __restrict__ cnt_tris, uint32_t* __restrict__ err,
                                              const uint32_t* __restrict__ perm, uint32_t* node_visits) {
  const uint32_t slot = blockIdx.x * TB + threadIdx.x;
  if (slot >= M) return;
  const uint32_t i = perm ? perm[slot] : slot;  // lanes take rays in spatially sorted order when given
  char* rp = rays + (uint64_t)i * stride;
  float4 a, b;
  float tfar;
  load_ray<ALIGNED>(rp, a, b, tfar);
  uint32_t nvis = 0, ntri = 0;
  if (!(a.w <= tfar)) {
    if (COUNT) { cnt_nodes[i] = 0; cnt_tris[i] = 0; }
    return;
  }
  TRay r;
  setup_ray(r, a, b, tfar);
  Hit best;
  best.t = INFINITY;
  best.prim = best.geom = 0xffffffffu;
  best.un = best.vn = best.dn = best.ngx = best.ngy = best.ngz = 0.0f;
  float lim = widen_up(tfar);

  __shared__ uint64_t lds_stack[LDS_SLOTS > 0 ? LDS_SLOTS * TB : 1];
  uint64_t spill_mem[STACK_CAP];
  RingStack<LDS_SLOTS> stack;
  stack.init(lds_stack, spill_mem);
  int smin = DIST_NONE;  // least entry distance on the stack (closest hit)
  uint32_t cur = sc.root;
  bool occluded = false;
  // every node and triangle record is reached at most once per ray, so the
  // loop runs at most num_nodes + num_tris times; the cap turns a corrupt
  // structure into an error instead of a hang
  // (node and triangle counts are below 2^31 each, so the bound fits 32 bits)
  const uint32_t max_iter = sc.num_nodes + sc.num_tris + 16u;
  uint32_t iter = 0;
  while (true) {
    if (++iter > max_iter) {
      raise_error(err, 2u);
      break;
    }
    if (!(cur & REF_LEAF)) {
      if (cur >= sc.num_nodes) {
        raise_error(err, 4u);
        break;
      }
      NodeHit h;
      intersect_node<OCCLUDED>(sc.nodes, cur, r, lim, h);
      if (COUNT) {
        nvis++;
        if (node_visits) atomicAdd(&node_visits[cur], 1u);
      }
      if (OCCLUDED ? push_any_order(h, stack, err, cur) : push_near_to_far(h, stack, smin, lim, err, cur)) {
        continue;
      }
    } else {
      uint32_t ti = cur & ~REF_LEAF;
      while (true) {
        if (ti >= sc.num_tris) {
          raise_error(err, 4u);
          break;
        }
        TriTest h;
        const bool valid = tri_test<PL>(r, sc.tris + ti, h);
        if (COUNT) ntri++;
        if (valid) {
          if (OCCLUDED) {
            occluded = true;
            break;
          }
          const bool better = best.geom == 0xffffffffu || h.t < best.t ||
                              (h.t == best.t && (h.geom < best.geom || (h.geom == best.geom && h.prim < best.prim)));
          if (better) {
            best.t = h.t;
            best.un = h.un; best.vn = h.vn; best.dn = h.dn;
            best.ngx = h.ngx; best.ngy = h.ngy; best.ngz = h.ngz;
            best.prim = h.prim; best.geom = h.geom;
          }
        }
        if (h.flags & TRI_LAST) break;
        ti++;
      }
      if (OCCLUDED && occluded) break;
      if (!OCCLUDED && best.geom != 0xffffffffu) lim = widen_up(fminf(best.t, tfar));
    }
    // pop the next entry that can still hold a closer hit
    bool got = false;
    const int dlim = dist_limit(lim);
    while (!stack.empty()) {
      const uint2 e = stack.pop();
      if (!OCCLUDED) smin = below_dist(e.y);
      if (OCCLUDED || (int)e.y <= dlim) {
        cur = e.x;
        got = true;
        break;
      }
      if (smin > dlim) {
        // every entry left is farther than the closest hit so far
        stack.clear();
        smin = DIST_NONE;
        break;
      }
    }
    if (!got) break;
  }
  if (COUNT) { cnt_nodes[i] = nvis; cnt_tris[i] = ntri; }
  if (OCCLUDED) {
    if (occluded) *reinterpret_cast<float*>(rp + 32) = -INFINITY;
  } else if (best.geom != 0xffffffffu) {
    float* f = reinterpret_cast<float*>(rp);
    uint32_t* u = reinterpret_cast<uint32_t*>(rp);
    f[8] = best.t;
    f[12] = best.ngx;
    f[13] = best.ngy;
    f[14] = best.ngz;
    f[15] = best.un / best.dn;
    f[16] = best.vn / best.dn;
    u[17] = best.prim;
    u[18] = best.geom;
    u[19] = inst_id;
  }
}

__device__ inline void write_hit(const Hit& best, char* rp, uint32_t inst_id) {
  float* f = reinterpret_cast<float*>(rp);
  uint32_t* u = reinterpret_cast<uint32_t*>(rp);
  f[8] = best.t;
  f[12] = best.ngx;
  f[13] = best.ngy;
  f[14] = best.ngz;
  f[15] = best.un / best.dn;
  f[16] = best.vn / best.dn;
  u[17] = best.prim;
  u[18] = best.geom;
  u[19] = inst_id;
}

// Persistent variant: a fixed grid of waves pulls rays from a global counter.
// A lane whose ray is finished takes a new one as soon as at least
// `refill_min` lanes of its wave are idle (and the hits of the ended rays are
// written then, all at once: the stores, the two divisions and the branch run
// for ten lanes or more instead of for one or two in nearly every step; 1920 x
// 1080 camera rays on a 2.1 M triangle terrain take 379 us, 407 before, the
// Pluecker test on a soup 995 us, 1092 before), so incoherent rays of very
// different lengths keep the SIMD lanes busy (Aila and Laine, "Understanding
// the efficiency of ray traversal on GPUs", HPG 2009). Each loop iteration is
// one traversal step (one node, or one leaf plus the pop that follows) for
// every active lane. Every wave leaves the loop once the counter has passed
// M and its lanes are idle.
// Resident 256-lane blocks per compute unit the persistent kernel is
// compiled for (one wave per SIMD each): the register budget follows from it.
// 6 (at most 80 VGPRs, no spills) measured fastest on the 2^20-triangle soup
// with 2^24 incoherent rays: 1655 Mrays/s closest hit against 1585 at 7 (72
// VGPRs, five of them spilled to scratch in the node step); 5 compiles to the
// same code as 6. A 16-entry LDS stack (32 KB per block) leaves room for 5.
constexpr int TRACE_MIN_BLOCKS = 6;

// The stream of a batch that ray slot `slot` belongs to.
__device__ inline const BatchItem& stream_of(const BatchItem* __restrict__ items, uint32_t nitems, uint32_t slot) {
  uint32_t lo = 0, hi = nitems - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (items[mid].first <= slot) lo = mid; else hi = mid - 1;
  }
  return items[lo];
}

// BATCH: the ray slots 0..M-1 are the concatenation of the streams in
// `items` (sorted by `first`); a lane finds its stream by binary search and
// starts at that stream's scene root.
template <bool OCCLUDED, bool ALIGNED, bool COUNT, int LDS_SLOTS, bool PL, bool BATCH = false>
__global__ __launch_bounds__(TB, LDS_SLOTS > 12 ? 5 : TRACE_MIN_BLOCKS) void k_trace_p(DevScene sc, char* __restrict__ rays, uint32_t M, uint64_t stride,
                                                uint32_t inst_id, uint32_t* __restrict__ cnt_nodes,
                                                uint32_t* __restrict__ cnt_tris, uint32_t* __restrict__ err,
                                                const uint32_t* __restrict__ perm, uint32_t* __restrict__ next,
                                                int refill_min, RayRuns rr, uint32_t* node_visits,
                                                const BatchItem* __restrict__ items, uint32_t nitems) {
  const int lane = threadIdx.x & 63;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  __shared__ uint64_t lds_stack[LDS_SLOTS > 0 ? LDS_SLOTS * TB : 1];
  uint64_t spill_mem[STACK_CAP];
  RingStack<LDS_SLOTS> stack;
  stack.init(lds_stack, spill_mem);
  int smin = DIST_NONE;  // least entry distance on the stack (closest hit)

  TRay r;
  Hit best;
  float lim = 0.0f;
  uint32_t cur = REF_IDLE, ray = 0, nvis = 0, ntri = 0;
  char* lrp = nullptr;      // BATCH: this lane's record
  uint32_t lroot = 0;       // BATCH: its scene's root
  bool pool_empty = false;
  WavePool pool;
  pool.init(rr, M);
  // a ray touches each node and triangle record at most once
  // (node and triangle counts are below 2^31 each, so the bound fits 32 bits)
  const uint32_t max_iter = sc.num_nodes + sc.num_tris + 16u;
  uint32_t iter = 0;

  while (true) {
    // ---- refill idle lanes (wave-uniform decision)
    const uint64_t idle = __ballot(cur >= REF_DONE);
    const int nidle = __popcll(idle);
    if (nidle >= (pool_empty ? 64 : refill_min)) {
      if (cur == REF_DONE) {
        cur = REF_IDLE;
        if (COUNT) { cnt_nodes[ray] = nvis; cnt_tris[ray] = ntri; }
        if (!OCCLUDED && best.geom != 0xffffffffu) write_hit(best, BATCH ? lrp : rays + (uint64_t)ray * stride, inst_id);
      }
      if (pool_empty) break;
      const uint32_t slot = pool.take(rr, next, M, nidle, (uint32_t)__popcll(idle & lt), lane);
      pool_empty = pool.empty();
      if (cur == REF_IDLE && slot != 0xffffffffu) {
        char* src;
        if (BATCH) {
          const BatchItem& it = stream_of(items, nitems, slot);
          ray = slot - it.first;
          lrp = it.rays + (uint64_t)ray * it.stride;
          lroot = it.root;
          src = lrp;
        } else {
          ray = perm ? perm[slot] : slot;
          src = rays + (uint64_t)ray * stride;
        }
        float4 a, b;
        float tfar;
        load_ray<ALIGNED>(src, a, b, tfar);
        if (a.w <= tfar) {
          setup_ray(r, a, b, tfar);
          best.t = INFINITY;
          best.prim = best.geom = 0xffffffffu;
          best.un = best.vn = best.dn = best.ngx = best.ngy = best.ngz = 0.0f;
          lim = widen_up(tfar);
          cur = BATCH ? lroot : sc.root;
          stack.init(lds_stack, spill_mem);
          smin = DIST_NONE;
          nvis = ntri = 0;
          iter = 0;
        } else if (COUNT) {
          cnt_nodes[ray] = 0;
          cnt_tris[ray] = 0;
        }
      }
    }

    // ---- one traversal step; a lane whose ray ends in it becomes REF_DONE
    if (++iter > max_iter && cur < REF_DONE) {
      raise_error(err, 2u);
      cur = REF_DONE;
    }
    if (!(cur & REF_LEAF)) {
      if (cur >= sc.num_nodes) {
        raise_error(err, 4u);
        cur = REF_DONE;
      } else {
        if (COUNT) {
          nvis++;
          if (node_visits) atomicAdd(&node_visits[cur], 1u);
        }
        NodeHit h;
        intersect_node<OCCLUDED>(sc.nodes, cur, r, lim, h);
        if (!(OCCLUDED ? push_any_order(h, stack, err, cur) : push_near_to_far(h, stack, smin, lim, err, cur)))
          cur = REF_EMPTY;
      }
    } else if (cur < REF_DONE) {
      // one triangle per step: a lane in a long leaf does not hold the
      // wave's other lanes in a triangle loop
      const uint32_t ti = cur & ~REF_LEAF;
      if (ti >= sc.num_tris) {
        raise_error(err, 4u);
        cur = REF_DONE;
      } else {
        TriTest h;
        const bool valid = tri_test<PL>(r, sc.tris + ti, h);
        if (COUNT) ntri++;
        cur = (h.flags & TRI_LAST) ? REF_EMPTY : cur + 1u;  // the leaf's next record
        if (valid) {
          if (OCCLUDED) {
            *reinterpret_cast<float*>((BATCH ? lrp : rays + (uint64_t)ray * stride) + 32) = -INFINITY;
            cur = REF_DONE;
          } else {
            const bool better = best.geom == 0xffffffffu || h.t < best.t ||
                                (h.t == best.t && (h.geom < best.geom || (h.geom == best.geom && h.prim < best.prim)));
            if (better) {
              best.t = h.t;
              best.un = h.un; best.vn = h.vn; best.dn = h.dn;
              best.ngx = h.ngx; best.ngy = h.ngy; best.ngz = h.ngz;
              best.prim = h.prim; best.geom = h.geom;
              lim = widen_up(fminf(best.t, r.tfar));
            }
          }
        }
      }
    }
    if (cur == REF_EMPTY) {
      // pop the next entry that can still hold a closer hit
      cur = REF_DONE;
      const int dlim = dist_limit(lim);
      while (!stack.empty()) {
        const uint2 e = stack.pop();
        if (!OCCLUDED) smin = below_dist(e.y);
        if (OCCLUDED || (int)e.y <= dlim) {
          cur = e.x;
          break;
        }
        if (smin > dlim) {
          // every entry left is farther than the closest hit so far
          stack.clear();
          smin = DIST_NONE;
          break;
        }
      }
    }
  }
}

// ------------------------------------------------------- small streams --

// A stream too small to fill the GPU with one ray per lane: eight lanes share
// a ray. In a node step lane c tests child c, in a leaf step triangle c of the
// leaf, and a pop looks at eight entries, so a step is a fraction of the
// one-lane kernels' instructions, and a wave waits for the longest of 8 rays
// instead of 64. What bounds it is the chain of dependent steps of the longest
// ray (about 0.8 us each, most of it the node's load): 1073 camera rays on a
// 131 k triangle terrain take 38 us a call, 85 with a lane a ray. Ray state is the same in a group's eight lanes; every branch depends on
// it (or on a ballot of the group), so the group stays together.
constexpr int GL = 8;            // lanes of a ray
constexpr int GR = 64 / GL;      // rays of a block (one wave)

template <int CTRL>
__device__ inline uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}
// The value of lane (c ^ X) of the group.
__device__ inline uint32_t gx1(uint32_t v) { return dpp<0xB1>(v); }   // quad_perm [1,0,3,2]
__device__ inline uint32_t gx2(uint32_t v) { return dpp<0x4E>(v); }   // quad_perm [2,3,0,1]
__device__ inline uint32_t gx3(uint32_t v) { return dpp<0x1B>(v); }   // quad_perm [3,2,1,0]
__device__ inline uint32_t gx7(uint32_t v) { return dpp<0x141>(v); }  // row_half_mirror
__device__ inline float gmin(float v) {
  v = fminf(v, __uint_as_float(gx1(__float_as_uint(v))));
  v = fminf(v, __uint_as_float(gx2(__float_as_uint(v))));
  return fminf(v, __uint_as_float(gx7(__float_as_uint(v))));
}

template <bool OCCLUDED, bool ALIGNED, bool PL, bool BATCH = false>
__global__ __launch_bounds__(64) void k_trace_g(DevScene sc, char* __restrict__ rays, uint32_t M, uint64_t stride,
                                                uint32_t inst_id, uint32_t* __restrict__ err, uint32_t cap,
                                                const BatchItem* __restrict__ items, uint32_t nitems) {
  extern __shared__ uint64_t group_stack[];  // cap entries for each ray, entry e of ray g at [e * GR + g]
  const uint32_t c = threadIdx.x & (GL - 1), g = threadIdx.x / GL;
  const uint32_t i = blockIdx.x * GR + g;
  if (i >= M) return;
  char* rp = rays + (uint64_t)i * stride;
  uint32_t root = sc.root;
  if (BATCH) {
    const BatchItem& it = stream_of(items, nitems, i);
    rp = it.rays + (uint64_t)(i - it.first) * it.stride;
    root = it.root;
  }
  float4 a, b;
  float tfar;
  load_ray<ALIGNED>(rp, a, b, tfar);
  if (!(a.w <= tfar)) return;
  TRay r;
  setup_ray(r, a, b, tfar);
  Hit best;  // the best of the triangles that this lane tested
  best.t = INFINITY;
  best.prim = best.geom = 0xffffffffu;
  best.un = best.vn = best.dn = best.ngx = best.ngy = best.ngz = 0.0f;
  float lim = widen_up(tfar);
  bool occluded = false;
  lds_u64* stack = (lds_u64*)group_stack + g;
  uint32_t sp = 0, cur = root;
  const uint32_t gshift = g * GL;
  auto group = [&](bool x) { return (uint32_t)(__ballot(x) >> gshift) & 0xffu; };
  // this lane's plane bytes: near and far of each axis
  const uint32_t onx = 32u + (r.negx ? 8u : 0u) + c, ony = 48u + (r.negy ? 8u : 0u) + c, onz = 64u + (r.negz ? 8u : 0u) + c;
  const uint32_t ofx = 72u + 2 * c - onx, ofy = 104u + 2 * c - ony, ofz = 136u + 2 * c - onz;  // (the other of the two)
  const uint32_t max_iter = sc.num_nodes + sc.num_tris + 16u;
  uint32_t iter = 0;
  while (true) {
    if (++iter > max_iter) {
      raise_error(err, 2u);
      break;
    }
    if (!(cur & REF_LEAF)) {
      if (cur >= sc.num_nodes) {
        raise_error(err, 4u);
        break;
      }
      const char* np = reinterpret_cast<const char*>(sc.nodes + cur);
      const uint4 w0 = *reinterpret_cast<const uint4*>(np), w1 = *reinterpret_cast<const uint4*>(np + 16);
      const uint8_t* nb = reinterpret_cast<const uint8_t*>(np);
      const float qnx = (float)nb[onx], qfx = (float)nb[ofx], qny = (float)nb[ony], qfy = (float)nb[ofy],
                  qnz = (float)nb[onz], qfz = (float)nb[ofz];
      const uint64_t meta = (uint64_t)w1.z | ((uint64_t)w1.w << 32);
      const uint32_t mb = (uint32_t)(meta >> (8 * c)) & 0xffu;
      // (the same operations as intersect_node())
      const float sx = __uint_as_float((w0.w & 0xffu) << 23), sy = __uint_as_float(((w0.w >> 8) & 0xffu) << 23),
                  sz = __uint_as_float(((w0.w >> 16) & 0xffu) << 23);
      const float dx = __uint_as_float(w0.x) - r.ox, dy = __uint_as_float(w0.y) - r.oy, dz = __uint_as_float(w0.z) - r.oz;
      const float tnx = __builtin_fmaf(qnx, sx * r.rnx, dx * r.rnx), tfx = __builtin_fmaf(qfx, sx * r.rfx, dx * r.rfx);
      const float tny = __builtin_fmaf(qny, sy * r.rny, dy * r.rny), tfy = __builtin_fmaf(qfy, sy * r.rfy, dy * r.rfy);
      const float tnz = __builtin_fmaf(qnz, sz * r.rnz, dz * r.rnz), tfz = __builtin_fmaf(qfz, sz * r.rfz, dz * r.rfz);
      const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, r.tlo));
      const float tf = fminf(fminf(tfx, tfy), fminf(tfz, lim));
      const bool hit = (tn <= tf) && (mb != 0u);
      const uint32_t mask = group(hit);
      if (mask) {
        const uint32_t cb = w1.x - 0x80u, tb = (w1.y | REF_LEAF) - 1u;
        const uint32_t n = (uint32_t)__popc(mask);
        uint32_t rank, first;
        if (OCCLUDED) {
          rank = (uint32_t)__popc(mask & ((1u << c) - 1u));
          first = (uint32_t)__builtin_ctz(mask);
        } else {
          // rank by entry distance; the low bits make the keys distinct
          const uint32_t key = hit ? (__float_as_uint(tn) & ~7u) | c : 0xffffffffu;
          const uint32_t m = gx7(key);
          rank = (gx1(key) < key) + (gx2(key) < key) + (gx3(key) < key) + (m < key) + (gx1(m) < key) + (gx2(m) < key) +
                 (gx3(m) < key);
          first = (uint32_t)__builtin_ctz(group(hit && rank == 0u));
        }
        if (sp + n > cap) {
          raise_error(err, 1u);
          break;
        }
        // the nearest is next, the others are pushed farthest first
        if (hit && rank > 0u)
          stack[(sp + n - 1u - rank) * GR] = pack_entry(make_uint2(meta_ref(mb, cb, tb), __float_as_uint(tn)));
        sp += n - 1u;
        cur = meta_ref((uint32_t)(meta >> (8 * first)) & 0xffu, cb, tb);
        continue;
      }
    } else {
      const uint32_t ti = cur & ~REF_LEAF;
      if (ti >= sc.num_tris) {
        raise_error(err, 4u);
        break;
      }
      TriTest h;
      bool valid = false;
      h.flags = 0u;
      if (c < sc.num_tris - ti) valid = tri_test<PL>(r, sc.tris + ti + c, h);
      // records up to the leaf's last one
      const uint32_t last = group((h.flags & TRI_LAST) != 0u);
      valid = valid && (last == 0u || c <= (uint32_t)__builtin_ctz(last));
      if (OCCLUDED) {
        if (group(valid)) {
          occluded = true;
          break;
        }
      } else {
        if (valid && (best.geom == 0xffffffffu || h.t < best.t ||
                      (h.t == best.t && (h.geom < best.geom || (h.geom == best.geom && h.prim < best.prim))))) {
          best.t = h.t;
          best.un = h.un; best.vn = h.vn; best.dn = h.dn;
          best.ngx = h.ngx; best.ngy = h.ngy; best.ngz = h.ngz;
          best.prim = h.prim; best.geom = h.geom;
        }
        if (group(valid)) lim = widen_up(fminf(gmin(best.t), tfar));
      }
      if (last == 0u) {
        cur += GL;
        continue;
      }
    }
    // pop the next entry that can still hold a closer hit, eight at a time
    bool got = false;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    while (sp > 0u) {
      const uint2 e = c < sp ? unpack_entry(stack[(sp - 1u - c) * GR]) : make_uint2(0u, 0x7f800000u);
      const uint32_t ok = group(c < sp && (OCCLUDED || __uint_as_float(e.y) <= lim));
      if (ok) {
        const uint32_t k = (uint32_t)__builtin_ctz(ok);
        sp -= k + 1u;
        cur = unpack_entry(stack[sp * GR]).x;
        got = true;
        break;
      }
      sp = sp > GL ? sp - GL : 0u;
    }
    if (!got) break;
  }
  if (OCCLUDED) {
    if (occluded && c == 0u) *reinterpret_cast<float*>(rp + 32) = -INFINITY;
    return;
  }
  // the least (t, geomID, primID) of the group; a lane that holds it writes it
  // (two may hold the same triangle, reached through two leaves). Distances as
  // ordered integers: NaN after every number, and a lane without a hit last.
  int t = __float_as_int(best.t + 0.0f);
  t = best.t != best.t || best.geom == 0xffffffffu ? 0x7fffffff : t ^ ((t >> 31) & 0x7fffffff);
  const int mine = t;
  uint32_t geom = best.geom, prim = best.prim;
  auto least = [&](int t2, uint32_t g2, uint32_t p2) {
    const bool less = t2 < t || (t2 == t && (g2 < geom || (g2 == geom && p2 < prim)));
    t = less ? t2 : t;
    geom = less ? g2 : geom;
    prim = less ? p2 : prim;
  };
  least((int)gx1((uint32_t)t), gx1(geom), gx1(prim));
  least((int)gx2((uint32_t)t), gx2(geom), gx2(prim));
  least((int)gx7((uint32_t)t), gx7(geom), gx7(prim));
  if (best.geom != 0xffffffffu && mine == t && best.geom == geom && best.prim == prim) {
    float* f = reinterpret_cast<float*>(rp);
    uint32_t* u = reinterpret_cast<uint32_t*>(rp);
    f[8] = best.t;
    f[12] = best.ngx;
    f[13] = best.ngy;
    f[14] = best.ngz;
    f[15] = best.un / best.dn;
    f[16] = best.vn / best.dn;
    u[17] = best.prim;
    u[18] = best.geom;
    u[19] = inst_id;
  }
}

// ------------------------------------------------------------- two-level --

// Two-level traversal of a scene with instances. The top tree's leaves are
// InstRec records; reaching one pushes a REF_INST_EXIT entry, moves the ray
// into the object's space with the record's world-to-object transform
// (kernels/geometry/instance_intersector.cpp:52-71 for closest hit, :73-98
// for occlusion) and continues at the object tree's root; popping the exit
// entry restores the world-space ray from its record. Both trees share one
// stack, so the current hit distance culls object entries and top entries
// alike (t has the same meaning in both spaces). Persistent and refilled as
// k_trace_p. Hits are ordered by (t, instID, geomID, primID).
// ctx_inst != RTC_INVALID_GEOMETRY_ID: the query context's one-level
// instance stack is already in use, so every instance push fails and only
// the scene's own triangles are tested (kernels/common/instance_stack.h:21-38).
template <bool OCCLUDED, bool ALIGNED, bool CNT = false>
__global__ __launch_bounds__(TB, 5) void k_trace_inst(DevTop top, char* __restrict__ rays, uint32_t M,
                                                      uint64_t stride, uint32_t ctx_inst, uint32_t* __restrict__ err,
                                                      uint32_t* __restrict__ next, int refill_min, RayRuns rr,
                                                      uint32_t* __restrict__ top_visits = nullptr,
                                                      uint32_t* __restrict__ obj_visits = nullptr,
                                                      uint32_t target_obj = 0xffffffffu) {
  const int lane = threadIdx.x & 63;
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  __shared__ uint64_t lds_stack[8 * TB];
  // the world-space ray and its reciprocals while the lane is in a moved
  // object (restored from here on the way out, not reloaded and divided again)
  __shared__ float4 lds_world[3 * TB];
  uint64_t spill_mem[STACK_CAP];
  RingStack<8> stack;
  stack.init(lds_stack, spill_mem);
  int smin = DIST_NONE;  // least entry distance on the stack (closest hit)

  // a ray that ends: closest hit, its hit is still to be finished
  constexpr uint32_t END = OCCLUDED ? REF_IDLE : REF_DONE;
  TRay r;
  Hit best;
  uint32_t best_inst = 0;
  float lim = 0.0f;
  uint32_t cur = REF_IDLE, ray = 0, inst = 0;
  // in an object tree (else the top tree); r in an instance's object space;
  // an object of a robust scene (bits of a register: a bool costs a lane mask)
  constexpr uint32_t IN_OBJ = 1u, MOVED = 2u, ROBUST = 4u;
  uint32_t where = 0u;
  const QNode8* onodes = nullptr;
  const TriRec* otris = nullptr;
  uint32_t onn = 0, otn = 0;
  uint32_t oidx = 0xffffffffu;  // the object the lane is in (counted variant)
  bool pool_empty = false;
  WavePool pool;
  pool.init(rr, M);
  const uint32_t max_iter = (uint32_t)min(top.max_iter, (uint64_t)0xffffffffu);
  uint32_t iter = 0;

  while (true) {
    // ---- refill idle lanes (wave-uniform decision)
    const uint64_t idle = __ballot(cur >= REF_DONE);
    const int nidle = __popcll(idle);
    if (nidle >= (pool_empty ? 64 : refill_min)) {
      if (!OCCLUDED && cur == REF_DONE) {
        cur = REF_IDLE;
        if (best.geom != 0xffffffffu) {
          float* f = reinterpret_cast<float*>(rays + (uint64_t)ray * stride);
          const float dn = f[8], un = f[15], vn = f[16];
          f[8] = best.t;
          f[15] = un / dn;
          f[16] = vn / dn;
        }
      }
      if (pool_empty) break;
      const uint32_t slot = pool.take(rr, next, M, nidle, (uint32_t)__popcll(idle & lt), lane);
      pool_empty = pool.empty();
      if (cur == REF_IDLE && slot != 0xffffffffu) {
        ray = slot;
        float4 a, b;
        float tfar;
        load_ray<ALIGNED>(rays + (uint64_t)ray * stride, a, b, tfar);
        if (a.w <= tfar) {
          setup_ray(r, a, b, tfar);
          best.t = INFINITY;
          best.prim = best.geom = 0xffffffffu;
          best.un = best.vn = best.dn = best.ngx = best.ngy = best.ngz = 0.0f;
          best_inst = 0xffffffffu;
          lim = widen_up(tfar);
          cur = top.root;
          where = 0u;
          stack.init(lds_stack, spill_mem);
          smin = DIST_NONE;
          iter = 0;
        }
      }
    }

    // ---- one traversal step
    if (++iter > max_iter && cur < REF_DONE) {
      raise_error(err, 2u);
      cur = END;
    }
    if (!(cur & REF_LEAF)) {
      const QNode8* nodes = where ? onodes : top.nodes;
      if (cur >= (where ? onn : top.num_nodes)) {
        raise_error(err, 4u);
        cur = END;
      } else {
        if (CNT) {
          if (!where) {
            if (top_visits) atomicAdd(top_visits + cur, 1u);
          } else if (obj_visits && oidx == target_obj) {
            atomicAdd(obj_visits + cur, 1u);
          }
        }
        NodeHit h;
        intersect_node<OCCLUDED>(nodes, cur, r, lim, h);
        if (!(OCCLUDED ? push_any_order(h, stack, err, cur) : push_near_to_far(h, stack, smin, lim, err, cur)))
          cur = REF_EMPTY;
      }
    } else if (cur < REF_DONE) {
      const uint32_t at = cur & ~REF_LEAF;
      if (at >= (where ? otn : top.num_insts)) {
        raise_error(err, 4u);
        cur = END;
      } else if (where) {
        // one triangle of the current object
        TriTest h;
        const bool valid = (where & ROBUST) ? tri_test<true>(r, otris + at, h) : tri_test<false>(r, otris + at, h);
        cur = (h.flags & TRI_LAST) ? REF_EMPTY : cur + 1u;
        if (valid) {
          if (OCCLUDED) {
            *reinterpret_cast<float*>(rays + (uint64_t)ray * stride + 32) = -INFINITY;
            cur = REF_IDLE;
          } else {
            const bool better =
                best.geom == 0xffffffffu || h.t < best.t ||
                (h.t == best.t &&
                 (inst < best_inst ||
                  (inst == best_inst &&
                   (h.geom < best.geom || (h.geom == best.geom && h.prim < best.prim)))));
            if (better) {
              // the hit goes to the record at once, so that only the fields
              // the comparison needs stay in registers; u and v wait there as
              // their numerators, with the denominator where the distance goes
              best.t = h.t;
              best.prim = h.prim;
              best.geom = h.geom;
              best_inst = inst;
              float* f = reinterpret_cast<float*>(rays + (uint64_t)ray * stride);
              uint32_t* u = reinterpret_cast<uint32_t*>(f);
              f[8] = h.dn;
              f[12] = h.ngx;
              f[13] = h.ngy;
              f[14] = h.ngz;
              f[15] = h.un;
              f[16] = h.vn;
              u[17] = h.prim;
              u[18] = h.geom;
              u[19] = inst;
              lim = widen_up(fminf(best.t, r.tfar));
            }
          }
        }
      } else {
        // an instance record of the top tree
        const float4* q = reinterpret_cast<const float4*>(top.insts + at);
        const float4 m0 = q[0], m1 = q[1], m2 = q[2];
        const uint4 w = reinterpret_cast<const uint4*>(top.insts + at)[3];
        const bool identity = (w.z & INST_IDENTITY) != 0u;
        // the rest of a multi-record leaf resumes after this instance
        if (!(w.z & TRI_LAST) && !stack.push(make_uint2((at + 1u) | REF_LEAF, pack_dist(DIST_ALWAYS, smin))))
          raise_error(err, 1u);
        cur = REF_EMPTY;
        if ((identity || ctx_inst == 0xffffffffu) && w.y < top.num_objects) {
          const DevScene o = top.objects[w.y];
          if (o.num_nodes > 0) {
            if (!stack.push(make_uint2(REF_INST_EXIT, pack_dist(DIST_ALWAYS, smin)))) raise_error(err, 1u);
            if (!identity) {
              lds_world[threadIdx.x] = make_float4(r.ox, r.oy, r.oz, r.dx);
              lds_world[TB + threadIdx.x] = make_float4(r.dy, r.dz, r.rnx, r.rny);
              lds_world[2 * TB + threadIdx.x] = make_float4(r.rnz, r.rfx, r.rfy, r.rfz);
              // columns vx = m[0..2], vy = m[3..5], vz = m[6..8], p = m[9..11]
              const float ox = __builtin_fmaf(r.ox, m0.x, __builtin_fmaf(r.oy, m0.w, __builtin_fmaf(r.oz, m1.z, m2.y)));
              const float oy = __builtin_fmaf(r.ox, m0.y, __builtin_fmaf(r.oy, m1.x, __builtin_fmaf(r.oz, m1.w, m2.z)));
              const float oz = __builtin_fmaf(r.ox, m0.z, __builtin_fmaf(r.oy, m1.y, __builtin_fmaf(r.oz, m2.x, m2.w)));
              const float dx = __builtin_fmaf(r.dx, m0.x, __builtin_fmaf(r.dy, m0.w, r.dz * m1.z));
              const float dy = __builtin_fmaf(r.dx, m0.y, __builtin_fmaf(r.dy, m1.x, r.dz * m1.w));
              const float dz = __builtin_fmaf(r.dx, m0.z, __builtin_fmaf(r.dy, m1.y, r.dz * m2.x));
              setup_ray(r, make_float4(ox, oy, oz, r.tnear), make_float4(dx, dy, dz, 0.0f), r.tfar);
              where = MOVED;
            }
            where |= IN_OBJ | (o.robust ? ROBUST : 0u);
            inst = identity ? ctx_inst : w.x;
            if (CNT) oidx = w.y;
            onodes = o.nodes;
            otris = o.tris;
            onn = o.num_nodes;
            otn = o.num_tris;
            cur = o.root;
          }
        }
      }
    }
    if (cur == REF_EMPTY) {
      // pop the next entry that can still hold a closer hit; an exit entry
      // returns the ray to world space
      cur = END;
      const int dlim = dist_limit(lim);
      while (!stack.empty()) {
        const uint2 e = stack.pop();
        if (!OCCLUDED) smin = below_dist(e.y);
        if (e.x == REF_INST_EXIT) {
          const bool moved = (where & MOVED) != 0u;
          where = 0u;
          if (moved) {
            const float4 a = lds_world[threadIdx.x], b = lds_world[TB + threadIdx.x];
            const float4 c = lds_world[2 * TB + threadIdx.x];
            r.ox = a.x; r.oy = a.y; r.oz = a.z; r.dx = a.w;
            r.dy = b.x; r.dz = b.y; r.rnx = b.z; r.rny = b.w;
            r.rnz = c.x; r.rfx = c.y; r.rfy = c.z; r.rfz = c.w;
            r.negx = !(r.rnx >= 0.0f);
            r.negy = !(r.rny >= 0.0f);
            r.negz = !(r.rnz >= 0.0f);
          }
          continue;
        }
        if (OCCLUDED || (int)e.y <= dlim) {
          cur = e.x;
          break;
        }
        if (smin > dlim) {
          // every entry left is farther than the closest hit so far
          stack.clear();
          smin = DIST_NONE;
          break;
        }
      }
    }
  }
}

__global__ void k_zero_counters(uint32_t* p) { p[threadIdx.x * COUNTER_STRIDE] = 0u; }

// Records of queries in host memory. What a query reads of a record is its
// first RAY_WORDS words, what it may write the distance and the hit: PCIe carries
// those 36 of 80 bytes each way, straight between pinned host memory and the
// device records (a word a thread, so that both sides' accesses are whole lines).
// A hit always writes its normal, and no hit's normal is NO_NORMAL (a NaN fails
// the hit tests).
__global__ __launch_bounds__(TB) void k_unpack_rays(const uint32_t* __restrict__ in, uint32_t* __restrict__ recs,
                                                    uint32_t words, uint32_t rec_words) {
  const uint32_t t = blockIdx.x * TB + threadIdx.x;
  if (t >= words) return;
  const uint32_t i = t / RAY_WORDS, w = t - i * RAY_WORDS;
  recs[(size_t)i * rec_words + w] = in[t];
  if (w == 0 && rec_words > 12) recs[(size_t)i * rec_words + 12] = NO_NORMAL;
}
__global__ __launch_bounds__(TB) void k_pack_hits(const uint32_t* __restrict__ recs, uint32_t* __restrict__ out,
                                                  uint32_t words, uint32_t rec_words) {
  const uint32_t t = blockIdx.x * TB + threadIdx.x;
  if (t >= words) return;
  const uint32_t per = rec_words > 12 ? HIT_WORDS : 1u, i = t / per, w = t - i * per;
  out[t] = recs[(size_t)i * rec_words + (w == 0 ? 8u : 11u + w)];
}

// Sort key of a ray: 30-bit Morton code of its origin in the scene box
// (origins outside are clamped to the box faces); inactive rays sort last.
__global__ __launch_bounds__(TB) void k_ray_keys(const char* __restrict__ rays, uint32_t M, uint64_t stride, float lx,
                                                 float ly, float lz, float sx, float sy, float sz,
                                                 uint32_t* __restrict__ keys, uint32_t* __restrict__ vals) {
  const uint32_t i = blockIdx.x * TB + threadIdx.x;
  if (i >= M) return;
  const float* f = reinterpret_cast<const float*>(rays + (uint64_t)i * stride);
  const float ox = f[0], oy = f[1], oz = f[2], tnear = f[3], tfar = f[8];
  uint32_t key = 0xffffffffu;
  if (tnear <= tfar) {
    const uint32_t qx = (uint32_t)fminf(fmaxf((ox - lx) * sx, 0.0f), 1023.0f);
    const uint32_t qy = (uint32_t)fminf(fmaxf((oy - ly) * sy, 0.0f), 1023.0f);
    const uint32_t qz = (uint32_t)fminf(fmaxf((oz - lz) * sz, 0.0f), 1023.0f);
    key = spread3(qx) | (spread3(qy) << 1) | (spread3(qz) << 2);
  }
  keys[i] = key;
  vals[i] = i;
}

// Grid and runs of a persistent launch over M rays, and whether it needs the
// counters (runs beyond every wave's first).
struct RayPlan {
  dim3 grid;
  RayRuns runs;
  bool counter;
};

RayPlan ray_plan(uint32_t M, int resident, const TraceParams& tp) {
  // no more blocks than are resident at once: a wave's own first run must not
  // wait for another wave to end
  const uint32_t per_cu = (uint32_t)std::max(1, std::min(tp.blocks_per_cu, resident));
  const uint32_t runs = div_up(M, RAY_RUN);
  uint32_t blocks = std::min((uint32_t)tp.cus * per_cu, div_up(runs, TB / 64));
  const uint32_t qs = blocks >= COUNTERS ? COUNTERS_LOG2 : 0u;  // (a grid is a multiple of its queues)
  blocks = (((blocks - 1u) >> qs) + 1u) << qs;
  return {dim3(blocks), {runs, qs}, (uint64_t)blocks * (TB / 64) < runs};
}

// Resident blocks per compute unit of a kernel (asked once per kernel).
template <auto KERNEL>
int resident_blocks() {
  static const int n = [] {
    int b = 0;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, KERNEL, TB, 0) == hipSuccess && b > 0 ? b : TRACE_MIN_BLOCKS;
  }();
  return n;
}

struct LaunchArgs {
  DevScene sc;
  char* rays;
  uint32_t M;
  uint64_t stride;
  uint32_t inst_id;
  uint32_t *cnt_nodes, *cnt_tris, *err;
  const uint32_t* perm;
  uint32_t* counter;
  int refill;
  uint32_t* node_visits;
  bool persistent;
  const TraceParams* tp;
  hipStream_t s;
};

template <bool OCC, bool AL, bool CNT, int SL, bool PL>
void launch_one(const LaunchArgs& a) {
  if (!a.persistent) {
    hipLaunchKernelGGL((k_trace<OCC, AL, CNT, SL, PL>), dim3(div_up(a.M, TB)), dim3(TB), 0, a.s, a.sc, a.rays, a.M,
                       a.stride, a.inst_id, a.cnt_nodes, a.cnt_tris, a.err, a.perm, a.node_visits);
    return;
  }
  const RayPlan p = ray_plan(a.M, resident_blocks<k_trace_p<OCC, AL, CNT, SL, PL>>(), *a.tp);
  if (p.counter) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(COUNTERS), 0, a.s, a.counter);
  hipLaunchKernelGGL((k_trace_p<OCC, AL, CNT, SL, PL>), p.grid, dim3(TB), 0, a.s, a.sc, a.rays, a.M, a.stride,
                     a.inst_id, a.cnt_nodes, a.cnt_tris, a.err, a.perm, a.counter, a.refill, p.runs, a.node_visits,
                     nullptr, 0u);
}

template <bool OCC, bool AL, bool CNT, bool PL>
void launch_slots(const LaunchArgs& a) {
  if (a.tp->lds_slots <= 0) launch_one<OCC, AL, CNT, 0, PL>(a);
  else if (a.tp->lds_slots <= 8) launch_one<OCC, AL, CNT, 8, PL>(a);
  else if (a.tp->lds_slots <= 12) launch_one<OCC, AL, CNT, 12, PL>(a);
  else launch_one<OCC, AL, CNT, 16, PL>(a);
}

// The largest streams that eight lanes a ray serve better (kernel us, eight
// lanes against one):
//                                      8192       32768       49152       65536
//   camera, 131 k terrain             49 :  85   53 :  87    66 :  96    69 :  80
//   camera, 2.1 M terrain             64 : 107   81 : 111    90 : 131    85 : 119
//   camera, 16 k sphere               49 :  73   59 :  79    67 :  84    73 :  80
//   random, 250 k sphere              70 : 105   86 : 116   104 : 117   111 : 127
//   random, 2^20 soup                262 : 394  280 : 408   313 : 397   351 : 401
//   random, 262 k soup               147 : 247  197 : 243   223 : 240   265 : 236
//   random, 262 k soup, robust       153 : 253  193 : 255   237 : 251   277 : 250
//   random occlusion, 262 k soup      33 :  52   53 :  57    59 :  58    59 :  59
//   random occlusion, 2^20 soup       46 :  68   75 :  85    82 :  85    83 :  84
//   camera occlusion, 131 k terrain   39 :  63   41 :  71    72 :  72    62 :  65
// The GPU fills up there, and one lane a ray needs fewer instructions. At 65536
// closest-hit rays five of seven still gain, 9 to 29 %, and two lose 11 and 12 %.
constexpr uint32_t GROUP_MAX_RAYS = 65536, GROUP_MAX_RAYS_OCC = 32768;
// A ray's stack is all in LDS: 256 entries are 16 KB a wave. (Trees of a few
// million triangles need fewer than 80.)
constexpr uint32_t GROUP_MAX_STACK = 256;

bool use_groups(const DevScene& sc, uint32_t M, bool occluded, const TraceParams& tp) {
  return tp.persistent && tp.groups && M <= (occluded ? GROUP_MAX_RAYS_OCC : GROUP_MAX_RAYS) && sc.max_stack < GROUP_MAX_STACK;
}

template <bool OCC, bool AL, bool PL>
void launch_group(const LaunchArgs& a) {
  const uint32_t cap = a.sc.max_stack + 1u;
  hipLaunchKernelGGL((k_trace_g<OCC, AL, PL>), dim3(div_up(a.M, GR)), dim3(64), cap * GR * 8, a.s, a.sc, a.rays, a.M,
                     a.stride, a.inst_id, a.err, cap, nullptr, 0u);
}

template <bool PL>
void launch_pl(const LaunchArgs& a, bool count, bool occluded, bool aligned) {
  if (!count && !a.perm && use_groups(a.sc, a.M, occluded, *a.tp)) {
    if (occluded) {
      if (aligned) launch_group<true, true, PL>(a);
      else launch_group<true, false, PL>(a);
    } else {
      if (aligned) launch_group<false, true, PL>(a);
      else launch_group<false, false, PL>(a);
    }
    return;
  }
  if (count) {
    if (occluded) launch_slots<true, false, true, PL>(a);
    else launch_slots<false, false, true, PL>(a);
  } else if (occluded) {
    if (aligned) launch_slots<true, true, false, PL>(a);
    else launch_slots<true, false, false, PL>(a);
  } else {
    if (aligned) launch_slots<false, true, false, PL>(a);
    else launch_slots<false, false, false, PL>(a);
  }
}

void launch_trace(const DevScene& sc, void* rays, uint32_t M, uint64_t stride, bool occluded, uint32_t inst_id,
                  uint32_t* cnt_nodes, uint32_t* cnt_tris, uint32_t* err, hipStream_t s, const TraceParams& tp,
                  RaySorter* sorter, uint32_t* node_visits, uint32_t* counter) {
  if (M == 0 || sc.num_nodes == 0) return;
  const bool aligned = ((uintptr_t)rays % 16 == 0) && (stride % 16 == 0);
  const dim3 grid(div_up(M, TB)), block(TB);
  char* rp = (char*)rays;
  const bool count = cnt_nodes != nullptr;
  const uint32_t* perm = nullptr;
  if (tp.sort_rays && sorter && M >= tp.sort_min) {
    sorter->keys.reserve((size_t)M * 4);
    sorter->vals.reserve((size_t)M * 4);
    hipLaunchKernelGGL(k_ray_keys, grid, block, 0, s, rp, M, stride, sc.lo[0], sc.lo[1], sc.lo[2], sc.scale[0],
                       sc.scale[1], sc.scale[2], sorter->keys.as<uint32_t>(), sorter->vals.as<uint32_t>());
    sorter->sort.sort_pairs(sorter->keys.as<uint32_t>(), sorter->vals.as<uint32_t>(), M, 0, 32, s);
    perm = sorter->vals.as<uint32_t>();
  }
  const bool persistent = tp.persistent && (sorter || counter);
  const int rmin = occluded ? tp.refill_min_occ : tp.refill_min;
  const int refill = rmin < 1 ? 1 : (rmin > 64 ? 64 : rmin);  // 64 idle lanes always refill
  if (persistent && !counter) {
    sorter->counter.reserve(COUNTER_BYTES);
    counter = sorter->counter.as<uint32_t>();
  }
  LaunchArgs la{sc, rp, M, stride, inst_id, cnt_nodes, cnt_tris, err, perm, persistent ? counter : nullptr, refill,
                count ? node_visits : nullptr, persistent, &tp, s};
  if (sc.robust) launch_pl<true>(la, count, occluded, aligned);
  else launch_pl<false>(la, count, occluded, aligned);
  RTG_HIP(hipGetLastError());
}

template <bool OCC, bool AL, bool PL, int SL>
void launch_batch_slots(const DevScene& sc, const BatchItem* items, uint32_t nitems, uint32_t M, uint32_t* err,
                        uint32_t* counter, hipStream_t s, const TraceParams& tp) {
  const int rmin = OCC ? tp.refill_min_occ : tp.refill_min;
  const int refill = rmin < 1 ? 1 : (rmin > 64 ? 64 : rmin);
  if (use_groups(sc, M, OCC, tp)) {
    const uint32_t cap = sc.max_stack + 1u;
    hipLaunchKernelGGL((k_trace_g<OCC, AL, PL, true>), dim3(div_up(M, GR)), dim3(64), cap * GR * 8, s, sc,
                       (char*)nullptr, M, (uint64_t)0, 0xffffffffu, err, cap, items, nitems);
    return;
  }
  const RayPlan p = ray_plan(M, resident_blocks<k_trace_p<OCC, AL, false, SL, PL, true>>(), tp);
  if (p.counter) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(COUNTERS), 0, s, counter);
  hipLaunchKernelGGL((k_trace_p<OCC, AL, false, SL, PL, true>), p.grid, dim3(TB), 0, s, sc, (char*)nullptr, M,
                     (uint64_t)0, 0xffffffffu, (uint32_t*)nullptr, (uint32_t*)nullptr, err, (const uint32_t*)nullptr,
                     counter, refill, p.runs, (uint32_t*)nullptr, items, nitems);
}

// (LDS stack rings of 8 or of 12 entries per lane: lds_slots up to 8, or more)
template <bool OCC, bool AL, bool PL>
void launch_batch_one(const DevScene& sc, const BatchItem* items, uint32_t nitems, uint32_t M, uint32_t* err,
                      uint32_t* counter, hipStream_t s, const TraceParams& tp) {
  if (tp.lds_slots <= 8) launch_batch_slots<OCC, AL, PL, 8>(sc, items, nitems, M, err, counter, s, tp);
  else launch_batch_slots<OCC, AL, PL, 12>(sc, items, nitems, M, err, counter, s, tp);
}

void launch_trace_batch(const DevScene& sc, const BatchItem* items, uint32_t nitems, uint32_t M, bool occluded,
                        bool aligned, uint32_t* err, uint32_t* counter, hipStream_t s, const TraceParams& tp) {
  if (M == 0 || nitems == 0 || sc.num_nodes == 0) return;
  if (sc.robust) {
    if (occluded) {
      if (aligned) launch_batch_one<true, true, true>(sc, items, nitems, M, err, counter, s, tp);
      else launch_batch_one<true, false, true>(sc, items, nitems, M, err, counter, s, tp);
    } else {
      if (aligned) launch_batch_one<false, true, true>(sc, items, nitems, M, err, counter, s, tp);
      else launch_batch_one<false, false, true>(sc, items, nitems, M, err, counter, s, tp);
    }
  } else {
    if (occluded) {
      if (aligned) launch_batch_one<true, true, false>(sc, items, nitems, M, err, counter, s, tp);
      else launch_batch_one<true, false, false>(sc, items, nitems, M, err, counter, s, tp);
    } else {
      if (aligned) launch_batch_one<false, true, false>(sc, items, nitems, M, err, counter, s, tp);
      else launch_batch_one<false, false, false>(sc, items, nitems, M, err, counter, s, tp);
    }
  }
  RTG_HIP(hipGetLastError());
}

template <bool OCC, bool AL, bool CNT>
void launch_inst_one(const DevTop& top, char* rays, uint32_t M, uint64_t stride, uint32_t ctx_inst, uint32_t* err,
                     uint32_t* counter, int refill, hipStream_t s, const TraceParams& tp, uint32_t* top_visits,
                     uint32_t* obj_visits, uint32_t target_obj) {
  const RayPlan p = ray_plan(M, resident_blocks<k_trace_inst<OCC, AL, CNT>>(), tp);
  if (p.counter) hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(COUNTERS), 0, s, counter);
  hipLaunchKernelGGL((k_trace_inst<OCC, AL, CNT>), p.grid, dim3(TB), 0, s, top, rays, M, stride, ctx_inst, err,
                     counter, refill, p.runs, top_visits, obj_visits, target_obj);
}

void launch_trace_inst(const DevTop& top, void* rays, uint32_t M, uint64_t stride, bool occluded, uint32_t ctx_inst,
                       uint32_t* err, hipStream_t s, const TraceParams& tp, RaySorter* sorter, uint32_t* counter) {
  if (M == 0 || top.num_nodes == 0) return;
  const bool aligned = ((uintptr_t)rays % 16 == 0) && (stride % 16 == 0);
  const int rmin = occluded ? tp.refill_min_occ_inst : tp.refill_min;
  const int refill = rmin < 1 ? 1 : (rmin > 64 ? 64 : rmin);
  if (!counter) {
    sorter->counter.reserve(COUNTER_BYTES);
    counter = sorter->counter.as<uint32_t>();
  }
  char* rp = (char*)rays;
  auto go = [&](auto occ, auto al) {
    launch_inst_one<occ(), al(), false>(top, rp, M, stride, ctx_inst, err, counter, refill, s, tp, nullptr, nullptr,
                                        0xffffffffu);
  };
  using T = std::true_type;
  using F = std::false_type;
  if (occluded) {
    if (aligned) go(T(), T());
    else go(T(), F());
  } else {
    if (aligned) go(F(), T());
    else go(F(), F());
  }
  RTG_HIP(hipGetLastError());
}

void launch_trace_inst_counted(const DevTop& top, void* rays, uint32_t M, uint64_t stride, uint32_t* err,
                               uint32_t* counter, uint32_t* top_visits, uint32_t* obj_visits, uint32_t target_obj,
                               hipStream_t s, const TraceParams& tp) {
  if (M == 0 || top.num_nodes == 0) return;
  const bool aligned = ((uintptr_t)rays % 16 == 0) && (stride % 16 == 0);
  const int refill = tp.refill_min < 1 ? 1 : (tp.refill_min > 64 ? 64 : tp.refill_min);
  char* rp = (char*)rays;
  if (aligned)
    launch_inst_one<false, true, true>(top, rp, M, stride, 0xffffffffu, err, counter, refill, s, tp, top_visits,
                                       obj_visits, target_obj);
  else
    launch_inst_one<false, false, true>(top, rp, M, stride, 0xffffffffu, err, counter, refill, s, tp, top_visits,
                                        obj_visits, target_obj);
  RTG_HIP(hipGetLastError());
}

void unpack_rays(const uint32_t* in, void* recs, uint32_t n, bool occluded, hipStream_t s) {
  hipLaunchKernelGGL(k_unpack_rays, dim3(div_up((size_t)n * RAY_WORDS, TB)), dim3(TB), 0, s, in, (uint32_t*)recs,
                     n * RAY_WORDS, occluded ? 12u : 20u);
}

void pack_hits(const void* recs, uint32_t* out, uint32_t n, bool occluded, hipStream_t s) {
  const uint32_t words = n * (occluded ? 1u : HIT_WORDS);
  hipLaunchKernelGGL(k_pack_hits, dim3(div_up(words, TB)), dim3(TB), 0, s, (const uint32_t*)recs, out, words,
                     occluded ? 12u : 20u);
}

namespace {
constexpr int NOALLOC_MAX_GPUS = 64;
std::mutex g_noalloc_mtx;
uint32_t* g_noalloc_ptr[NOALLOC_MAX_GPUS] = {};

__global__ void k_fill_words(uint32_t* p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * TB + threadIdx.x;
  if (i < n) p[i] = v;
}
}  // namespace

void noalloc_setup(int ordinal) {
  if (ordinal < 0 || ordinal >= NOALLOC_MAX_GPUS) throw hip_error(hipErrorInvalidDevice, "GPU ordinal out of range");
  std::lock_guard<std::mutex> g(g_noalloc_mtx);
  if (g_noalloc_ptr[ordinal]) return;
  void* p = nullptr;
  const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
  if (e != hipSuccess || p == nullptr)
    throw hip_error(e != hipSuccess ? e : hipErrorInvalidSymbol,
                    std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
  g_noalloc_ptr[ordinal] = static_cast<uint32_t*>(p);
}

uint32_t* noalloc_scratch(int ordinal) {
  if (ordinal < 0 || ordinal >= NOALLOC_MAX_GPUS) return nullptr;
  std::lock_guard<std::mutex> g(g_noalloc_mtx);
  return g_noalloc_ptr[ordinal];
}

void fill_words(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_fill_words, dim3(div_up(n, TB)), dim3(TB), 0, s, p, n, v);
  RTG_HIP(hipGetLastError());
}

}  // namespace rtg

