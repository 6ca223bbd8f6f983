// Traversal kernel launcher.
#pragma once
#include "bvh_types.h"
#include "gpu_util.h"
#include "sort.h"

namespace rtg {

// Launch-shape parameters of the traversal (chosen per device, tunable).
struct TraceParams {
  // LDS stack entries per lane (0: private stack, 8, 12 or 16). On the
  // 2^20-triangle soup 2^24 incoherent rays, closest hit, take 6.26 ms at 12,
  // 6.64 at 8 and 6.92 at 16 (16 fits 5 blocks of 256 lanes per CU, 12 and 8
  // fit 6), 14.5 with a private stack; 2^23 occlusion rays there 1.96, 2.03,
  // 2.18 and 3.65.
  int lds_slots = 12;
  int sort_rays = 0;        // trace in origin-Morton order (a permutation; records stay in place)
  uint32_t sort_min = 65536;  // smallest stream that is reordered
  int persistent = 1;       // persistent waves pulling rays from a counter
  // Idle lanes of a wave that trigger a refill. A refill stalls the wave
  // for one ray-record load (and, once per RAY_RUN rays, a global counter's
  // atomic). The line is flat: 2^24 rays in the 2^20-triangle soup take 6.24 ms
  // at 8, 6.25 at 10, 6.28 at 16, 6.33 at 24 and 6.52 at 32; the Pluecker test
  // on a soup (985 to 1014 us) and camera rays on a terrain (322 to 332) show no
  // order from 6 to 20. Occlusion rays, 2^23 in the soup: 1.98 ms at 8, 1.96 at
  // 16, 1.97 at 24, 1.99 at 32 and 2.08 at 40; camera rays on a terrain 260, 260,
  // 256, 264 and 264 us.
  int refill_min = 10;      // closest hit
  int refill_min_occ = 24;  // occlusion rays, which finish sooner
  // Occlusion rays through a two-level scene: two million camera rays through
  // 10,000 instances and their shadow rays take 2.65 ms at 6, 2.69 at 8, 2.64 at
  // 12, 2.65 at 16, 2.68 at 20 and 2.76 at 24 (closest hit and occlusion alike).
  int refill_min_occ_inst = 12;
  int groups = 1;           // small streams with eight lanes a ray (0: one lane, as large ones)
  int cus = 256;            // compute units (set from the device)
  int blocks_per_cu = 8;    // 256-thread blocks per compute unit for the persistent grid (at most those resident)
};

// Ray counters of a persistent launch, one for each XCD, 256 B apart.
constexpr uint32_t COUNTERS_LOG2 = 3, COUNTERS = 1u << COUNTERS_LOG2;
constexpr uint32_t COUNTER_STRIDE = 64;  // in words
constexpr size_t COUNTER_BYTES = COUNTERS * COUNTER_STRIDE * 4;

// One ray stream of a batched traversal (device memory).
struct BatchItem {
  char* rays;        // records, `stride` bytes apart
  uint64_t stride;
  uint32_t first;    // slot of its first ray in the concatenation of all streams
  uint32_t count;
  uint32_t root;     // root node of its scene
  uint32_t pad;
};

// Per-thread buffers of the ray reordering.
struct RaySorter {
  DevBuf keys, vals, counter;
  RadixSorter sort;
};

// Traces M ray records (RTCRayHit for closest hit, RTCRay for occlusion)
// spaced `stride` bytes apart in device memory, in place. cnt_nodes /
// cnt_tris (optional, M entries each) receive per-ray node visits and
// triangle tests. err (device or pinned host memory) receives
// bit 0 on a traversal stack overflow.
// node_visits (optional, with the counters): one atomic increment per node
// visit, indexed like the QNode8 array.
// counter (optional): the persistent kernel's ray counters (COUNTER_BYTES);
// without it the sorter's is used, and with neither the grid covers every ray.
void launch_trace(const DevScene& sc, void* rays, uint32_t M, uint64_t stride, bool occluded, uint32_t inst_id,
                  uint32_t* cnt_nodes, uint32_t* cnt_tris, uint32_t* err, hipStream_t s,
                  const TraceParams& tp, RaySorter* sorter, uint32_t* node_visits = nullptr,
                  uint32_t* counter = nullptr);

// One persistent launch over several ray streams of scenes that share sc's
// node and triangle arrays (a batched build). items (device memory) sorted
// by first; M = total rays. Records traced in place. counter:
// COUNTER_BYTES of device memory, cleared by a kernel (the sequence can be captured in a hipGraph).
void launch_trace_batch(const DevScene& sc, const BatchItem* items, uint32_t nitems, uint32_t M, bool occluded,
                        bool aligned, uint32_t* err, uint32_t* counter, hipStream_t s, const TraceParams& tp);

// Two-level traversal of a scene with instances (top tree over InstRec
// leaves, object trees in top.objects); otherwise as launch_trace. ctx_inst
// is the query context's instID[0]; counter (COUNTER_BYTES) or, if null,
// the sorter's supplies the ray counters.
void launch_trace_inst(const DevTop& top, void* rays, uint32_t M, uint64_t stride, bool occluded, uint32_t ctx_inst,
                       uint32_t* err, hipStream_t s, const TraceParams& tp, RaySorter* sorter,
                       uint32_t* counter = nullptr);

// Closest-hit two-level traversal that also counts the rays that enter each
// node of the top tree (top_visits, one word per top node, may be null) and
// of object target_obj's tree (obj_visits, one word per node of that object,
// summed over all its instances; may be null).
void launch_trace_inst_counted(const DevTop& top, void* rays, uint32_t M, uint64_t stride, uint32_t* err,
                               uint32_t* counter, uint32_t* top_visits, uint32_t* obj_visits, uint32_t target_obj,
                               hipStream_t s, const TraceParams& tp);

// Words of a record that a query reads, and of RTCRayHit that a hit writes (the
// distance, then words 12 to 19).
constexpr uint32_t RAY_WORDS = 9, HIT_WORDS = 9;
constexpr uint32_t NO_NORMAL = 0x7fffffffu;  // first word of the normal of a record without a hit
// n device records (80 B RTCRayHit or 48 B RTCRay) from their RAY_WORDS words,
// and what the query wrote of them (HIT_WORDS, or for occlusion the distance).
// in and out: pinned host memory. n is below 2^24.
void unpack_rays(const uint32_t* in, void* recs, uint32_t n, bool occluded, hipStream_t s);
void pack_hits(const void* recs, uint32_t* out, uint32_t n, bool occluded, hipStream_t s);

// Scratch of the no-allocation queries: the persistent kernel's ray counters
// (the words at multiples of COUNTER_STRIDE), with the traversal error bits
// in word 1; one fixed array per GPU, held until the process ends.
constexpr uint32_t NOALLOC_SCRATCH_WORDS = COUNTERS * COUNTER_STRIDE;
constexpr uint32_t NOALLOC_MAX_RAYS = 1u << 31;  // the counter word's range, with room for every wave's overshoot
// Looks up the device address of this GPU's copy of the scratch array; the
// GPU `ordinal` must be current. Once per GPU (later calls return at once);
// throws hip_error when the lookup fails.
void noalloc_setup(int ordinal);
// Device address of GPU `ordinal`'s scratch array, or nullptr before noalloc_setup.
uint32_t* noalloc_scratch(int ordinal);
// Writes v to n words at p on stream s (a kernel, so the call can be captured).
void fill_words(uint32_t* p, uint32_t n, uint32_t v, hipStream_t s);

}  // namespace rtg
