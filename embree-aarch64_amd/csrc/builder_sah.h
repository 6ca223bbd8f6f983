// Top-down binned-SAH binary tree over the valid primitive references, built
// level by level on the GPU. Its output has the same form as the radix tree
// of the Morton builder (child / parent / range arrays over final primitive
// positions), so the bottom-up SAH refit and the 8-wide collapse run on
// either tree unchanged.
#pragma once
#include <vector>

#include "bvh_types.h"
#include "gpu_util.h"
#include "mlp.h"

namespace rtg {

struct SahScratch {
  DevBuf idx[2], blo[2], bhi[2], sid[2], segs[3][3], tiny, bins[2], splits, below, before, counters, roots;
  PinnedBuf stage;  // the trees' segments, read by the first kernel
  HostPost post;    // a level's counts, read while it runs
};

// One tree of the forest: positions [first, first+count), count >= 2.
struct SahRoot {
  uint32_t first, count;
  float clo[3], chi[3];  // bounds of lo+hi over its references
};

// Where the device finds the trees' root ids (NIL, 0xffffffff, if missing) and
// the build's error bits, once the work queued on the stream has run.
struct SahRoots {
  const uint32_t* roots = nullptr;
  const uint32_t* error = nullptr;
};

// Inputs: n valid references, `vals` holding their primref indices and
// slo/shi their boxes in that order, and the trees to build (disjoint
// position ranges of at least two references). Outputs: vals reordered so
// that every inner node covers a contiguous position range; child/
// parent_int/parent_leaf/range filled for the inner nodes (an inner node's
// id is its split position, so ids lie in [0, n-2]; ids no tree uses keep
// parent_int = REF_EMPTY).
// `learned` (may be null) replaces the half-area term of the split cost.
// The build is still queued on the stream when the call returns.
// Segments of at most median_below (<= 64) references are split at their
// median position all the way down instead of by binned SAH.
void build_sah_tree(uint32_t n, uint32_t* vals, const float4* slo, const float4* shi,
                    const std::vector<SahRoot>& trees, uint32_t* child, uint32_t* parent_int,
                    uint32_t* parent_leaf, uint2* range, const LearnedCost* learned,
                    uint32_t median_below, SahScratch& S, SahRoots& out, hipStream_t s);

}  // namespace rtg
