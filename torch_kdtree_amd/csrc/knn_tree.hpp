// KD-tree KNN traversal kernels for gfx950.
//
// One query per lane.  Each lane runs the reference's near-first depth-first search
// (src/kdtree.cpp:16-110) without a stack or a tag array: the state is the node index, its
// depth, the projected point pp (D registers) and far_mask, the levels of the current path that were
// entered through their far child: what the reference's per-node tags hold for the nodes on the
// active path (nodes off the path are never revisited).  Pruning takes every decision the reference
// takes that can change the result, and the candidate insertion repeats its arithmetic, so with
// the reference tie policy every lane produces what the reference CPU search produces.
//
// Queries arrive in an order given by `order` (a presort below: Morton buckets of the query
// positions by default, or buckets by near leaf), so the lanes of a wavefront walk similar paths
// and their record loads coalesce.
#pragma once

#include <type_traits>

#include "gpu_common.hpp"

namespace tk {

// Device view of a tree.  kBatched: the arrays belong to an arena of many trees and this lane's
// tree starts at the per-lane offsets below (set per query); otherwise the offsets are zero and
// fold away.  Leaf offsets hold arena-wide record positions in both cases.
template <typename T, bool kBatched = false>
struct TreeView {
    const T* __restrict__ split;            // [n_nodes] heap order
    const unsigned char* __restrict__ recs; // [n_points] records, structured order
    const int32_t* __restrict__ leaf_off;   // [n_leaves + 1]
    const int32_t* __restrict__ shuffled;   // [n_points] original index of a structured position
    const int32_t* __restrict__ inv_shuffled; // [n_points] structured position of an original index
    const unsigned char* __restrict__ boxes;  // [n_nodes + n_leaves] point boxes, heap order
    int levels;
    int32_t n_nodes;
    // batched only: where this tree's nodes, boxes, leaf offsets and records start in the arena
    int32_t node_base = 0, box_base = 0, leaf_base = 0, rec_base = 0;
    // point boxes of each leaf's record groups (kGroupRecs records from the leaf's first), and the
    // index of each leaf's first group box; null: no group tests
    const unsigned char* __restrict__ group_boxes = nullptr;
    const int32_t* __restrict__ group_base = nullptr;
    // Every split value separates its node's points (true when all coordinates and split values
    // are finite).  A NaN coordinate leaves std::sort's order unspecified and an overflowing median
    // is +-inf, so the lower-index policy then prunes with point boxes only (they hold the actual
    // extents of every subtree whatever the order).
    bool split_bounds = true;
    // Lower-index searches launch the 64-bit keyed list's kernel (kTieOK false) rather than the
    // KBestTie one: a cloud whose neighbours tie often, where nearly every lane would be searched
    // twice.  Read by the launcher.
    bool lower_direct = false;

    __device__ __forceinline__ T split_at(int32_t node) const { return split[kBatched ? node_base + node : node]; }
    __device__ __forceinline__ int32_t leaf_begin(int32_t leaf) const {
        return leaf_off[kBatched ? leaf_base + leaf : leaf];
    }
    __device__ __forceinline__ int32_t leaf_end(int32_t leaf) const {
        return leaf_off[kBatched ? leaf_base + leaf + 1 : leaf + 1];
    }
    __device__ __forceinline__ int32_t box_of(int32_t heap_node) const {
        return kBatched ? box_base + heap_node : heap_node;
    }
};

// base[i] for 0 <= i < 2^31, addressed with a 32-bit byte offset (keeps i a 32-bit value; a
// sign-extended 64-bit index would tie each k-list key to an aligned register pair).
__device__ __forceinline__ int32_t load_i32_at(const int32_t* __restrict__ base, int32_t i) {
    return *reinterpret_cast<const int32_t*>(reinterpret_cast<const char*>(base) + ((uint32_t)i << 2));
}

// Records per group box (the host writes them in runs of the same length), and the mean leaf
// size from which a tree gets group boxes.
constexpr int kGroupRecs = 16;
constexpr int kGroupMinLeaf = 4 * kGroupRecs;

// Threads per block of the traversal kernel; per-lane LDS staging slots are strided by it.
#ifndef TK_TREE_BLOCK
#define TK_TREE_BLOCK 128
#endif
#ifndef TK_STAGE_CHUNK_F32
#define TK_STAGE_CHUNK_F32 8
#endif
#ifndef TK_STAGE_CHUNK_F32_LOWER
#define TK_STAGE_CHUNK_F32_LOWER 4
#endif
#ifndef TK_STAGE_CHUNK_SMALLK
#define TK_STAGE_CHUNK_SMALLK 8
#endif
#ifndef TK_STAGE_CHUNK_F32_K16
#define TK_STAGE_CHUNK_F32_K16 16
#endif
#ifndef TK_SCAN_LOADS_F32
#define TK_SCAN_LOADS_F32 4
#endif
#ifndef TK_STAGE_CHUNK_F64
#define TK_STAGE_CHUNK_F64 16
#endif
#ifndef TK_SCAN_LOADS_F64
#define TK_SCAN_LOADS_F64 4
#endif
#ifndef TK_STAGE_CHUNK_WIDE
#define TK_STAGE_CHUNK_WIDE 4
#endif
// Occupancy target (waves per SIMD) of the register-list traversal kernels, for float searches
// with d <= 3 and lists of at most 16 (measured on MI355X, plain workload, k = 16):
//   reference policy, TK_F32_WAVES = 7: 72 VGPRs, no spills, 8.48 ms (5 waves: the same 72 VGPRs
//     scheduled differently, 8.77 ms; no target: 91 VGPRs, 9.14 ms; 8 waves: spills, 9.29 ms);
//   lower-index policy: lists of 8 and 16 (KBestTie, keyed like the reference policy's) take the
//     reference policy's shape (k = 16: 72 VGPRs, 8.29-8.63 ms); TK_F32_LOWER_WAVES = 7 for its
//     64-bit keyed lists (lists of at most 4; with that list at k = 16, chunks of 4 at 7 waves had
//     been best: 72 VGPRs and 16 bytes of spills, 9.75 ms; with chunks of 8, 92 VGPRs at 5 waves,
//     10.62 ms).
// Other kernels: see TK_F64_WAVES below, no target for the rest.
// TK_WAVES_PER_EU overrides every target (0 = no target anywhere).
#ifndef TK_WAVES_PER_EU
#define TK_WAVES_PER_EU -1
#endif
#ifndef TK_F32_WAVES
#define TK_F32_WAVES 7
#endif
#ifndef TK_F32_LOWER_WAVES
#define TK_F32_LOWER_WAVES 7
#endif
// Lower-index float searches with lists of 8, 16 or 32 keep the reference policy's list plus tie
// flags (KBestTie) instead of the 64-bit keyed list (0).
#ifndef TK_LOWER_TIE_LIST
#define TK_LOWER_TIE_LIST 1
#endif
// Double, d = 3, k = 16: no target (119 VGPRs, 4 waves; a 5-wave target spills 48 bytes, and a
// 4-wave one measured neutral).
#ifndef TK_F64_WAVES
#define TK_F64_WAVES 0
#endif
// kTie: the lower-index search keeps a KBestTie list (TreeList).
template <typename T, int D, int K, bool kLower, bool kTie = false>
struct TreeOccupancy {
    static constexpr int kWaves =
        TK_WAVES_PER_EU >= 0 ? TK_WAVES_PER_EU
        : (sizeof(T) == 4 && D <= 3 && K <= 16) ? (kLower && !kTie ? TK_F32_LOWER_WAVES : TK_F32_WAVES)
        : (sizeof(T) == 8 && D <= 3 && K == 16 && !kLower) ? TK_F64_WAVES
                                                           : 0;
};
#define TK_TREE_OCCUPANCY(T, D, K, L, TIE) __attribute__((amdgpu_waves_per_eu(TreeOccupancy<T, D, K, L, TIE>::kWaves > 0 ? TreeOccupancy<T, D, K, L, TIE>::kWaves : 1)))
// The same for the batched search kernels (more live state per lane: the cloud's offsets).
#ifndef TK_BATCH_WAVES_K16
#define TK_BATCH_WAVES_K16 4
#endif
#ifndef TK_BATCH_WAVES_K8
#define TK_BATCH_WAVES_K8 5
#endif
// k buckets 4 and 1 (67-75 VGPRs, 6 waves): 7- and 8-wave targets measured within noise.
#ifndef TK_BATCH_WAVES_K4
#define TK_BATCH_WAVES_K4 0
#endif
#ifndef TK_BATCH_WAVES_K1
#define TK_BATCH_WAVES_K1 0
#endif
template <typename T, int D, int K, bool kLower>
struct BatchOccupancy {
    static constexpr int kWaves =
        (sizeof(T) == 4 && D <= 3 && !kLower)
            ? (K == 16 ? TK_BATCH_WAVES_K16
                       : K == 8 ? TK_BATCH_WAVES_K8 : K == 4 ? TK_BATCH_WAVES_K4 : K == 1 ? TK_BATCH_WAVES_K1 : 0)
            : 0;
};
#define TK_BATCH_OCCUPANCY(T, D, K, L) __attribute__((amdgpu_waves_per_eu(BatchOccupancy<T, D, K, L>::kWaves > 0 ? BatchOccupancy<T, D, K, L>::kWaves : 1)))
constexpr int kTreeBlock = TK_TREE_BLOCK;
constexpr int kTreeBlockStride = kTreeBlock;

// The reference's own list, for trees with non-finite values under the reference tie policy.  Held
// in LDS: slot j of lane t lives at base[j * blockDim + t] (consecutive lanes hit consecutive banks).  A
// candidate is rejected only when d >= worst (src/nndistance.hpp:77) and
// is placed by the reference's binary search (upperBound, src/nndistance.hpp:41-60), so a NaN
// distance is taken and goes to the front, and the search's path through a list holding NaN
// entries decides where each later value lands; a NaN reaching the last slot makes worst NaN,
// after which every candidate is taken and every bound test fails, as in the reference.
template <typename T>
struct KBestExact {
    T* d;
    int32_t* s;
    int k;
    int stride;

    __device__ __forceinline__ void init() {
        for (int j = 0; j < k; ++j) {
            d[j * stride] = pos_inf<T>();
            s[j * stride] = 0;
        }
    }
    __device__ __forceinline__ T worst() const { return d[(k - 1) * stride]; }
    __device__ __forceinline__ bool accepts(T dist, int32_t) const { return !(dist >= worst()); }
    __device__ __forceinline__ void insert(T dist, int32_t sidx, int32_t) {
        int first = 0, count = k;
        while (count > 0) {
            const int step = count / 2;
            if (dist >= d[(first + step) * stride]) {
                first += step + 1;
                count -= step + 1;
            } else {
                count = step;
            }
        }
        if (first >= k) return;  // not reached after accepts(); kept as the reference keeps it
        for (int j = k - 1; j > first; --j) {
            d[j * stride] = d[(j - 1) * stride];
            s[j * stride] = s[(j - 1) * stride];
        }
        d[first * stride] = dist;
        s[first * stride] = sidx;
    }
};

// Lower-index policy on the reference policy's register list (one med3 per slot; the keys are
// structured indices, as under the reference policy, since the key order no longer decides
// anything: ties are settled by the flag below).  The two policies' lists can differ only through
// exact distance ties: when no point the search scans outside the list has a distance equal to the
// final worst W and the list's k distances are distinct, both hold the k points of smallest
// distance in ascending order.  `tie` records every event after which that may not hold:
// * a candidate equal to the current worst in the second pass (the first pass passes every
//   distance <= the stale worst, so a point at W is always a candidate, and the current worst it
//   then meets is >= W);
// * an insertion whose evicted entry equals the new worst (an evicted distance is >= W, and
//   equal to W only if equal to that worst, which never falls below W; empty slots aside);
// and unsure() adds equal distances among the k live entries (their order must follow the
// original index).  The search prunes with the lower-index policy's tests, so every point with
// distance <= W is scanned.  A lane that becomes unsure stops after that leaf pair and searches
// again, node by node, with the lower-index list (research_lower): rare on clouds without exact
// fp32 distance ties.  Trees whose clouds are full of them (lattices, rounded coordinates,
// duplicated points; Tree::tie_prone) launch the lower-index list's kernel instead.
template <typename T, int K>
struct KBestTie : KBest<T, K, false> {
    using Base = KBest<T, K, false>;
    bool tie;

    __device__ __forceinline__ void init(int k) {
        Base::init(k);
        tie = false;
    }
    static __device__ __forceinline__ bool accepts_stale(const typename Base::Stale& w, T dist, int32_t) {
        return dist <= w.d;
    }
    __device__ __forceinline__ bool admit(T dist, int32_t) {
        tie |= dist == Base::worst();
        return dist < Base::worst();
    }
    // (an entry at +inf is an empty slot: a +inf distance is never inserted, so evicting one is no tie)
    __device__ __forceinline__ void insert(T dist, int32_t key) {
        const T old = Base::worst();
        Base::insert(dist, key);
        tie |= dist < old && Base::worst() == old && old < pos_inf<T>();
    }
    __device__ __forceinline__ bool unsure(int k) const {
        bool t = tie;
#pragma unroll
        for (int j = 0; j + 1 < K; ++j) t |= j >= K - k && Base::d[j] == Base::d[j + 1];
        return t;
    }
    // unsure() during the search: equal entries are looked for only in a list without padding slots
    // (k == K, a wave-uniform test), where every adjacent pair is live
    __device__ __forceinline__ bool unsure_early(int k) const {
        bool t = tie;
        if (k == K) {
#pragma unroll
            for (int j = 0; j + 1 < K; ++j) t |= Base::d[j] == Base::d[j + 1];
        }
        return t;
    }
};

// The list of a single-tree register search.  Lower-index float searches with lists of 8, 16 or
// 32 take KBestTie (TK_LOWER_TIE_LIST 1): the 64-bit keyed list spends more issue slots per
// insertion than the med3 list plus the tie flags, and needs the original indices staged with the
// distances (plain workload, k = 16: 9.96-9.99 ms against 8.29-8.63; k = 32: 22.1-22.2 against
// 16.9-17.1).  Lists of at most 4 keep it: their insertions are short.
// kTieOK false: the 64-bit keyed list in any case (trees whose clouds tie often, Tree::tie_prone).
template <typename T, int K, bool kLower, bool kTieOK = true>
struct TreeList {
    using type = KBest<T, K, kLower>;
    static constexpr bool kTie = false;
};
template <int K, bool kTieOK>
struct TreeList<float, K, true, kTieOK> {
    static constexpr bool kTie = kTieOK && TK_LOWER_TIE_LIST && (K == 8 || K == 16 || K == 32);
    using type = typename std::conditional<kTie, KBestTie<float, K>, KBest<float, K, true>>::type;
};

// The original index of the record at structured position s: from the record where its layout
// has room for it, else from the tree's `shuffled` map (indexed, like the records, by position).
template <typename T, int D, bool kB>
__device__ __forceinline__ int32_t rec_orig(const TreeView<T, kB>& tv, int32_t s, const Rec<T, D>& r) {
    if constexpr (RecLayout<T, D>::kHasIdx)
        return r.o;
    else
        return load_i32_at(tv.shuffled, s);
}

template <typename T, int D, typename List, bool kB>
__device__ __forceinline__ void scan_leaf(const TreeView<T, kB>& tv, int32_t leaf, const Pt<T, D>& q, List& kb) {
    const int32_t beg = tv.leaf_begin(leaf);
    const int32_t end = tv.leaf_end(leaf);
    for (int32_t s = beg; s < end; ++s) {
        const Rec<T, D> r = load_rec<T, D>(tv.recs, s);
        const T dd = sq_dist<T, D>(q, r.c);
        const int32_t o = rec_orig(tv, s, r);
        if (kb.accepts(dd, o)) kb.insert(dd, s, o);
    }
}

// Bits l < 32 with l mod D == a.
template <int D>
__device__ __forceinline__ uint32_t axis_levels(int a) {
    uint32_t m = 0;
#pragma unroll
    for (int l = 0; l < 32; ++l)
        if (l % D == a) m |= 1u << l;
    return m;
}

// Pruning test of the lower-index policy: a side is skipped only when its bound exceeds worst.  A
// NaN bound (a NaN split value of a tree with non-finite coordinates) never prunes.
template <typename T>
__device__ __forceinline__ bool lower_passes(T bound, T worst) {
    return !(bound > worst);
}

// The lower-index policy's split-plane test: passes on trees whose splits do not bound their points.
template <typename T, int D, bool kB>
__device__ __forceinline__ bool lower_split_passes(const TreeView<T, kB>& tv, const Pt<T, D>& q, const Pt<T, D>& pp,
                                                   int a, T m, T worst) {
    return !tv.split_bounds || lower_passes(clean_bound<T, D>(q, pp, a, m), worst);
}

// The lower-index policy's far side test for the child `far_child` of split (a, m): the cell bound with one
// rounding per term and the box distance, both non-strict, so that a point at exactly the worst distance
// with a lower index is still found.
template <typename T, int D, bool kB>
__device__ __forceinline__ bool far_side_lower(const TreeView<T, kB>& tv, const Pt<T, D>& q, const Pt<T, D>& pp, int a,
                                               T m, int32_t far_child, T worst) {
    return lower_split_passes<T, D>(tv, q, pp, a, m, worst) &&
           lower_passes(aabb_bound<T, D>(tv.boxes, tv.box_of(far_child), q), worst);
}

// Whether a leaf can hold a point the list accepts (the reference scans it anyway; when the
// distance to its box is >= worst it would reject every point).
template <typename T, int D, bool kLower, bool kB>
__device__ __forceinline__ bool leaf_useful(const TreeView<T, kB>& tv, const Pt<T, D>& q, int32_t leaf, T worst) {
    const T b = aabb_bound<T, D>(tv.boxes, tv.box_of(tv.n_nodes + leaf), q);
    return kLower ? lower_passes(b, worst) : b < worst;
}

// Run-time axis access.  The element is taken from / put into a copy of the whole vector, so
// the lane state itself is only ever read and written whole and stays in registers (an
// element address computed from a run-time index would pin the surrounding object in memory).
template <typename T, int D>
__device__ __forceinline__ T ax_get(const Pt<T, D>& v, int a) {
    if constexpr (D == 1) {
        return v[0];
    } else {
        const Pt<T, D> c = v;
        return c[a];
    }
}

template <typename T, int D>
__device__ __forceinline__ void ax_set(Pt<T, D>& v, int a, T x) {
    if constexpr (D == 1) {
        v[0] = x;
    } else {
        Pt<T, D> c = v;
        c[a] = x;
        v = c;
    }
}

template <int D>
__device__ __forceinline__ int ax_next(int a) { return a + 1 == D ? 0 : a + 1; }
template <int D>
__device__ __forceinline__ int ax_prev(int a) { return a == 0 ? D - 1 : a - 1; }

// Records past the last point that a chunked leaf scan may read (and ignore): the record buffer is
// allocated with this many extra records, so the CH loads of a chunk need no per-point guard.
constexpr int kRecPad = 16;

// Leaf scan in two passes, for register lists.  Pass 1 computes the distances of CH consecutive
// records (loads issued back to back; those past the leaf are ignored), tests them against the
// worst distance at the start of the chunk and stages them in LDS; pass 2 pops each lane's
// accepted points in scan order and inserts those still accepted by the current list.  A
// wavefront then runs the insertion network once per accepted point of its busiest lane instead
// of once per point any lane accepts.  The outcome is that of a one-pass scan: the list after
// pass 2 holds exactly the points a one-pass scan would have inserted, because a point rejected
// by the stale worst is rejected by every later (smaller or equal) worst as well.
// In pass 2 a candidate that the current list rejects is inserted as +inf, which leaves the list
// unchanged: the insertion is then unconditional and updates the list in place.
template <typename T, int D, int K, bool kLower, int CH, int LD, int SB = kTreeBlockStride, bool kGroups = false,
          bool kB, typename List>
__device__ __forceinline__ void scan_leaf_staged(const TreeView<T, kB>& tv, int32_t leaf, const Pt<T, D>& q,
                                                 List& kb, T* __restrict__ st_d,
                                                 int32_t* __restrict__ st_o) {
    static_assert(CH % LD == 0 && CH <= 32, "a chunk is a whole number of load groups, at most 32 points");
    static_assert(!kGroups || kGroupRecs % CH == 0, "chunks nest in record groups");
    const int32_t beg = tv.leaf_begin(leaf);
    const int32_t end = tv.leaf_end(leaf);
    const int32_t gb = kGroups ? tv.group_base[leaf] : 0;
    for (int32_t c0 = beg; c0 < end; c0 += CH) {
        // With kGroups (the tree has group boxes): a group of records whose box lies at least the
        // worst distance away holds no point the list would take (every distance is at least the box
        // distance, in rounded arithmetic too), so skipping it changes nothing but the work.
        if (kGroups && (c0 - beg) % kGroupRecs == 0) {
            const T b = aabb_bound<T, D>(tv.group_boxes, gb + (c0 - beg) / kGroupRecs, q);
            if (kLower ? !lower_passes(b, kb.worst()) : !(b < kb.worst())) {
                c0 += kGroupRecs - CH;
                continue;
            }
        }
        const int n = min(CH, end - c0);
        const auto w = kb.stale();
        uint32_t mask = 0;
        // pass 1, LD records in flight at a time; every group is read (records past the leaf's
        // end are padding or the next leaf's, and are masked out), so the loads of a chunk are
        // issued without a data-dependent exit
#pragma unroll
        for (int g = 0; g < CH; g += LD) {
            Rec<T, D> rg[LD];
#pragma unroll
            for (int jj = 0; jj < LD; ++jj) rg[jj] = load_rec<T, D>(tv.recs, c0 + g + jj);
            // keeps the group's loads issued together ahead of their use
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int jj = 0; jj < LD; ++jj) {
                const int j = g + jj;
                const Rec<T, D>& r = rg[jj];
                const T dd = sq_dist<T, D>(q, r.c);
                const int32_t o = List::kOrigKeys ? rec_orig(tv, c0 + j, r) : 0;
                const bool acc = kb.accepts_stale(w, dd, o);
                mask |= acc ? (1u << j) : 0u;
                st_d[j * SB] = dd;
                if constexpr (List::kOrigKeys) st_o[j * SB] = o;
            }
        }
        mask &= n >= 32 ? ~0u : ((1u << n) - 1u);  // only the leaf's points
        // pass 2
        while (mask) {
            const int j = __builtin_ctz(mask);
            mask &= mask - 1u;
            const T dd = st_d[j * SB];
            const int32_t o = List::kOrigKeys ? st_o[j * SB] : 0;
            const bool ok = kb.admit(dd, o);
            kb.insert(ok ? dd : pos_inf<T>(), ok ? (List::kOrigKeys ? o : c0 + j) : 0x7fffffff);
        }
    }
}

template <int D>
__device__ __forceinline__ int axis_of_level(int l) { return l % D; }

// The search of one query; `kb` must be initialised.
//
// Besides pp (the reference's projected point) each lane carries far_mask, the levels at which the
// current path took a far child.  Leaves and far sides are tested against the distance from q to the
// bounding box of their points.
//
// Why the climb tests boxes alone, where the reference tests its split bound.  A level that the climb
// leaves resets pp[axis] = q[axis], whether it was entered through its far child, its far side was
// skipped or it is the leaf-parent.  So when level j is tested, pp is q on the axes of the path's levels
// below j and, elsewhere, q or the split plane of a far level above j on the path, beyond which all
// points below j lie.  The far child's points also lie beyond m_j on its axis.  On every axis the gap
// from q to the far child's box is therefore at least |pp - q| (|m_j - q| on axis j), and since both
// sums round one difference per axis and add the squares in axis order, the box distance is never below
// the bound, rounded values included.  A box distance below worst thus implies a bound below worst: the
// box decides.  A far side that the reference enters although its box distance is >= worst changes
// nothing: all its points would be rejected, and the resets that its walk leaves (the axes of the next
// levels below j) are among those the climb made.  Only at the leaf-parent does the reference's bound
// round twice ((pp - q) + (m - pp), pp not yet set to m), which can exceed the box distance by an ulp;
// there the reference's own test is kept.  The same holds for the lower-index policy's split bound,
// which rounds once at every level; that policy needs no pp at all.
// (Against the form that tested the split bound first wherever pp differed from q: plain workload,
// 16M queries, k = 16, 7.62 ms a query step against 7.82; k = 8, 5.93 against 6.12; lower-index policy,
// 8M queries, 4.50 against 4.71; d = 8, k = 32, 100K queries of 500K points, 24.1 against 29.1.)
//
// Climbing: a level whose far child is on the path, or whose far side was ruled out for good after the first
// leaf pair (bit set in far_mask), is simply left; the climb jumps from one other level to the next with bit
// scans.
// Lane state of one search: q, pp, the k-list, far_mask, node, level.  They are kept as
// separate variables of the kernel (not one aggregate), so that each can live in registers.

// Walks the near path from `node` down to the leaf-parent level.
template <typename T, int D, bool kB>
__device__ __forceinline__ void lane_descend(const TreeView<T, kB>& tv, const Pt<T, D>& q, int32_t& node, int& level) {
    int a = axis_of_level<D>(level);
    while (level < tv.levels - 1) {
        node = 2 * node + (ax_get(q, a) < tv.split_at(node) ? 1 : 2);
        ++level;
        a = ax_next<D>(a);
    }
}

// A query with a NaN coordinate forms only NaN distances and bounds.  The reference's insertion
// (src/nndistance.hpp:77-85) rejects a candidate only when d >= worst and places it at the upper
// bound found with `value >= *it`, so a NaN distance is always taken and goes to the front; every
// bound test against worst fails, so its search (src/kdtree.cpp:16-110) scans exactly the leaf
// its descent reaches (a NaN coordinate never compares below a split) and prunes the rest.  Under
// the reference policy the list is that leaf's last k records in reverse order, with their
// distances, then the untouched (+inf, 0) entries when the leaf holds fewer than k points.  The
// lower-index policy gives what the brute force gives (src/nndistance_g.cu:57 inserts only when
// d < worst, which a NaN never is): the empty list, (+inf, original index 0) in every slot.
template <typename T, int D>
__device__ __forceinline__ bool has_nan(const Pt<T, D>& q) {
    bool r = false;
#pragma unroll
    for (int i = 0; i < D; ++i) r |= __builtin_isnan(q[i]);
    return r;
}

// Record range of the leaf the descent of q reaches.
template <typename T, int D, bool kB>
__device__ __forceinline__ void descent_leaf(const TreeView<T, kB>& tv, const Pt<T, D>& q, int32_t& beg,
                                             int32_t& end) {
    int32_t node = 0;
    int a = 0;
    for (int level = 0; level < tv.levels; ++level) {
        node = 2 * node + (ax_get(q, a) < tv.split_at(node) ? 1 : 2);
        a = ax_next<D>(a);
    }
    const int32_t leaf = node - tv.n_nodes;
    beg = tv.leaf_begin(leaf);
    end = tv.leaf_end(leaf);
}

// The list of a NaN query under the reference policy, from an initialised list: slot c (0 =
// nearest) holds record end-1-c of the descent's leaf while that is in the leaf.  Under the
// lower-index policy the initialised list (+inf, original index 0) is already the result; a list
// keyed by structured index then takes the position of original index 0 as its key.
template <typename T, int D, int K, bool kLower, bool kB, typename List>
__device__ __forceinline__ void nan_fill(const TreeView<T, kB>& tv, const Pt<T, D>& q, int k, List& kb) {
    if constexpr (!kLower) {
        int32_t beg = 0, end = 0;
        descent_leaf<T, D, kB>(tv, q, beg, end);
        const int pad = K - k;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const int32_t rec = end - 1 - (j - pad);
            if (j >= pad && rec >= beg) kb.set(j, sq_dist<T, D>(q, load_rec<T, D>(tv.recs, rec).c), rec);
        }
    } else if constexpr (!List::kOrigKeys) {
        const int32_t s0 = load_i32_at(tv.inv_shuffled, 0);
#pragma unroll
        for (int j = 0; j < K; ++j) kb.set(j, kb.dist(j), s0);
    }
}

// Starts the search of the query in q.
template <typename T, int D, int K, bool kLower, bool kB, typename List>
__device__ __forceinline__ void lane_start(const TreeView<T, kB>& tv, int k, const Pt<T, D>& q, Pt<T, D>& pp,
                                           List& kb, uint32_t& far_mask, int32_t& node,
                                           int& level) {
    pp = q;
    kb.init(k);
    far_mask = 0;
    node = 0;
    level = 0;
    lane_descend<T, D>(tv, q, node, level);
}

// Scans the leaf pair of the current leaf-parent, then climbs to the next far side to enter and
// walks down to its leaf-parent.  Returns true when the search is complete.
template <typename T, int D, int K, bool kLower, int CH, int LD, int SB = kTreeBlockStride, bool kGroups = false,
          bool kB, typename List>
__device__ __forceinline__ bool lane_step(const TreeView<T, kB>& tv, const Pt<T, D>& q, Pt<T, D>& pp,
                                          List& kb, uint32_t& far_mask, int32_t& node, int& level,
                                          T* __restrict__ st_d, int32_t* __restrict__ st_o) {
    const int L = tv.levels;
    const int a_lp = axis_of_level<D>(L - 1);  // split axis of every leaf-parent
    {
        const T m = tv.split_at(node);
        const T qa = ax_get(q, a_lp);
        const bool lower = qa < m;
        const int32_t left_leaf = 2 * node + 1 - tv.n_nodes;
        const int32_t near_leaf = lower ? left_leaf : left_leaf + 1;
        const int32_t far_leaf = lower ? left_leaf + 1 : left_leaf;
        // near leaf, then the far leaf if the reference looks at it (one scan site for both)
#pragma nounroll
        for (int side = 0; side < 2; ++side) {
            const int32_t leaf = side ? far_leaf : near_leaf;
            // (under the lower-index policy the far leaf's box distance, tested next, is never below
            // its split bound)
            const bool looks = kLower || side == 0 || proj_bound<T, D>(q, pp, a_lp, m) < kb.worst();
            if (looks && leaf_useful<T, D, kLower>(tv, q, leaf, kb.worst()))
                scan_leaf_staged<T, D, K, kLower, CH, LD, SB, kGroups>(tv, leaf, q, kb, st_d, st_o);
        }
    }
    // After the first leaf pair: levels whose split plane lies no nearer than the worst entry are marked
    // in far_mask with those entered through their far child, so that no climb tests them.  On the plane's axis
    // the far child's box is no nearer than the plane, and the sum of squares no smaller than that axis'
    // square, rounded values included; worst only falls.  (The planes of a lane's path are a few loads that
    // its neighbours share; a climb to the root would test the box of every level.  Box tests per wavefront,
    // plain workload, 120 -> 65: 7.72 -> 7.25 ms; the batched replay 6.04 -> 5.88.)
    if (far_mask == 0 && tv.split_bounds) {
        const T w = kb.worst();
        for (int l0 = 0; l0 < level; l0 += D) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                const int l = l0 + a < level ? l0 + a : level;
                const T g = q[a] - tv.split_at(((node + 1) >> (level - l)) - 1);
                const bool beyond = kLower ? !lower_passes(g * g, w) : !(g * g < w);
                far_mask |= beyond && l < level ? 1u << l : 0u;
            }
        }
    }
    // Climb: the levels entered through their near child, deepest first; the first whose far child's
    // box passes is entered.  The box of the next candidate level is loaded while the current one
    // is tested.  The far child of such a level is the sibling of the path's child one level down.
    uint32_t near_lv = ((1u << level) - 1u) & ~far_mask;
    if (!near_lv) return true;
    int j = 31 - __builtin_clz(near_lv);
    int32_t c = ((node + 1) >> (level - 1 - j)) - 1;
    BoxVals<T, D> bx = load_box<T, D>(tv.boxes, tv.box_of(((c - 1) ^ 1) + 1));
    for (;;) {
        const uint32_t rest = near_lv ^ (1u << j);
        const int j2 = rest ? 31 - __builtin_clz(rest) : j;
        const int32_t c2 = ((node + 1) >> (level - 1 - j2)) - 1;
        const BoxVals<T, D> bx2 = load_box<T, D>(tv.boxes, tv.box_of(((c2 - 1) ^ 1) + 1));
        const T b = box_dist<T, D>(bx, q);
        if (kLower ? lower_passes(b, kb.worst()) : b < kb.worst()) {
            if constexpr (!kLower) {
                // the levels left on the way up reset pp on their axes; level j's far side sets its own
                const uint32_t left = ((1u << L) - 1u) & ~((2u << j) - 1u);
#pragma unroll
                for (int ax = 0; ax < D; ++ax) pp[ax] = (left & axis_levels<D>(ax)) ? q[ax] : pp[ax];
                ax_set(pp, axis_of_level<D>(j), tv.split_at((c - 1) >> 1));
            }
            far_mask = (far_mask & ((1u << j) - 1u)) | (1u << j);
            node = ((c - 1) ^ 1) + 1;
            level = j + 1;
            lane_descend<T, D>(tv, q, node, level);
            return false;
        }
        if (!rest) return true;
        near_lv = rest;
        j = j2;
        c = c2;
        bx = bx2;
    }
}

// The search with a generic list, one node at a time.  Reference policy: the reference's own walk
// (src/kdtree.cpp:16-110), step for step and without point boxes (trees with non-finite values, or splits that
// do not bound their points).  Lower-index policy: the same walk with that policy's tests (research_lower).
template <typename T, int D, bool kLower, typename List, bool kB>
__device__ __forceinline__ void knn_search_one(const TreeView<T, kB>& tv, const Pt<T, D>& q, List& kb) {
    Pt<T, D> pp = q;
    const int L = tv.levels;
    const int32_t nn = tv.n_nodes;
    int32_t node = 0;
    int level = 0;
    int a = 0;  // split axis of `node`: level mod D
    for (;;) {
        while (level < L - 1) {
            node = 2 * node + (ax_get(q, a) < tv.split_at(node) ? 1 : 2);
            ++level;
            a = ax_next<D>(a);
        }
        {
            const T m = tv.split_at(node);
            const T qa = ax_get(q, a);
            const bool lower = qa < m;
            const int32_t near_leaf = 2 * node + (lower ? 1 : 2) - nn;
            const int32_t far_leaf = 2 * node + (lower ? 2 : 1) - nn;
            if (!kLower || leaf_useful<T, D, kLower>(tv, q, near_leaf, kb.worst()))
                scan_leaf<T, D>(tv, near_leaf, q, kb);
            if (kLower ? lower_split_passes<T, D>(tv, q, pp, a, m, kb.worst()) &&
                             leaf_useful<T, D, kLower>(tv, q, far_leaf, kb.worst())
                       : proj_bound<T, D>(q, pp, a, m) < kb.worst())
                scan_leaf<T, D>(tv, far_leaf, q, kb);
            if (level == 0) return;
            ax_set(pp, a, qa);
        }
        bool entered = false;
        while (level > 0) {
            const int32_t child = node;
            node = (node - 1) >> 1;
            --level;
            a = ax_prev<D>(a);
            const T m2 = tv.split_at(node);
            const T q2 = ax_get(q, a);
            const bool lower2 = q2 < m2;
            if (child == 2 * node + (lower2 ? 1 : 2)) {
                const int32_t far_child = 2 * node + (lower2 ? 2 : 1);
                ax_set(pp, a, m2);
                if (kLower ? far_side_lower<T, D>(tv, q, pp, a, m2, far_child, kb.worst())
                           : proj_bound<T, D>(q, pp, a, m2) < kb.worst()) {
                    node = far_child;
                    ++level;
                    a = ax_next<D>(a);
                    entered = true;
                    break;
                }
            }
            ax_set(pp, a, q2);
        }
        if (!entered) return;
    }
}

// Stores val(j) for the slots j in [J0, J0 + N) that are live (j >= pad) to p[j - pad]; with vec
// (k == K and p 16-byte aligned) in 16-byte stores.
template <typename V, int J0, int N, typename F>
__device__ __forceinline__ void store_slots(V* __restrict__ p, bool vec, int pad, F&& val) {
    constexpr int kPer = 16 / (int)sizeof(V);
    if constexpr (N % kPer == 0) {
        if (vec) {
#pragma unroll
            for (int j = J0; j < J0 + N; j += kPer) {
                V tmp[kPer];
#pragma unroll
                for (int u = 0; u < kPer; ++u) tmp[u] = val(j + u);
                uint4 w;
                __builtin_memcpy(&w, tmp, 16);
                *reinterpret_cast<uint4*>(p + j) = w;
            }
            return;
        }
    }
#pragma unroll
    for (int j = J0; j < J0 + N; ++j)
        if (j >= pad) p[j - pad] = val(j);
}

// Writes one query's list to row qi of the outputs: distances, structured indices and (with
// out_o) original indices.  A list keyed by structured index (kOrig false) gathers the original
// ones through `shuffled`; one keyed by original index (the lower-index policy's 64-bit keyed
// list) gathers the structured ones through `inv_shuffled`.  The gathers of up to 16 slots are
// issued before their stores, so their latencies overlap instead of following one another (a
// 32-entry list goes out in two halves, which keeps the live registers below those of its
// search); when k == K and the three arrays are 16-byte aligned, the rows go out in 16-byte
// stores.
template <typename T, int K, bool kOrig, int J0 = 0, typename List>
__device__ __forceinline__ void store_list(const List& kb, int k, const TreeView<T>& tv, int64_t qi,
                                           T* __restrict__ out_d, int32_t* __restrict__ out_i,
                                           int64_t* __restrict__ out_o) {
    constexpr int N = K - J0 < 16 ? K - J0 : 16;
    const int pad = K - k;
    const bool vec = pad == 0 && ((((uintptr_t)out_d | (uintptr_t)out_i | (uintptr_t)out_o) & 15u) == 0);
    int32_t m[N] = {};
    if (kOrig || out_o) {
        const int32_t* map = kOrig ? tv.inv_shuffled : tv.shuffled;
#pragma unroll
        for (int u = 0; u < N; ++u) m[u] = load_i32_at(map, J0 + u >= pad ? kb.key(J0 + u) : 0);
    }
    T* od = out_d + qi * k;
    int32_t* oi = out_i + qi * k;
    store_slots<T, J0, N>(od, vec, pad, [&](int j) { return kb.dist(j); });
    store_slots<int32_t, J0, N>(oi, vec, pad, [&](int j) { return kOrig ? m[j - J0] : kb.key(j); });
    if (out_o)
        store_slots<int64_t, J0, N>(out_o + qi * k, vec, pad,
                                    [&](int j) { return (int64_t)(kOrig ? kb.key(j) : m[j - J0]); });
    if constexpr (J0 + N < K) store_list<T, K, kOrig, J0 + N>(kb, k, tv, qi, out_d, out_i, out_o);
}

// ---------------------------------------------------------------------------------------------
// Row stores through LDS for a full wavefront.  Lane l holds output row qi(l); stored lane by lane,
// every 16-byte store instruction touches 64 different rows (64 partial lines).  Passing a slab of
// SW bytes of each row through the wave's part of the leaf-scan staging buffer lets one
// instruction write 64 consecutive 16-byte chunks of the slab matrix instead: SW/16 lanes per row
// and 1024/SW whole row slabs per instruction.
// ---------------------------------------------------------------------------------------------

// The wave's part of a block's staging buffer T[CH * BLK] (lane i of the block owns elements i,
// i + BLK, i + 2*BLK, ...): CH segments of 64 elements, BLK elements apart.  Chunk c (16 bytes) of
// the wave's logical buffer lies in one segment, since a segment is a multiple of 16 bytes.
template <typename T, int BLK>
struct WaveStage {
    unsigned char* base;  // the wave's part of segment 0

    __device__ __forceinline__ uint4* chunk(int c) const {
        constexpr int kSeg = 64 * (int)sizeof(T);
        const int byte = c * 16;
        return reinterpret_cast<uint4*>(base + (byte / kSeg) * (BLK * (int)sizeof(T)) + byte % kSeg);
    }
};

// Orders the wave's LDS writes before its reads and the reads before the next writes.  A
// wavefront's LDS instructions execute in issue order, so only the compiler must keep them there.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Writes bytes [col, col + 16*NC) of every lane's row: v holds this lane's, row_bytes is the row
// stride of `base`, qr[p] the row of the lanes whose chunk pass p stores (row p*64/C + lane/C of
// the wave, C = SW/16 chunks per lane and slab).
template <typename T, int BLK, int SW, int NC>
__device__ __forceinline__ void wave_store_part(const WaveStage<T, BLK>& st, int lane, const int32_t (&qr)[SW / 16],
                                                unsigned char* __restrict__ base, int64_t row_bytes, int col,
                                                const uint4 (&v)[NC]) {
    constexpr int C = SW / 16;
    static_assert(NC % C == 0, "a row part is a whole number of slabs");
#pragma unroll
    for (int s = 0; s < NC / C; ++s) {
#pragma unroll
        for (int u = 0; u < C; ++u) *st.chunk(lane * C + u) = v[s * C + u];
        wave_lds_sync();
#pragma unroll
        for (int p = 0; p < C; ++p) {
            const uint4 w = *st.chunk(p * 64 + lane);
            *reinterpret_cast<uint4*>(base + qr[p] * row_bytes + col + s * SW + (lane % C) * 16) = w;
        }
        wave_lds_sync();
    }
}

// Slab width of the wave stores: at most 64 bytes, what the wave's staging part holds per lane
// (CH elements), and a divisor of every row part (up to 16 entries of 4, 8 or sizeof(T) bytes).
template <typename T, int K, int CH>
constexpr int wave_slab_bytes() {
    const int a = CH * (int)sizeof(T) < 64 ? CH * (int)sizeof(T) : 64;
    const int n4 = (K < 16 ? K : 16) * 4;
    return a < n4 ? a : n4;
}

// store_list for a full wavefront whose rows are k == K entries long and 16-byte aligned: the same
// values, through wave_store_part.  The distances go out before the index gathers are issued, so
// the two are not live at once.
template <typename T, int K, bool kOrig, int BLK, int SW, int J0 = 0, typename List>
__device__ __forceinline__ void store_list_wave(const List& kb, const TreeView<T>& tv,
                                                const WaveStage<T, BLK>& st, int lane,
                                                const int32_t (&qr)[SW / 16], T* __restrict__ out_d,
                                                int32_t* __restrict__ out_i, int64_t* __restrict__ out_o) {
    constexpr int N = K - J0 < 16 ? K - J0 : 16;
    {
        T tmp[N];
#pragma unroll
        for (int u = 0; u < N; ++u) tmp[u] = kb.dist(J0 + u);
        uint4 v[N * sizeof(T) / 16];
        __builtin_memcpy(v, tmp, sizeof(tmp));
        wave_store_part<T, BLK, SW>(st, lane, qr, reinterpret_cast<unsigned char*>(out_d), (int64_t)K * sizeof(T),
                                    J0 * (int)sizeof(T), v);
    }
    int32_t m[N] = {};
    if (kOrig || out_o) {
        const int32_t* map = kOrig ? tv.inv_shuffled : tv.shuffled;
#pragma unroll
        for (int u = 0; u < N; ++u) m[u] = load_i32_at(map, kb.key(J0 + u));
    }
    {
        int32_t tmp[N];
#pragma unroll
        for (int u = 0; u < N; ++u) tmp[u] = kOrig ? m[u] : kb.key(J0 + u);
        uint4 v[N * 4 / 16];
        __builtin_memcpy(v, tmp, sizeof(tmp));
        wave_store_part<T, BLK, SW>(st, lane, qr, reinterpret_cast<unsigned char*>(out_i), (int64_t)K * 4, J0 * 4, v);
    }
    if (out_o) {
        int64_t tmp[N];
#pragma unroll
        for (int u = 0; u < N; ++u) tmp[u] = (int64_t)(kOrig ? kb.key(J0 + u) : m[u]);
        uint4 v[N * 8 / 16];
        __builtin_memcpy(v, tmp, sizeof(tmp));
        wave_store_part<T, BLK, SW>(st, lane, qr, reinterpret_cast<unsigned char*>(out_o), (int64_t)K * 8, J0 * 8, v);
    }
    if constexpr (J0 + N < K)
        store_list_wave<T, K, kOrig, BLK, SW, J0 + N>(kb, tv, st, lane, qr, out_d, out_i, out_o);
}

template <typename T, int D>
__device__ __forceinline__ void load_query(const T* __restrict__ queries, int64_t qi, Pt<T, D>& q) {
#pragma unroll
    for (int i = 0; i < D; ++i) q[i] = queries[qi * D + i];
}

// Output rows of full wavefronts written through LDS (1) or lane by lane (0).
#ifndef TK_WAVE_STORES
#define TK_WAVE_STORES 1
#endif

// Points per staged chunk of the leaf scan (measured on MI355X), for float searches with d <= 3
// and lists of 8 or more: TK_STAGE_CHUNK_F32_K16 (16) for the single-tree reference-policy
// search with a 16-entry list (plain workload 8.32 ms against 8.44 at 8), TK_STAGE_CHUNK_F32 (8)
// for the other reference-policy ones (k = 8: 6.14 ms against 6.20 at 16; batched replay 21.76 ms
// against 21.93); the lower-index policy's KBestTie lists take the same, its 64-bit keyed lists
// TK_STAGE_CHUNK_F32_LOWER (4; 10.14 ms against 10.56 at 8).  For lists of at most 4 at d <= 3,
// TK_STAGE_CHUNK_SMALLK (8; single-tree k = 4: 4.78 ms against 4.91 at 4, k = 1: 3.75 against 3.80; batched
// 64-cloud replay, K = 4 1.16 ms against 1.24, K = 1 0.89 against 0.91).  TK_STAGE_CHUNK_WIDE (4) for d = 8, where a
// larger chunk's extra stale-worst pops cost more than its fewer exits; TK_STAGE_CHUNK_F64 for double.
// kB: the batched search.
template <typename T, int D, int K, bool kLower, bool kB = false, bool kTieOK = true>
struct StageBytes {
    static constexpr bool kTieList = !kB && TreeList<T, K, kLower, kTieOK>::kTie;
    static constexpr int kChunk =
        sizeof(T) == 4
            ? ((D <= 3 && K >= 8) ? (kLower && !kTieList ? TK_STAGE_CHUNK_F32_LOWER
                                                         : (K == 16 && !kB ? TK_STAGE_CHUNK_F32_K16 : TK_STAGE_CHUNK_F32))
                                  : (D <= 3 ? TK_STAGE_CHUNK_SMALLK : TK_STAGE_CHUNK_WIDE))
            : TK_STAGE_CHUNK_F64;
    static constexpr int kLoads = sizeof(T) == 4 ? (TK_SCAN_LOADS_F32 < kChunk ? TK_SCAN_LOADS_F32 : kChunk)
                                                 : (TK_SCAN_LOADS_F64 < kChunk ? TK_SCAN_LOADS_F64 : kChunk);
    static constexpr int kBytes = kChunk * kTreeBlock * ((int)sizeof(T) + (kLower ? 4 : 0));
};

// The list interface of scan_leaf / knn_search_one over a register list.
template <typename T, typename L>
struct RegListRef {
    L& l;
    __device__ __forceinline__ T worst() const { return l.worst(); }
    __device__ __forceinline__ bool accepts(T dist, int32_t orig) const { return l.accepts(dist, orig); }
    __device__ __forceinline__ void insert(T dist, int32_t, int32_t orig) { l.insert(dist, orig); }
};

// The lower-index search of q again, node by node with the 64-bit keyed list (little code beside
// the staged search, for the rare unsure lane), into kb, with the original indices turned into
// structured ones.
template <typename T, int D, int K, bool kB>
__device__ __forceinline__ void research_lower(const TreeView<T, kB>& tv, const Pt<T, D>& q, int k,
                                               KBestTie<T, K>& kb) {
    KBest<T, K, true> ex;
    ex.init(k);
    RegListRef<T, KBest<T, K, true>> ref{ex};
    knn_search_one<T, D, true>(tv, q, ref);
#pragma unroll
    for (int j = 0; j < K; ++j) kb.set(j, ex.dist(j), load_i32_at(tv.inv_shuffled, ex.key(j)));
}

// One lane per query.  The lanes of a wavefront take 64 consecutive presorted queries and run
// their searches to completion together: neighbouring queries walk the tree nearly in step, which
// keeps the wavefront's control flow and loads coherent.  (Handing a finished lane the next query
// was measured to be slower: it breaks that lockstep.)  BLK threads per block, leaf chunks of CH
// records with LD loads in flight.
template <typename T, int D, int K, bool kLower, int CH, int LD, int BLK, bool kGroups = false, bool kTieOK = true>
__device__ __forceinline__ void tree_search_lanes(const TreeView<T>& tv, const T* __restrict__ queries, int64_t nq,
                                                  const int32_t* __restrict__ order, int k, T* __restrict__ out_d,
                                                  int32_t* __restrict__ out_i, int64_t* __restrict__ out_o) {
    static_assert(CH <= kRecPad, "a chunk may read at most kRecPad records past a leaf's end");
    static_assert(BLK % 64 == 0, "whole wavefronts per block");
    using List = typename TreeList<T, K, kLower, kTieOK>::type;
    constexpr bool kO = List::kOrigKeys;  // list keys are original indices (staged with the distances)
    constexpr bool kTie = TreeList<T, K, kLower, kTieOK>::kTie;
    __shared__ __align__(16) T stage_d[CH * BLK];
    __shared__ int32_t stage_o[kO ? CH * BLK : 1];
    // t = wave0 + lane with wave0 in scalars; the lane index and the row are found again after the
    // search, so that no per-lane index has to stay live through it
    const int wave_off = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & ~63u));
    const int64_t wave0 = xcd_tile(blockIdx.x, gridDim.x) * BLK + wave_off;
    if (wave0 + (int)(threadIdx.x & 63u) >= nq) return;
    Pt<T, D> q, pp;
    List kb;
    uint32_t far_mask;
    int32_t node;
    int level;
    {
        const int64_t t = wave0 + (int)(threadIdx.x & 63u);
        load_query<T, D>(queries, order ? (int64_t)order[t] : t, q);
    }
    lane_start<T, D, K, kLower>(tv, k, q, pp, kb, far_mask, node, level);
    if (has_nan<T, D>(q)) {
        nan_fill<T, D, K, kLower>(tv, q, k, kb);
    } else {
        // (a KBestTie lane stops after the leaf pair where it becomes unsure: it is searched again
        // in any case)
        while (!lane_step<T, D, K, kLower, CH, LD, BLK, kGroups>(tv, q, pp, kb, far_mask, node, level,
                                                              stage_d + threadIdx.x, stage_o + (kO ? threadIdx.x : 0))) {
            if constexpr (kTie)
                if (kb.unsure_early(k)) break;
        }
        if constexpr (kTie)
            if (kb.unsure(k)) research_lower<T, D, K>(tv, q, k, kb);
    }
    // (the lane index from mbcnt in a volatile asm, and the row by an atomic load, so that the
    // compiler recomputes both here rather than carrying the first values through the search)
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    const int32_t qi = order ? __hip_atomic_load(order + wave0 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT)
                             : (int32_t)(wave0 + lane);  // nq < 2^31
    constexpr int SW = wave_slab_bytes<T, K, CH>();
    // (float only: the double kernels already run at 2 to 5 waves per SIMD, where the stores' extra
    // registers cost a wave for some lists)
    if constexpr (TK_WAVE_STORES && sizeof(T) == 4 && K >= 8 && SW >= 32) {
        // When the wave's 64 queries all exist, every lane of the wave is here (the search loop has
        // ended for all of them) and the wave's rows go out through its part of stage_d.  The wave's
        // first position comes from scalars, so that t need not stay live through the search.
        const bool full = wave0 + 64 <= nq;
        const bool vec = k == K && ((((uintptr_t)out_d | (uintptr_t)out_i | (uintptr_t)out_o) & 15u) == 0);
        if (full && vec) {
            constexpr int C = SW / 16;
            int32_t qr[C];
#pragma unroll
            for (int p = 0; p < C; ++p) qr[p] = __shfl(qi, p * (64 / C) + lane / C, 64);
            const WaveStage<T, BLK> st{reinterpret_cast<unsigned char*>(stage_d + wave_off)};
            store_list_wave<T, K, kO, BLK, SW>(kb, tv, st, lane, qr, out_d, out_i, out_o);
            return;
        }
    }
    store_list<T, K, kO>(kb, k, tv, qi, out_d, out_i, out_o);
}

// kGroups: the tree has record-group boxes (tv.group_boxes), and leaf scans test them.  kTieOK
// false: a lower-index search keeps the 64-bit keyed list (a tree whose cloud ties often).
template <typename T, int D, int K, bool kLower, bool kGroups = false, bool kTieOK = true>
__global__ __launch_bounds__(kTreeBlock) TK_TREE_OCCUPANCY(T, D, K, kLower, (TreeList<T, K, kLower, kTieOK>::kTie))
void knn_tree_kernel(TreeView<T> tv, const T* __restrict__ queries, int64_t nq, const int32_t* __restrict__ order,
                     int k, T* __restrict__ out_d, int32_t* __restrict__ out_i, int64_t* __restrict__ out_o) {
    tree_search_lanes<T, D, K, kLower, StageBytes<T, D, K, kLower, false, kTieOK>::kChunk,
                      StageBytes<T, D, K, kLower, false, kTieOK>::kLoads, kTreeBlock, kGroups, kTieOK>(
        tv, queries, nq, order, k, out_d, out_i, out_o);
}

// The same search with its launch shape as template parameters: the prebuilt variants an autotuner
// picks among (leaf chunk CH with LD loads in flight, BLK threads per block, an occupancy target of
// WAVES waves per SIMD, 0 = none).  Results do not depend on them.
template <typename T, int D, int K, bool kLower, int CH, int LD, int BLK, int WAVES>
__global__ __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(WAVES > 0 ? WAVES : 1))) void knn_tree_kernel_v(
    TreeView<T> tv, const T* __restrict__ queries, int64_t nq, const int32_t* __restrict__ order, int k,
    T* __restrict__ out_d, int32_t* __restrict__ out_i, int64_t* __restrict__ out_o) {
    tree_search_lanes<T, D, K, kLower, CH, LD, BLK>(tv, queries, nq, order, k, out_d, out_i, out_o);
}

constexpr int kLdsBlock = 64;

// Reference tie policy on a tree with a non-finite coordinate or split value: the reference's walk
// step for step (no point boxes) with the reference's list (KBestExact), one lane per query.
// Queries with a NaN coordinate need no special case here.
template <typename T, int D>
__global__ __launch_bounds__(kLdsBlock) void knn_tree_exact_kernel(TreeView<T> tv, const T* __restrict__ queries,
                                                                    int64_t nq, const int32_t* __restrict__ order,
                                                                    int k, T* __restrict__ out_d,
                                                                    int32_t* __restrict__ out_i,
                                                                    int64_t* __restrict__ out_o) {
    extern __shared__ unsigned char smem[];
    const int64_t t = xcd_tile(blockIdx.x, gridDim.x) * kLdsBlock + threadIdx.x;
    if (t >= nq) return;
    const int64_t qi = order ? (int64_t)order[t] : t;
    T* sd = reinterpret_cast<T*>(smem);
    int32_t* ss = reinterpret_cast<int32_t*>(sd + (size_t)k * kLdsBlock);
    KBestExact<T> kb{sd + threadIdx.x, ss + threadIdx.x, k, kLdsBlock};
    kb.init();
    Pt<T, D> q;
    load_query<T, D>(queries, qi, q);
    knn_search_one<T, D, false>(tv, q, kb);
    for (int j = 0; j < k; ++j) {
        const int32_t sj = kb.s[j * kLdsBlock];
        out_d[qi * k + j] = kb.d[j * kLdsBlock];
        out_i[qi * k + j] = sj;
        if (out_o) out_o[qi * k + j] = tv.shuffled[sj];
    }
}

inline size_t exact_list_bytes(int k, size_t tsize) { return (size_t)k * kLdsBlock * (tsize + 4); }

// ---------------------------------------------------------------------------------------------
// Query presorts.  Each presort kernel writes one integer key per query; a stable radix sort of
// (key, row) (radix_sort.hip) then gives the order, so the order is
// deterministic: equal keys keep increasing rows.
//
// Leaf keys: each query descends to the leaf on its near side (no pruning); leaves are numbered
// left to right, so neighbouring keys are neighbouring cells of space.
// ---------------------------------------------------------------------------------------------
constexpr int kPresortBlock = 256;

template <typename T, int D>
__global__ __launch_bounds__(kPresortBlock) void leaf_bucket_kernel(TreeView<T> tv, const T* __restrict__ queries,
                                                                     int64_t nq, int shift,
                                                                     uint32_t* __restrict__ key) {
    const int64_t i = (int64_t)blockIdx.x * kPresortBlock + threadIdx.x;
    if (i >= nq) return;
    Pt<T, D> q;
    load_query<T, D>(queries, i, q);
    int32_t node = 0;
    int a = 0;
    for (int level = 0; level < tv.levels; ++level) {
        node = 2 * node + (ax_get(q, a) < tv.split_at(node) ? 1 : 2);
        a = ax_next<D>(a);
    }
    key[i] = (uint32_t)((node - tv.n_nodes) >> shift);
}

// ---------------------------------------------------------------------------------------------
// Morton keys: the Morton code of a query's cell in a 2^B-per-axis grid over a box (B*D <= 24).
// The forward presort uses the queries' own bounding box and the finest grid, so queries
// outside the tree's cloud are grouped by where they really are.  The backward's canonical
// order uses the reference points' bounding box and B from canonical_morton_bits(Q, D)
// (knn_gpu.hpp), the same rule in the single-tree and the batched backward.
// ---------------------------------------------------------------------------------------------
// Bits per axis of the forward presort's grid (measured on MI355X): d = 3, 8 bits (a 24-bit key,
// still three radix passes; plain workload traversal 7.92 ms against 8.23 with 7 bits, depth 13
// 20.29 against 21.33); d = 8, 3 bits (24-bit key; 90.4 ms per 500K queries against 94.0 with 2).
#ifndef TK_MORTON_BITS_3D
#define TK_MORTON_BITS_3D 8
#endif
#ifndef TK_MORTON_BITS_8D
#define TK_MORTON_BITS_8D 3
#endif
template <int D>
struct MortonBits {
    static constexpr int kBits = D == 1 ? 20 : D == 2 ? 10 : D == 3 ? TK_MORTON_BITS_3D : TK_MORTON_BITS_8D;
    static constexpr int kBuckets = 1 << (kBits * D);
};

// Bits 0, 1, 2, .. of v at bits 0, D, 2D, .. (D = 2: 16 of them, D = 3: 10).
template <int D>
__host__ __device__ __forceinline__ uint32_t spread_bits(uint32_t v) {
    static_assert(D == 2 || D == 3, "interleaves of two and three axes");
    if constexpr (D == 2) {
        v = (v | (v << 8)) & 0x00ff00ffu;
        v = (v | (v << 4)) & 0x0f0f0f0fu;
        v = (v | (v << 2)) & 0x33333333u;
        v = (v | (v << 1)) & 0x55555555u;
    } else {
        v = (v | (v << 16)) & 0x030000ffu;
        v = (v | (v << 8)) & 0x0300f00fu;
        v = (v | (v << 4)) & 0x030c30c3u;
        v = (v | (v << 2)) & 0x09249249u;
    }
    return v;
}

// Integer coordinates of q's cell; lo/hi are the box, converted to float.  Queries outside the box fall
// into the boundary cells.
template <typename T, int D>
__device__ __forceinline__ void grid_cell(const float* lo, const float* hi, int bits, const T* __restrict__ q,
                                          uint32_t (&x)[D]) {
    const float cells = (float)(1 << bits);
#pragma unroll
    for (int a = 0; a < D; ++a) {
        const float scale = hi[a] > lo[a] ? cells / (hi[a] - lo[a]) : 0.0f;
        const float v = ((float)q[a] - lo[a]) * scale;
        x[a] = (uint32_t)fminf(fmaxf(v, 0.0f), cells - 1.0f);
    }
}

// Morton code of q's cell: bit b of axis a at bit b * D + a.
template <typename T, int D>
__device__ __forceinline__ uint32_t morton_cell(const float* lo, const float* hi, int bits, const T* __restrict__ q) {
    uint32_t x[D];
    grid_cell<T, D>(lo, hi, bits, q, x);
    uint32_t code = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        if constexpr (D == 1) {
            code = x[a];
        } else if constexpr (D <= 3) {
            code |= spread_bits<D>(x[a]) << a;
        } else {
            for (int b = 0; b < bits; ++b) code |= ((x[a] >> b) & 1u) << (b * D + a);
        }
    }
    return code;
}

// Hilbert index of a cell of the grid with kBits bits an axis: the cell's integer coordinates go
// through Skilling's transpose transform (J. Skilling, "Programming the Hilbert curve", AIP Conf.
// Proc. 707, 2004: undo the excess work, then Gray-encode), and the transposed coordinates are
// interleaved most significant bit first.  Consecutive indices are adjacent cells, which the
// Z-order's jumps between blocks of cells are not.  Bound by VALU issue; without branches, with the Gray
// code's suffix parities and the interleave by doubling shifts: 16M queries, d = 3,
// 127 -> 78 us against the loops over bits.
template <int D, int kBits>
__host__ __device__ __forceinline__ uint32_t hilbert_index(uint32_t (&x)[D]) {
    static_assert(D <= 3 && kBits >= 1 && kBits <= (D == 1 ? 31 : D == 2 ? 16 : 10), "one, two and three axes");
#pragma unroll
    for (int k = kBits - 1; k > 0; --k) {
        const uint32_t p = (1u << k) - 1u;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            // bit k of x[a] set: invert the low bits of x[0]; else exchange those of x[0] and x[a]
            const uint32_t set = 0u - ((x[a] >> k) & 1u);
            const uint32_t t = (x[0] ^ x[a]) & p & ~set;
            x[0] ^= t | (p & set);
            if (a > 0) x[a] ^= t;
        }
    }
#pragma unroll
    for (int a = 1; a < D; ++a) x[a] ^= x[a - 1];
    uint32_t t = x[D - 1] >> 1;  // bit j becomes the parity of the bits above j
    t ^= t >> 1;
    t ^= t >> 2;
    t ^= t >> 4;
    t ^= t >> 8;
    t ^= t >> 16;
#pragma unroll
    for (int a = 0; a < D; ++a) x[a] ^= t;
    uint32_t code = 0;
#pragma unroll
    for (int a = 0; a < D; ++a) {
        if constexpr (D == 1) code = x[a];
        else code |= spread_bits<D>(x[a]) << (D - 1 - a);
    }
    return code;
}

// Bounding box of n points, one partial box per workgroup: part[block][0..D) = min, [D..2D) = max (NaN
// coordinates left out).  The reader reduces the partials (reduce_boxes): no atomics, whose
// same-address updates took 20 of the 27 us of a 1M-point box, and nothing to initialise.
constexpr int kBoxBlock = 256;
constexpr int kMaxBoxParts = 512;  // most workgroups of bbox_kernel

inline int box_parts(int64_t n) {
    const int64_t b = (n + 4 * kBoxBlock - 1) / (4 * kBoxBlock);
    return (int)(b < 1 ? 1 : b > kMaxBoxParts ? kMaxBoxParts : b);
}

// min / max over the 64 lanes, then over the workgroup's wavefronts through LDS; the result is in
// every thread.
template <typename T, int D>
__device__ __forceinline__ void block_box(T (&lo)[D], T (&hi)[D], T (*s_lo)[D], T (*s_hi)[D]) {
#pragma unroll
    for (int a = 0; a < D; ++a) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            lo[a] = fmin(lo[a], __shfl_xor(lo[a], off, 64));
            hi[a] = fmax(hi[a], __shfl_xor(hi[a], off, 64));
        }
    }
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            s_lo[w][a] = lo[a];
            s_hi[w][a] = hi[a];
        }
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < D; ++a) {
        lo[a] = s_lo[0][a];
        hi[a] = s_hi[0][a];
        for (int v = 1; v < kBoxBlock / 64; ++v) {
            lo[a] = fmin(lo[a], s_lo[v][a]);
            hi[a] = fmax(hi[a], s_hi[v][a]);
        }
    }
}

template <typename T, int D>
__global__ __launch_bounds__(kBoxBlock) void bbox_kernel(const T* __restrict__ pts, int64_t n, T* __restrict__ part) {
    __shared__ T s_lo[kBoxBlock / 64][D], s_hi[kBoxBlock / 64][D];
    T lo[D], hi[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        lo[a] = pos_inf<T>();
        hi[a] = -pos_inf<T>();
    }
    const int64_t stride = (int64_t)gridDim.x * kBoxBlock;
#pragma unroll 4
    for (int64_t i = (int64_t)blockIdx.x * kBoxBlock + threadIdx.x; i < n; i += stride) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            const T v = pts[i * D + a];
            lo[a] = fmin(lo[a], v);
            hi[a] = fmax(hi[a], v);
        }
    }
    block_box<T, D>(lo, hi, s_lo, s_hi);
    if (threadIdx.x < D) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            if (a == (int)threadIdx.x) {
                part[(int64_t)blockIdx.x * 2 * D + a] = lo[a];
                part[(int64_t)blockIdx.x * 2 * D + D + a] = hi[a];
            }
        }
    }
}

// Cell keys over the box of n_part partials (bbox_kernel): the Hilbert index with kHilbert (the forward
// presort at d <= 3: plain workload traversal 7.78 ms against 7.88 with the Morton code, fp64
// workload 1.41 against 1.49; at d = 8 the Morton code is faster, 90.6 against 92.2 ms), else the
// Morton code (always for the backward's canonical order).  Every workgroup reduces the partials,
// then strides over the queries (at most kMaxKeyBlocks workgroups, so that the reduction stays small
// beside the queries).
constexpr int kMaxKeyBlocks = 1024;
inline unsigned key_blocks(int64_t nq) {
    const int64_t b = (nq + kBoxBlock - 1) / kBoxBlock;
    return (unsigned)(b > kMaxKeyBlocks ? kMaxKeyBlocks : b);
}
template <typename T, int D, bool kHilbert>
__global__ __launch_bounds__(kBoxBlock) void morton_bucket_kernel(const T* __restrict__ queries, int64_t nq,
                                                                  const T* __restrict__ part, int n_part, int bits,
                                                                  uint32_t* __restrict__ key) {
    __shared__ T s_lo[kBoxBlock / 64][D], s_hi[kBoxBlock / 64][D];
    T blo[D], bhi[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        blo[a] = pos_inf<T>();
        bhi[a] = -pos_inf<T>();
    }
    for (int p = threadIdx.x; p < n_part; p += kBoxBlock) {
#pragma unroll
        for (int a = 0; a < D; ++a) {
            blo[a] = fmin(blo[a], part[(int64_t)p * 2 * D + a]);
            bhi[a] = fmax(bhi[a], part[(int64_t)p * 2 * D + D + a]);
        }
    }
    block_box<T, D>(blo, bhi, s_lo, s_hi);
    float lo[D], hi[D];
#pragma unroll
    for (int a = 0; a < D; ++a) {
        lo[a] = (float)blo[a];
        hi[a] = (float)bhi[a];
    }
    const int64_t stride = (int64_t)gridDim.x * kBoxBlock;
    for (int64_t i = (int64_t)blockIdx.x * kBoxBlock + threadIdx.x; i < nq; i += stride)
        if constexpr (kHilbert) {
            uint32_t x[D];
            grid_cell<T, D>(lo, hi, MortonBits<D>::kBits, queries + i * D, x);
            key[i] = hilbert_index<D, MortonBits<D>::kBits>(x);
        } else {
            key[i] = morton_cell<T, D>(lo, hi, bits, queries + i * D);
        }
}

}  // namespace tk
