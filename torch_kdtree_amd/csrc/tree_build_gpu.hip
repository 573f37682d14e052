// GPU tree build: the layout of createKDTree (src/kdtree.hpp:418-534) built on the device, for one
// tree or for many trees at once (a forest over one concatenated point array).
//
// The reference recurses node by node: at a node of depth l it sorts the node's points by axis
// l mod dims, takes the median of compMedian (src/kdtree.hpp:392-401) as split value, gives the
// first n/2 points to the left child and the rest to the right (src/kdtree.hpp:447-452).  Here
// every depth is one step over all nodes of all trees:
//   1. key[p] = the sortable bits of coordinate (l mod dims) of the point at position p;
//   2. a stable radix sort of (key, p) over the whole array;
//   3. a stable radix sort of the result by node (segment) number, which regroups the positions
//      node by node with each node's points in coordinate order;
//   4. the permutation is composed with that order, and each node's median is read off.
// From the depth at which every node of a tree holds at most kTailPoints points, one kernel (gb_tail_kernel)
// does all its remaining depths: a workgroup takes a node and sorts its descendants' points in LDS by
// (coordinate, previous position), the order the two stable sorts give.
// A single tree stays on the GPU: kernels write its records, index maps, leaf offsets, point boxes and
// group boxes straight into the device tree, and look at a sample of the cloud for exact ties.  The
// trees of a forest are copied to the host.
//
// Bound: the depths above the tail, each a chain of short launches (500K points: 7 of 14 depths).
// 500K points, depth 14, the whole build: 6.9 -> 1.16 ms against a form that sorted every depth over the
// whole array and made records, boxes and the tie sample on the host.
//
// Exactness: the node sizes, split values and leaf contents equal those of the reference
// whenever no node has two points with equal coordinates on its split axis.  With such ties the
// reference's two std::sort calls (one permutation, applied to both arrays: std::sort's moves
// follow its comparison outcomes alone) order the tied points in the order libstdc++'s introsort
// leaves them, which only a sequential emulation could follow; this build orders them by their
// previous position.  It is therefore opt-in; the default build stays the host restatement.
// Points with a NaN coordinate are refused: std::sort's order for them is the introsort's
// accident too.  The host build accepts them and reproduces the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

#include "gpu_common.hpp"
#include "knn_gpu.hpp"
#include "knn_tree.hpp"
#include "tree.hpp"

namespace tk {
namespace {

constexpr int kGbBlock = 256;

__device__ __forceinline__ uint32_t sortable(float x) {
    const uint32_t u = __float_as_uint(x);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ uint64_t sortable(double x) {
    const uint64_t u = (uint64_t)__double_as_longlong(x);
    return (u >> 63) ? ~u : (u | (uint64_t(1) << 63));
}

// Tree of arena position p: the last c with base[c] <= p (bases ascending, base[nc] = total).
__device__ __forceinline__ int tree_of(const int64_t* __restrict__ base, int nc, int64_t p) {
    int lo = 0, hi = nc - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (base[mid] <= p)
            lo = mid;
        else
            hi = mid - 1;
    }
    return lo;
}

// Node (segment) of local position p at depth l in a tree of n points: the reference's split
// rule, n/2 points to the left child and n - n/2 to the right.
__device__ __forceinline__ uint32_t segment_of(int64_t p, int64_t n, int depth) {
    int64_t off = 0, cnt = n;
    uint32_t s = 0;
    for (int i = 0; i < depth; ++i) {
        const int64_t h = cnt >> 1;
        if (p < off + h) {
            cnt = h;
            s = 2 * s;
        } else {
            off += h;
            cnt -= h;
            s = 2 * s + 1;
        }
    }
    return s;
}

// Points [off, off + cnt) of node `node` of depth `depth` in a tree of n points, by the same rule.
__device__ __forceinline__ void node_range(int64_t n, int depth, uint32_t node, int64_t& off, int64_t& cnt) {
    off = 0;
    cnt = n;
    for (int i = depth - 1; i >= 0; --i) {
        const int64_t h = cnt >> 1;
        if ((node >> i) & 1u) {
            off += h;
            cnt -= h;
        } else {
            cnt = h;
        }
    }
}

// What the build met: a NaN among the coordinates it sorted on, a non-finite coordinate, a
// non-finite split value.
enum : int32_t { kFlagNan = 1, kFlagCoord = 2, kFlagSplit = 4 };

struct ForestDev {
    const int64_t* base;      // [nc + 1] first point of each tree in the arena
    const int32_t* levels;    // [nc]
    const int32_t* tail;      // [nc] first depth that gb_tail_kernel does (its levels where there is none)
    const int64_t* split_base;  // [nc] first split value of each tree
    int nc;
};

// key[j] = word `word` (0 low, 1 high) of the sortable coordinate of position p = order[j] (or j);
// positions of trees whose depths over the whole array are done get key 0, so they keep their order.
template <typename T>
__global__ __launch_bounds__(kGbBlock) void gb_key_kernel(const T* __restrict__ pts, int dims,
                                                          const uint32_t* __restrict__ perm,
                                                          const uint32_t* __restrict__ order, int64_t n,
                                                          ForestDev f, int depth, int axis, int word,
                                                          uint32_t* __restrict__ key, uint32_t* __restrict__ val,
                                                          int32_t* __restrict__ flags) {
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n) return;
    const uint32_t p = order ? order[j] : (uint32_t)j;
    const int c = tree_of(f.base, f.nc, p);
    uint32_t k = 0;
    if (f.tail[c] > depth) {
        const T x = pts[(size_t)perm[p] * dims + axis];
        if (x != x) atomicOr(flags, kFlagNan);
        if constexpr (sizeof(T) == 4) {
            k = sortable(x);
        } else {
            const uint64_t u = sortable(x);
            k = word ? (uint32_t)(u >> 32) : (uint32_t)u;
        }
    }
    key[j] = k;
    val[j] = p;
}

// key[j] = node number (over all trees) of position p = order[j] at this depth.
__global__ __launch_bounds__(kGbBlock) void gb_segment_kernel(const uint32_t* __restrict__ order, int64_t n, ForestDev f,
                                                              int depth, const uint32_t* __restrict__ seg_base,
                                                              uint32_t* __restrict__ key, uint32_t* __restrict__ val) {
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n) return;
    const uint32_t p = order[j];
    const int c = tree_of(f.base, f.nc, p);
    const int64_t b = f.base[c];
    const uint32_t s = f.tail[c] > depth ? segment_of((int64_t)p - b, f.base[c + 1] - b, depth) : 0u;
    key[j] = seg_base[c] + s;
    val[j] = p;
}

__global__ __launch_bounds__(kGbBlock) void gb_compose_kernel(const uint32_t* __restrict__ perm,
                                                              const uint32_t* __restrict__ order, int64_t n,
                                                              uint32_t* __restrict__ out) {
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n) return;
    out[j] = perm[order[j]];
}

__global__ __launch_bounds__(kGbBlock) void gb_iota_kernel(uint32_t* __restrict__ out, int64_t n) {
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n) return;
    out[j] = (uint32_t)j;
}

// Split values of the nodes at this depth: task t is node s of tree c (task_base[c] <= t <
// task_base[c + 1]); the node's points, sorted on its axis, sit at its local offset.  The median
// is compMedian's: the middle point for an odd count, else half the sum of the two middle points
// (the sum rounded in T, the halving exact).
template <typename T>
__global__ __launch_bounds__(kGbBlock) void gb_median_kernel(const T* __restrict__ pts, int dims,
                                                             const uint32_t* __restrict__ perm, ForestDev f,
                                                             int depth, int axis,
                                                             const int64_t* __restrict__ task_base,
                                                             int64_t n_tasks, T* __restrict__ split,
                                                             int32_t* __restrict__ flags) {
    const int64_t t = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (t >= n_tasks) return;
    const int c = tree_of(task_base, f.nc, t);
    const uint32_t s = (uint32_t)(t - task_base[c]);
    const int64_t b = f.base[c];
    int64_t off, cnt;
    node_range(f.base[c + 1] - b, depth, s, off, cnt);
    const int64_t mid = b + off + (cnt >> 1);
    const T hi = pts[(size_t)perm[mid] * dims + axis];
    T m = hi;
    if ((cnt & 1) == 0) {
        const T lo = pts[(size_t)perm[mid - 1] * dims + axis];
        m = (lo + hi) * T(0.5);
    }
    if (!__builtin_isfinite(m)) atomicOr(flags, kFlagSplit);
    split[f.split_base[c] + ((int64_t(1) << depth) - 1) + s] = m;
}

// Structured points and local original indices: out[j] = pts[perm[j]], idx[j] = perm[j] - base.
template <typename T>
__global__ __launch_bounds__(kGbBlock) void gb_gather_kernel(const T* __restrict__ pts, int dims,
                                                             const uint32_t* __restrict__ perm, int64_t n, ForestDev f,
                                                             T* __restrict__ out, int32_t* __restrict__ idx) {
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n) return;
    const uint32_t p = perm[j];
    const int c = tree_of(f.base, f.nc, j);
    idx[j] = (int32_t)((int64_t)p - f.base[c]);
    for (int a = 0; a < dims; ++a) out[(size_t)j * dims + a] = pts[(size_t)p * dims + a];
}

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kGbBlock - 1) / kGbBlock); }

int bits_for_count(uint64_t count) {  // bits to number `count` values 0..count-1
    int b = 0;
    while (b < 32 && (uint64_t(1) << b) < count) ++b;
    return b;
}

// Leaf offsets of the reference's split rule (n/2 left, n - n/2 right at every node).
std::vector<int32_t> leaf_offsets(int64_t n, int levels) {
    std::vector<int64_t> sizes{n};
    for (int l = 0; l < levels; ++l) {
        std::vector<int64_t> next;
        next.reserve(sizes.size() * 2);
        for (int64_t s : sizes) {
            next.push_back(s / 2);
            next.push_back(s - s / 2);
        }
        sizes.swap(next);
    }
    std::vector<int32_t> off(sizes.size() + 1, 0);
    for (size_t i = 0; i < sizes.size(); ++i) off[i + 1] = off[i] + (int32_t)sizes[i];
    return off;
}

// The word of lane ^ M (M a power of two below 64) of the wavefront.
template <int M>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
    const int x = (int)v;
    if constexpr (M == 1) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0xb1, 0xf, 0xf, false);       // quad_perm 1,0,3,2
    else if constexpr (M == 2) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0x4e, 0xf, 0xf, false);  // quad_perm 2,3,0,1
    else if constexpr (M == 8) return (uint32_t)__builtin_amdgcn_update_dpp(x, x, 0x128, 0xf, 0xf, false); // row_ror 8
    else if constexpr (M < 32) return (uint32_t)__builtin_amdgcn_ds_swizzle(x, (M << 10) | 0x1f);
    else return (uint32_t)__shfl_xor(x, M, 64);
}
template <int M>
__device__ __forceinline__ uint64_t lane_xor(uint64_t v) {
    return (uint64_t)lane_xor<M>((uint32_t)(v >> 32)) << 32 | lane_xor<M>((uint32_t)v);
}

// Depths from l0 (ForestDev::tail) to the end for one node of depth l0 per workgroup.  Descendant node c of
// depth l0 + i keeps its points in slots [c * P, (c + 1) * P), P = P0 >> i, where P0 <= kTailPoints is the
// smallest power of two that holds the node (its descendants then have at most P points).  A slot holds the
// sortable coordinate and a tag: the point's rank in its node (the order of the depth before, which breaks
// ties as a stable sort does) above its index in the workgroup's tile; empty slots sort last.  A bitonic sort
// orders all descendants of a depth at once, each thread holding kTailItems consecutive slots in registers:
// exchanges within them are register moves, within a wavefront lane permutations, and only the few of 256
// slots and more go through LDS.  Bound by VALU issue (500K points: 138 us for 7 depths from nodes of 3,907;
// with every exchange in LDS 137 us for 6 from nodes of 1,954, and one more 120 us depth over the whole array).
constexpr int kTailPoints = 4096;
constexpr int kTailItems = 4;
constexpr int kTailBlock = kTailPoints / kTailItems;
constexpr uint32_t kTailEmpty = 0xffffffffu;

template <typename T>
using Sortable = decltype(sortable(T()));

// (key, tag) of the slot pair's other element, and which of the two this slot keeps.
template <typename K>
__device__ __forceinline__ void keep_one(K& k, uint32_t& t, K ok, uint32_t ot, bool want_min) {
    const bool less = k < ok || (k == ok && t < ot);
    const bool take = less != want_min;  // (an empty slot equals only empty slots: either choice is the same)
    k = take ? ok : k;
    t = take ? ot : t;
}

// Exchanges at distance J slots of a bitonic stage with runs of `run` slots (whole descendants, run == P,
// ascending; e0 = the thread's first slot).
template <int J, typename K>
__device__ __forceinline__ void bitonic_step(K (&k)[kTailItems], uint32_t (&t)[kTailItems], int e0, int run, int P) {
    if constexpr (J < kTailItems) {
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) {
            if (u & J) continue;
            const bool up = ((e0 + u) & run) == 0 || run == P;
            K ka = k[u], kb = k[u | J];
            uint32_t ta = t[u], tb = t[u | J];
            const bool swap = (ka > kb || (ka == kb && ta > tb)) == up;
            k[u] = swap ? kb : ka;
            k[u | J] = swap ? ka : kb;
            t[u] = swap ? tb : ta;
            t[u | J] = swap ? ta : tb;
        }
    } else {
        constexpr int M = J / kTailItems;
        const bool low = (e0 & J) == 0;
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) {
            const bool up = ((e0 + u) & run) == 0 || run == P;
            keep_one(k[u], t[u], lane_xor<M>(k[u]), lane_xor<M>(t[u]), low == up);
        }
    }
}

template <typename T>
__global__ __launch_bounds__(kTailBlock) void gb_tail_kernel(const T* __restrict__ pts, int dims, uint32_t* perm,
                                                             ForestDev f, const int64_t* __restrict__ task_base,
                                                             int64_t task0, T* __restrict__ split,
                                                             int32_t* __restrict__ flags) {
    using K = Sortable<T>;
    __shared__ K s_key[kTailPoints];
    __shared__ uint32_t s_tag[kTailPoints];  // rank << 16 | tile index
    __shared__ uint32_t point[kTailPoints];  // the tile's points (arena indices)
    const int t = threadIdx.x, e0 = t * kTailItems;
    const int64_t task = task0 + blockIdx.x;
    const int c = tree_of(task_base, f.nc, task);
    const uint32_t seg = (uint32_t)(task - task_base[c]);
    const int l0 = f.tail[c];
    int64_t off, cnt;
    node_range(f.base[c + 1] - f.base[c], l0, seg, off, cnt);
    const int64_t first = f.base[c] + off;
    const int n = (int)cnt;
    const int levels = f.levels[c];
    for (int e = t; e < n; e += kTailBlock) point[e] = perm[first + e];
    K key[kTailItems];
    uint32_t tag[kTailItems];
#pragma unroll
    for (int u = 0; u < kTailItems; ++u) tag[u] = e0 + u < n ? (uint32_t)(e0 + u) << 16 | (uint32_t)(e0 + u) : kTailEmpty;
    __syncthreads();
    int bad = 0;
    int P = kTailPoints;
    while (P > 1 && P / 2 >= n) P >>= 1;
    for (int l = l0; l < levels; ++l, P >>= 1) {
        const int axis = l % dims;
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) {
            key[u] = ~K(0);
            if (tag[u] != kTailEmpty) {
                const T x = pts[(size_t)point[tag[u] & 0xffffu] * dims + axis];
                if (x != x) bad |= kFlagNan;
                key[u] = sortable(x);
            }
        }
        for (int run = 2; run <= P; run <<= 1) {
            for (int j = run >> 1; j >= 64 * kTailItems; j >>= 1) {
                // distances beyond a wavefront's slots
#pragma unroll
                for (int u = 0; u < kTailItems; ++u) {
                    s_key[e0 + u] = key[u];
                    s_tag[e0 + u] = tag[u];
                }
                __syncthreads();
                const bool low = (e0 & j) == 0;
#pragma unroll
                for (int u = 0; u < kTailItems; ++u) {
                    const int o = (e0 + u) ^ j;
                    const bool up = ((e0 + u) & run) == 0 || run == P;
                    keep_one(key[u], tag[u], s_key[o], s_tag[o], low == up);
                }
                __syncthreads();
            }
            if (run >= 256) bitonic_step<128>(key, tag, e0, run, P);
            if (run >= 128) bitonic_step<64>(key, tag, e0, run, P);
            if (run >= 64) bitonic_step<32>(key, tag, e0, run, P);
            if (run >= 32) bitonic_step<16>(key, tag, e0, run, P);
            if (run >= 16) bitonic_step<8>(key, tag, e0, run, P);
            if (run >= 8) bitonic_step<4>(key, tag, e0, run, P);
            if (run >= 4) bitonic_step<2>(key, tag, e0, run, P);
            bitonic_step<1>(key, tag, e0, run, P);
        }
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) s_tag[e0 + u] = tag[u];
        __syncthreads();
        // medians, one descendant node per thread
        const int nodes = 1 << (l - l0);
        for (int s = t; s < nodes; s += kTailBlock) {
            int64_t o, m;
            node_range(n, l - l0, (uint32_t)s, o, m);
            const int mid = s * P + (int)(m >> 1);
            const T hi = pts[(size_t)point[s_tag[mid] & 0xffffu] * dims + axis];
            T med = hi;
            if ((m & 1) == 0) {
                const T lo = pts[(size_t)point[s_tag[mid - 1] & 0xffffu] * dims + axis];
                med = (lo + hi) * T(0.5);
            }
            if (!__builtin_isfinite(med)) bad |= kFlagSplit;
            split[f.split_base[c] + ((int64_t(1) << l) - 1) + ((int64_t)seg << (l - l0)) + s] = med;
        }
        __syncthreads();
        // ranks: the next depth's children take their slots, or the order goes out
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) s_tag[e0 + u] = kTailEmpty;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) {
            if (tag[u] == kTailEmpty) continue;
            const int s = (e0 + u) / P, r = (e0 + u) & (P - 1);
            int64_t o, m;
            node_range(n, l - l0, (uint32_t)s, o, m);
            if (l + 1 == levels) {
                perm[first + o + r] = point[tag[u] & 0xffffu];
                continue;
            }
            const int h = (int)(m >> 1), child = r < h ? 0 : 1, rank = r - child * h;
            s_tag[s * P + child * (P >> 1) + rank] = (uint32_t)rank << 16 | (tag[u] & 0xffffu);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kTailItems; ++u) tag[u] = s_tag[e0 + u];
        __syncthreads();
    }
    if (bad) atomicOr(flags, bad);
}

// ------------------------------------------------------------------------------------------
// The device tree of a single tree, from its permutation.
// ------------------------------------------------------------------------------------------
// Records, index maps and the kRecPad zero records after the last point.
template <typename T, int D>
__global__ __launch_bounds__(kGbBlock) void gb_records_kernel(const T* __restrict__ pts, const uint32_t* __restrict__ perm,
                                                              int64_t n, unsigned char* __restrict__ recs,
                                                              int32_t* __restrict__ shuffled, int32_t* __restrict__ inv,
                                                              int32_t* __restrict__ flags) {
    using L = RecLayout<T, D>;
    const int64_t j = (int64_t)blockIdx.x * kGbBlock + threadIdx.x;
    if (j >= n + kRecPad) return;
    uint32_t w[L::kWords] = {};
    if (j < n) {
        const uint32_t p = perm[j];
        T c[D];
        bool finite = true;
#pragma unroll
        for (int a = 0; a < D; ++a) {
            c[a] = pts[(size_t)p * D + a];
            finite = finite && __builtin_isfinite(c[a]);
        }
        if (!finite) atomicOr(flags, kFlagCoord);
        __builtin_memcpy(w, c, sizeof(c));
        if constexpr (L::kHasIdx) w[L::kIdxWord] = p;
        shuffled[j] = (int32_t)p;
        inv[p] = (int32_t)j;
    }
    uint32_t* out = reinterpret_cast<uint32_t*>(recs + (size_t)j * L::kBytes);
    if constexpr (L::kWords % 4 == 0) {
#pragma unroll
        for (int i = 0; i < L::kWords; i += 4) *reinterpret_cast<uint4*>(out + i) = make_uint4(w[i], w[i + 1], w[i + 2], w[i + 3]);
    } else {
#pragma unroll
        for (int i = 0; i < L::kWords; ++i) out[i] = w[i];
    }
}

template <typename T, int D>
__device__ __forceinline__ void store_box(unsigned char* __restrict__ boxes, int64_t i, const T (&lo)[D], const T (&hi)[D]) {
    constexpr int kPad = BoxLayout<T, D>::kPad;
    T v[2 * kPad] = {};
#pragma unroll
    for (int a = 0; a < D; ++a) {
        v[a] = lo[a];
        v[kPad + a] = hi[a];
    }
    T* out = reinterpret_cast<T*>(boxes + (size_t)i * BoxLayout<T, D>::kBytes);
#pragma unroll
    for (int a = 0; a < 2 * kPad; ++a) out[a] = v[a];
}

// Box of the records [b, e), each lane of W (a power of two, at most 64) taking every W-th; the result in
// every lane.  NaN coordinates are left out (fmin / fmax), as in the host build's boxes.
template <typename T, int D, int W>
__device__ __forceinline__ void lane_box(const unsigned char* __restrict__ recs, int64_t b, int64_t e, int lane, T (&lo)[D],
                                         T (&hi)[D]) {
#pragma unroll
    for (int a = 0; a < D; ++a) {
        lo[a] = pos_inf<T>();
        hi[a] = -pos_inf<T>();
    }
    for (int64_t s = b + lane; s < e; s += W) {
        const Rec<T, D> r = load_rec<T, D>(recs, (int32_t)s);
#pragma unroll
        for (int a = 0; a < D; ++a) {
            lo[a] = fmin(lo[a], r.c[a]);
            hi[a] = fmax(hi[a], r.c[a]);
        }
    }
#pragma unroll
    for (int a = 0; a < D; ++a) {
#pragma unroll
        for (int o = (W < 64 ? W : 64) / 2; o > 0; o >>= 1) {
            lo[a] = fmin(lo[a], __shfl_xor(lo[a], o, 64));
            hi[a] = fmax(hi[a], __shfl_xor(hi[a], o, 64));
        }
    }
}

// Leaf offsets and leaf boxes, W threads a leaf: 16 for small leaves, a whole workgroup for big ones.
template <typename T, int D, int W>
__global__ __launch_bounds__(kGbBlock) void gb_leaves_kernel(const unsigned char* __restrict__ recs, int64_t n, int levels,
                                                             int32_t* __restrict__ leaf_off,
                                                             unsigned char* __restrict__ boxes) {
    const int64_t leaf = ((int64_t)blockIdx.x * kGbBlock + threadIdx.x) / W;
    const int64_t n_leaves = int64_t(1) << levels;
    if (leaf >= n_leaves) return;
    int64_t off, cnt;
    node_range(n, levels, (uint32_t)leaf, off, cnt);
    T lo[D], hi[D];
    lane_box<T, D, W>(recs, off, off + cnt, (int)(threadIdx.x % W), lo, hi);
    if constexpr (W > 64) {
        __shared__ T s_lo[W / 64][D], s_hi[W / 64][D];
        if ((threadIdx.x & 63) == 0) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                s_lo[threadIdx.x >> 6][a] = lo[a];
                s_hi[threadIdx.x >> 6][a] = hi[a];
            }
        }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < D; ++a) {
            for (int v = 0; v < W / 64; ++v) {
                lo[a] = fmin(lo[a], s_lo[v][a]);
                hi[a] = fmax(hi[a], s_hi[v][a]);
            }
        }
    }
    if (threadIdx.x % W == 0) {
        store_box<T, D>(boxes, n_leaves - 1 + leaf, lo, hi);
        leaf_off[leaf] = (int32_t)off;
        if (leaf == 0) leaf_off[n_leaves] = (int32_t)n;
    }
}

// Boxes of the h depths above depth `bottom` (whose boxes are there): a workgroup takes one node of
// depth bottom - h, h <= 7 (one thread per node of depth `bottom` below it).
constexpr int kUpDepths = 7;
constexpr int kUpBlock = 1 << kUpDepths;
template <typename T, int D>
__global__ __launch_bounds__(kUpBlock) void gb_up_kernel(unsigned char* __restrict__ boxes, int bottom, int h) {
    __shared__ T s_lo[kUpBlock][D], s_hi[kUpBlock][D];
    const int t = threadIdx.x;
    const int64_t top = blockIdx.x;
    T lo[D], hi[D];
    if (t < (1 << h)) {
        const BoxVals<T, D> b = load_box<T, D>(boxes, (int32_t)((int64_t(1) << bottom) - 1 + (top << h) + t));
#pragma unroll
        for (int a = 0; a < D; ++a) {
            s_lo[t][a] = b.lo[a];
            s_hi[t][a] = b.hi[a];
        }
    }
    for (int i = 1; i <= h; ++i) {
        __syncthreads();
        const bool on = t < (1 << (h - i));
        if (on) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                lo[a] = fmin(s_lo[2 * t][a], s_lo[2 * t + 1][a]);
                hi[a] = fmax(s_hi[2 * t][a], s_hi[2 * t + 1][a]);
            }
            store_box<T, D>(boxes, (int64_t(1) << (bottom - i)) - 1 + (top << (h - i)) + t, lo, hi);
        }
        __syncthreads();
        if (on) {
#pragma unroll
            for (int a = 0; a < D; ++a) {
                s_lo[t][a] = lo[a];
                s_hi[t][a] = hi[a];
            }
        }
    }
}

// Group boxes (16 lanes each): group g belongs to the last leaf whose first group is at most g.
template <typename T, int D>
__global__ __launch_bounds__(kGbBlock) void gb_groups_kernel(const unsigned char* __restrict__ recs, int64_t n, int levels,
                                                             const int32_t* __restrict__ group_base, int32_t n_groups,
                                                             unsigned char* __restrict__ gboxes) {
    static_assert(kGroupRecs == 16, "one record per lane");
    const int64_t g = ((int64_t)blockIdx.x * kGbBlock + threadIdx.x) / kGroupRecs;
    if (g >= n_groups) return;
    int32_t lo_leaf = 0, hi_leaf = (int32_t)(int64_t(1) << levels) - 1;
    while (lo_leaf < hi_leaf) {
        const int32_t mid = lo_leaf + (hi_leaf - lo_leaf + 1) / 2;
        if (group_base[mid] <= g) lo_leaf = mid;
        else hi_leaf = mid - 1;
    }
    int64_t off, cnt;
    node_range(n, levels, (uint32_t)lo_leaf, off, cnt);
    const int64_t b = off + (g - group_base[lo_leaf]) * kGroupRecs;
    const int64_t e = min(off + cnt, b + kGroupRecs);
    T lo[D], hi[D];
    lane_box<T, D, kGroupRecs>(recs, b, e, (int)(threadIdx.x % kGroupRecs), lo, hi);
    if (threadIdx.x % kGroupRecs == 0) store_box<T, D>(gboxes, g, lo, hi);
}

// The sample of cloud_ties_often (knn_gpu.hip): up to kTieLeaves leaves, kTieLeafPoints points of each.
// Workgroup a < D counts the distinct values on axis a (a hash set in LDS; -0 equals 0, and a double
// enters as a 32-bit mix of its bits, a step of MurmurHash3's 64-bit finaliser); the last ones count, per
// leaf, the points that repeat an earlier point of the leaf's sample.
constexpr int kTieLeaves = 256;
constexpr int kTieLeafPoints = 64;
constexpr int kTieBlock = 1024;
constexpr int kTieSlots = 2 * kTieLeaves * kTieLeafPoints;

__device__ __forceinline__ uint32_t value_mix(float x) { return x == 0.f ? 0u : __float_as_uint(x); }
__device__ __forceinline__ uint32_t value_mix(double x) {
    if (x == 0.0) return 0u;
    uint64_t u = (uint64_t)__double_as_longlong(x);
    u ^= u >> 33;
    u *= 0xff51afd7ed558ccdull;
    u ^= u >> 33;
    return (uint32_t)u;
}

template <typename T, int D>
__global__ __launch_bounds__(kTieBlock) void gb_ties_kernel(const unsigned char* __restrict__ recs, int64_t n, int levels,
                                                            int32_t* __restrict__ counts) {
    extern __shared__ uint32_t table[];
    __shared__ int32_t total;
    const int t = threadIdx.x;
    const int64_t n_leaves = int64_t(1) << levels;
    const int leaves = (int)min(n_leaves, (int64_t)kTieLeaves);
    // record of sample point e (leaf e / 64 of the sample, its point e % 64), -1 beyond the leaf
    const auto record = [&](int e) -> int64_t {
        int64_t off, cnt;
        node_range(n, levels, (uint32_t)((int64_t)(e / kTieLeafPoints) * n_leaves / leaves), off, cnt);
        const int r = e % kTieLeafPoints;
        return r < cnt ? off + r : -1;
    };
    if (t == 0) total = 0;
    if (blockIdx.x < D) {
        for (int i = t; i < kTieSlots; i += kTieBlock) table[i] = kTailEmpty;
        __syncthreads();
        int mine = 0;
        for (int e = t; e < leaves * kTieLeafPoints; e += kTieBlock) {
            const int64_t s = record(e);
            if (s < 0) continue;
            const Rec<T, D> r = load_rec<T, D>(recs, (int32_t)s);
            T x = r.c[0];
#pragma unroll
            for (int a = 1; a < D; ++a)
                if (a == (int)blockIdx.x) x = r.c[a];
            const uint32_t v = min(value_mix(x), kTailEmpty - 1u);
            // (at most half of the slots fill up, so the probe ends)
            for (uint32_t h = (v * 2654435761u) % kTieSlots;; h = (h + 1) % kTieSlots) {
                const uint32_t old = atomicCAS(&table[h], kTailEmpty, v);
                if (old == kTailEmpty) ++mine;
                if (old == kTailEmpty || old == v) break;
            }
        }
        atomicAdd(&total, mine);
        __syncthreads();
        if (t == 0) counts[2 + blockIdx.x] = total;
    } else {
        __syncthreads();
        int dups = 0, sampled = 0;
        const int e = (int)(blockIdx.x - D) * kTieBlock + t;
        if (e < leaves * kTieLeafPoints) {
            const int64_t s = record(e);
            if (s >= 0) {
                sampled = 1;
                const Rec<T, D> r = load_rec<T, D>(recs, (int32_t)s);
                bool dup = false;
                for (int64_t u = s - e % kTieLeafPoints; u < s && !dup; ++u) {
                    const Rec<T, D> o = load_rec<T, D>(recs, (int32_t)u);
                    dup = true;
#pragma unroll
                    for (int a = 0; a < D; ++a) dup = dup && o.c[a] == r.c[a];
                }
                dups = dup;
            }
        }
        if (dups) atomicAdd(&counts[0], 1);
        if (sampled) atomicAdd(&total, 1);
        __syncthreads();
        if (t == 0) atomicAdd(&counts[1], total);
    }
}

// Small arrays and flags that go to the device in one copy.
struct HostPack {
    std::vector<unsigned char> bytes;
    template <typename U>
    size_t add(const U* p, size_t n) {
        const size_t at = (bytes.size() + 7) & ~size_t(7);
        bytes.resize(at + n * sizeof(U));
        if (n) std::memcpy(&bytes[at], p, n * sizeof(U));
        return at;
    }
};
constexpr int kGbInts = 16;  // flags, then the tie sample's counts: duplicates, points, distinct per axis

// Enqueues the kernels that fill the device tree and the tie counts.
template <typename T, int D>
void fill_device_tree(const T* pts, const uint32_t* perm, const Tree& t, DeviceTree& d, int32_t n_groups, int32_t* ints,
                      hipStream_t s) {
    const int64_t n = t.n_points;
    hipLaunchKernelGGL((gb_records_kernel<T, D>), dim3(grid_for(n + kRecPad)), dim3(kGbBlock), 0, s, pts, perm, n, d.recs,
                       d.shuffled, d.inv_shuffled, ints);
    if (n >= 512 * (int64_t)t.n_leaves)
        hipLaunchKernelGGL((gb_leaves_kernel<T, D, kGbBlock>), dim3(grid_for((int64_t)t.n_leaves * kGbBlock)), dim3(kGbBlock),
                           0, s, d.recs, n, t.levels, d.leaf_off, d.boxes);
    else
        hipLaunchKernelGGL((gb_leaves_kernel<T, D, 16>), dim3(grid_for((int64_t)t.n_leaves * 16)), dim3(kGbBlock), 0, s,
                           d.recs, n, t.levels, d.leaf_off, d.boxes);
    TK_HIP_CHECK(hipGetLastError());
    for (int bottom = t.levels; bottom > 0;) {
        const int h = std::min(bottom, kUpDepths);
        hipLaunchKernelGGL((gb_up_kernel<T, D>), dim3(1u << (bottom - h)), dim3(kUpBlock), 0, s, d.boxes, bottom, h);
        bottom -= h;
    }
    if (n_groups)
        hipLaunchKernelGGL((gb_groups_kernel<T, D>), dim3(grid_for((int64_t)n_groups * kGroupRecs)), dim3(kGbBlock), 0, s,
                           d.recs, n, t.levels, d.group_base, n_groups, d.group_boxes);
    const int dup_blocks = kTieLeaves * kTieLeafPoints / kTieBlock;
    const void* fn = reinterpret_cast<const void*>(&gb_ties_kernel<T, D>);
    TK_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, kTieSlots * 4));
    hipLaunchKernelGGL((gb_ties_kernel<T, D>), dim3(D + dup_blocks), dim3(kTieBlock), kTieSlots * 4, s, d.recs, n, t.levels,
                       ints + 1);
    TK_HIP_CHECK(hipGetLastError());
}

const char* const kNanMessage =
    "GPU tree build: the points contain NaN (the host build, builder=\"cpu\", accepts them and orders "
    "them as the reference does)";

// The trees' permutations and split values on the device: all kernels on s.
template <typename T>
struct ForestSort {
    std::unique_ptr<StreamScratch> scratch;
    HostPack pack;  // the source of an asynchronous copy: lives until the stream has been waited for
    std::vector<int64_t> base, split_base;
    int64_t n = 0, n_split = 0;
    uint32_t* perm = nullptr;  // [n] arena index of each structured position
    T* split = nullptr;        // [n_split]
    int32_t* ints = nullptr;   // [kGbInts]
    ForestDev f{};

    // split_out: where the split values go (null: scratch)
    void run(const T* pts, const int64_t* n_points, const int32_t* levels, int nc, int dims, T* split_out, hipStream_t s) {
        base.assign(nc + 1, 0);
        split_base.assign(nc, 0);
        for (int c = 0; c < nc; ++c) {
            base[c + 1] = base[c] + n_points[c];
            split_base[c] = n_split;
            n_split += total_nodes(levels[c]);
        }
        n = base[nc];
        // Depths [0, tail) of a tree are sorted over the whole array, the rest node by node in LDS.  Each
        // tree has its own: with the deepest tree's for all, the small clouds beside a big one came to the
        // tail in nodes of a few points, a workgroup each (one cloud of 1M points and 200 of 2,048 with 12 levels,
        // plan included: 23.3 ms, now 12.7; 14.6 with every depth over the whole array).
        std::vector<int32_t> tail((size_t)nc);
        std::vector<int64_t> tail_task((size_t)nc + 1, 0);
        int l0 = 0;
        for (int c = 0; c < nc; ++c) {
            int l = 0;
            while (l < levels[c] && ((n_points[c] + (int64_t(1) << l) - 1) >> l) > kTailPoints) ++l;
            tail[(size_t)c] = l;
            tail_task[(size_t)c + 1] = tail_task[(size_t)c] + (l < levels[c] ? int64_t(1) << l : 0);
            l0 = std::max(l0, l);
        }
        // per depth of the first kind: node numbering (segment bases) and median task bases
        std::vector<uint32_t> seg_base((size_t)l0 * nc);
        std::vector<int64_t> task_base((size_t)l0 * (nc + 1));
        std::vector<uint64_t> seg_total(l0);
        for (int l = 0; l < l0; ++l) {
            uint64_t sb = 0;
            int64_t tb = 0;
            for (int c = 0; c < nc; ++c) {
                seg_base[(size_t)l * nc + c] = (uint32_t)sb;
                task_base[(size_t)l * (nc + 1) + c] = tb;
                const bool active = tail[(size_t)c] > l;
                sb += active ? (uint64_t(1) << l) : 1u;
                tb += active ? (int64_t(1) << l) : 0;
            }
            task_base[(size_t)l * (nc + 1) + nc] = tb;
            seg_total[l] = sb;
            if (sb > (uint64_t(1) << 32)) throw std::runtime_error("GPU tree build: too many nodes at one depth");
        }
        const std::vector<int32_t> zeros(kGbInts, 0);
        const size_t at_ints = pack.add(zeros.data(), zeros.size());
        const size_t at_base = pack.add(base.data(), base.size());
        const size_t at_levels = pack.add(levels, (size_t)nc);
        const size_t at_tail = pack.add(tail.data(), tail.size());
        const size_t at_split = pack.add(split_base.data(), split_base.size());
        const size_t at_seg = pack.add(seg_base.data(), seg_base.size());
        const size_t at_task = pack.add(task_base.data(), task_base.size());
        const size_t at_tail_task = pack.add(tail_task.data(), tail_task.size());

        size_t total = 0;
        const auto take = [&](size_t bytes) {
            const size_t at = total;
            total += (bytes + 255) & ~size_t(255);
            return at;
        };
        const size_t at_pack = take(pack.bytes.size());
        const size_t at_perm = take(4 * (size_t)n), at_perm2 = take(4 * (size_t)n);
        const bool global = l0 > 0;
        const size_t nw = global ? 4 * (size_t)n : 0;
        const size_t at_key = take(nw), at_val = take(nw), at_key_s = take(nw), at_val_s = take(nw);
        const size_t ws_bytes = global ? radix_sort_workspace(n) : 0;
        const size_t at_ws = take(ws_bytes);
        const size_t at_spl = take(split_out ? 0 : sizeof(T) * (size_t)n_split);
        scratch.reset(new StreamScratch(total, s));
        unsigned char* m = static_cast<unsigned char*>(scratch->ptr);
        TK_HIP_CHECK(hipMemcpyAsync(m + at_pack, pack.bytes.data(), pack.bytes.size(), hipMemcpyHostToDevice, s));
        const unsigned char* dp = m + at_pack;
        ints = reinterpret_cast<int32_t*>(m + at_pack + at_ints);
        f = ForestDev{reinterpret_cast<const int64_t*>(dp + at_base), reinterpret_cast<const int32_t*>(dp + at_levels),
                      reinterpret_cast<const int32_t*>(dp + at_tail), reinterpret_cast<const int64_t*>(dp + at_split), nc};
        const uint32_t* d_seg = reinterpret_cast<const uint32_t*>(dp + at_seg);
        const int64_t* d_task = reinterpret_cast<const int64_t*>(dp + at_task);
        split = split_out ? split_out : reinterpret_cast<T*>(m + at_spl);
        perm = reinterpret_cast<uint32_t*>(m + at_perm);
        uint32_t* perm_next = reinterpret_cast<uint32_t*>(m + at_perm2);
        uint32_t* key = reinterpret_cast<uint32_t*>(m + at_key);
        uint32_t* val = reinterpret_cast<uint32_t*>(m + at_val);
        uint32_t* key_s = reinterpret_cast<uint32_t*>(m + at_key_s);
        uint32_t* val_s = reinterpret_cast<uint32_t*>(m + at_val_s);
        void* ws = m + at_ws;
        if (n == 0) return;
        hipLaunchKernelGGL(gb_iota_kernel, dim3(grid_for(n)), dim3(kGbBlock), 0, s, perm, n);
        TK_HIP_CHECK(hipGetLastError());
        for (int l = 0; l < l0; ++l) {
            const int axis = l % dims;
            // coordinate order (two 32-bit words for doubles: low word first, then high, both stable)
            const int words = sizeof(T) == 8 ? 2 : 1;
            for (int w = 0; w < words; ++w) {
                hipLaunchKernelGGL(gb_key_kernel<T>, dim3(grid_for(n)), dim3(kGbBlock), 0, s, pts, dims, perm,
                                   w == 0 ? (const uint32_t*)nullptr : val_s, n, f, l, axis, words == 2 ? w : 0, key,
                                   val, ints);
                TK_HIP_CHECK(hipGetLastError());
                radix_sort_pairs(key, val, key_s, val_s, n, 32, ws, ws_bytes, s);
            }
            // node order, stable: each node's points stay in coordinate order
            const int seg_bits = bits_for_count(seg_total[l]);
            if (seg_bits > 0) {
                hipLaunchKernelGGL(gb_segment_kernel, dim3(grid_for(n)), dim3(kGbBlock), 0, s, val_s, n, f, l,
                                   d_seg + (size_t)l * nc, key, val);
                TK_HIP_CHECK(hipGetLastError());
                radix_sort_pairs(key, val, key_s, val_s, n, seg_bits, ws, ws_bytes, s);
            }
            hipLaunchKernelGGL(gb_compose_kernel, dim3(grid_for(n)), dim3(kGbBlock), 0, s, perm, val_s, n, perm_next);
            TK_HIP_CHECK(hipGetLastError());
            std::swap(perm, perm_next);
            const int64_t tasks = task_base[(size_t)l * (nc + 1) + nc];
            if (tasks > 0) {
                hipLaunchKernelGGL(gb_median_kernel<T>, dim3(grid_for(tasks)), dim3(kGbBlock), 0, s, pts, dims, perm, f,
                                   l, axis, d_task + (size_t)l * (nc + 1), tasks, split, ints);
                TK_HIP_CHECK(hipGetLastError());
            }
        }
        // (a launch takes fewer than 2^32 threads; forests of very many small clouds have more workgroups than that)
        constexpr int64_t kTailTasks = int64_t(1) << 21;
        static_assert(kTailTasks * kTailBlock < (int64_t(1) << 32), "threads of a launch");
        for (int64_t t0 = 0; t0 < tail_task[(size_t)nc]; t0 += kTailTasks) {
            const unsigned tasks = (unsigned)std::min(kTailTasks, tail_task[(size_t)nc] - t0);
            hipLaunchKernelGGL(gb_tail_kernel<T>, dim3(tasks), dim3(kTailBlock), 0, s, pts, dims, perm, f,
                               reinterpret_cast<const int64_t*>(dp + at_tail_task), t0, split, ints);
            TK_HIP_CHECK(hipGetLastError());
        }
    }
};

template <typename T>
std::vector<Tree*> build_forest_typed(const T* pts, const int64_t* n_points, const int32_t* levels, int nc, int dims,
                                      hipStream_t s) {
    ForestSort<T> fs;
    fs.run(pts, n_points, levels, nc, dims, nullptr, s);
    const int64_t n = fs.n;
    // structured points and local original indices
    StreamScratch out_pts(sizeof(T) * (size_t)n * dims, s), out_idx(sizeof(int32_t) * (size_t)n, s);
    if (n > 0) {
        hipLaunchKernelGGL(gb_gather_kernel<T>, dim3(grid_for(n)), dim3(kGbBlock), 0, s, pts, dims, fs.perm, n, fs.f,
                           static_cast<T*>(out_pts.ptr), static_cast<int32_t*>(out_idx.ptr));
        TK_HIP_CHECK(hipGetLastError());
    }
    int32_t flags = 0;
    std::vector<T> split_h(fs.n_split);
    std::vector<T> pts_h((size_t)n * dims);
    std::vector<int32_t> idx_h(n);
    TK_HIP_CHECK(hipMemcpyAsync(&flags, fs.ints, sizeof(int32_t), hipMemcpyDeviceToHost, s));
    TK_HIP_CHECK(hipMemcpyAsync(split_h.data(), fs.split, sizeof(T) * split_h.size(), hipMemcpyDeviceToHost, s));
    TK_HIP_CHECK(hipMemcpyAsync(pts_h.data(), out_pts.ptr, sizeof(T) * pts_h.size(), hipMemcpyDeviceToHost, s));
    TK_HIP_CHECK(hipMemcpyAsync(idx_h.data(), out_idx.ptr, sizeof(int32_t) * idx_h.size(), hipMemcpyDeviceToHost, s));
    TK_HIP_CHECK(hipStreamSynchronize(s));
    if (flags & kFlagNan) throw std::runtime_error(kNanMessage);

    std::vector<Tree*> out(nc, nullptr);
    try {
        for (int c = 0; c < nc; ++c) {
            std::unique_ptr<Tree> t(new Tree());
            t->dtype = sizeof(T) == 4 ? kF32 : kF64;
            t->dims = dims;
            t->levels = levels[c];
            t->n_points = (int32_t)n_points[c];
            t->n_nodes = total_nodes(levels[c]);
            t->n_leaves = (int32_t)(1u << levels[c]);
            t->split.resize(sizeof(T) * (size_t)t->n_nodes);
            std::memcpy(t->split.data(), split_h.data() + fs.split_base[c], t->split.size());
            t->leaf_off = leaf_offsets(n_points[c], levels[c]);
            t->points.resize(sizeof(T) * (size_t)n_points[c] * dims);
            std::memcpy(t->points.data(), pts_h.data() + (size_t)fs.base[c] * dims, t->points.size());
            t->shuffled.assign(idx_h.begin() + fs.base[c], idx_h.begin() + fs.base[c + 1]);
            finish_tree(*t);
            out[c] = t.release();
        }
    } catch (...) {
        for (Tree* t : out) delete t;
        throw;
    }
    return out;
}

template <typename T>
Tree* build_tree_typed(const T* pts, int64_t n_points, int levels, int dims, int device, hipStream_t s) {
    std::unique_ptr<Tree> t(new Tree());
    t->dtype = sizeof(T) == 4 ? kF32 : kF64;
    t->dims = dims;
    t->levels = levels;
    t->n_points = (int32_t)n_points;
    t->n_nodes = total_nodes(levels);
    t->n_leaves = (int32_t)(1u << levels);
    t->host_ready = false;
    // trees of big leaves: where each leaf's group boxes start
    std::vector<int32_t> gbase;
    if (tree_wants_groups(*t)) {
        const std::vector<int32_t> off = leaf_offsets(n_points, levels);
        gbase.assign(off.size(), 0);
        for (size_t i = 0; i + 1 < off.size(); ++i)
            gbase[i + 1] = gbase[i] + (off[i + 1] - off[i] + kGroupRecs - 1) / kGroupRecs;
    }
    const int32_t n_groups = gbase.empty() ? 0 : gbase.back();
    t->dev = alloc_device_tree(*t, device, n_groups);
    ForestSort<T> fs;
    try {
        DeviceTree& d = *t->dev;
        const int32_t lv = levels;
        fs.run(pts, &n_points, &lv, 1, dims, static_cast<T*>(d.split), s);
        if (n_groups)
            TK_HIP_CHECK(hipMemcpyAsync(d.group_base, gbase.data(), 4 * gbase.size(), hipMemcpyHostToDevice, s));
        switch (dims) {
            case 1: fill_device_tree<T, 1>(pts, fs.perm, *t, d, n_groups, fs.ints, s); break;
            case 2: fill_device_tree<T, 2>(pts, fs.perm, *t, d, n_groups, fs.ints, s); break;
            case 3: fill_device_tree<T, 3>(pts, fs.perm, *t, d, n_groups, fs.ints, s); break;
            case 8: fill_device_tree<T, 8>(pts, fs.perm, *t, d, n_groups, fs.ints, s); break;
            default: throw std::runtime_error("unsupported dims");
        }
        int32_t ints[kGbInts];
        TK_HIP_CHECK(hipMemcpyAsync(ints, fs.ints, sizeof(ints), hipMemcpyDeviceToHost, s));
        TK_HIP_CHECK(hipStreamSynchronize(s));
        if (ints[0] & kFlagNan) throw std::runtime_error(kNanMessage);
        t->finite = (ints[0] & (kFlagCoord | kFlagSplit)) == 0;
        if (!t->finite) d.group_boxes = nullptr, d.group_base = nullptr;
        // the decision of cloud_ties_often on the same sample
        const int64_t dups = ints[1], sampled = ints[2];
        bool ties = sampled >= 2 && dups * 256 > sampled;
        for (int a = 0; a < dims && sampled >= 2; ++a) ties = ties || (int64_t)ints[3 + a] * 2 < sampled;
        t->tie_prone = !t->finite || ties;
    } catch (...) {
        (void)hipStreamSynchronize(s);
        free_device_tree(*t);
        throw;
    }
    return t.release();
}

void check_build(const void* points, const int64_t* n_points, const int32_t* levels, int n_trees, int dims, int dtype) {
    if (n_trees < 1) throw std::runtime_error("GPU tree build: no trees");
    if (!dims_supported(dims))
        throw std::runtime_error("Could not find the KD-Tree for dimensionality " + std::to_string(dims));
    if (dtype != kF32 && dtype != kF64) throw std::runtime_error("Unsupported dtype");
    int64_t total = 0;
    for (int c = 0; c < n_trees; ++c) {
        const int L = levels[c];
        if (L < 1 || L > kMaxLevels)
            throw std::runtime_error("levels must be in [1, " + std::to_string(kMaxLevels) + "]");
        if (n_points[c] < 0 || n_points[c] >= (int64_t(1) << 31))
            throw std::runtime_error("Only 32 bit signed indexing implemented");
        if (n_points[c] < (int64_t(1) << (L - 1)))
            throw std::runtime_error(
                "Error: Ran out of points while building KD-Tree. Either you required too many levels, or you "
                "used a lot of coplanar points");
        total += n_points[c];
    }
    if (total > (int64_t(1) << 28)) throw std::runtime_error("GPU tree build: at most 2^28 points in one build");
    if (total > 0 && !points) throw std::runtime_error("invalid arguments");
}

}  // namespace

std::vector<Tree*> build_trees_gpu(const void* points, const int64_t* n_points, const int32_t* levels, int n_trees,
                                   int dims, int dtype, int device, void* stream) {
    check_build(points, n_points, levels, n_trees, dims, dtype);
    if (device < 0) TK_HIP_CHECK(hipGetDevice(&device));
    DeviceGuard g(device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == kF32) return build_forest_typed<float>(static_cast<const float*>(points), n_points, levels, n_trees, dims, s);
    return build_forest_typed<double>(static_cast<const double*>(points), n_points, levels, n_trees, dims, s);
}

Tree* build_tree_gpu(const void* points, int64_t n_points, int levels, int dims, int dtype, int device, void* stream) {
    const int32_t lv = levels;
    check_build(points, &n_points, &lv, 1, dims, dtype);
    if (device < 0) TK_HIP_CHECK(hipGetDevice(&device));
    DeviceGuard g(device);
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == kF32) return build_tree_typed<float>(static_cast<const float*>(points), n_points, levels, dims, device, s);
    return build_tree_typed<double>(static_cast<const double*>(points), n_points, levels, dims, device, s);
}

}  // namespace tk
