// KD-tree KNN search with G lanes per query (G = 4, 8 or 16), for gfx950.
//
// knn_tree.hpp gives every query one lane: the fewest instructions per query, but one serial chain
// of dependent loads per query (each level of the descent, each sibling box of the climb, each group
// of records), and 64 queries per wavefront.  A call with too few queries to fill the chip is bound by
// that chain; so is a search that scans hundreds of leaves, whose lanes' walks part (d = 8), and a
// list too long for one lane's registers.  Here the G lanes of a group share one query:
//   * descent: the lanes load the split values of the next log2(G) levels below the node at once, and
//     a ballot of the comparisons tells the path;
//   * leaf scan: each lane takes one record of every G, so records are read as contiguous runs;
//   * list: sorted over the lanes, E entries each; an insertion moves the entries of all lanes one
//     slot at once, the last entry of a lane going to the next lane by DPP;
//   * climb: each lane tests one level of the path (the box of its far child), all at the same time, and a ballot
//     picks the deepest level whose far side is to be entered.
// Every test uses the values and the rounding of knn_tree.hpp's search, so the visited leaves,
// their order and the outputs are the same bits.
//
// Why the climb may test its levels together: each test compares the distance to a box on the path with
// the worst distance, and neither changes during a climb (knn_tree.hpp says why the box alone decides).
// So the tests' order does not matter, and the search enters the deepest level that passes, as the
// serial climb does.
#pragma once

#include "knn_tree_launch.hpp"

namespace tk {

// ---------------------------------------------------------------------------------------------
// Group operations.  A group is G consecutive lanes of a wavefront, G <= 16, inside one DPP row.
// ---------------------------------------------------------------------------------------------
template <int CTRL, int BANK = 0xf>
__device__ __forceinline__ int dpp_i32(int old, int src) {
    return __builtin_amdgcn_update_dpp(old, src, CTRL, 0xf, BANK, false);
}

template <typename V, typename F>
__device__ __forceinline__ V per_word(const V& a, const V& b, F&& f) {
    int wa[sizeof(V) / 4], wb[sizeof(V) / 4];
    __builtin_memcpy(wa, &a, sizeof(V));
    __builtin_memcpy(wb, &b, sizeof(V));
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / 4); ++i) wa[i] = f(wa[i], wb[i]);
    V r;
    __builtin_memcpy(&r, wa, sizeof(V));
    return r;
}

constexpr int kDppRowShr1 = 0x111;
constexpr int kDppRowBcast = 0x150;  // row_newbcast: lane n of each row of 16 to the whole row

// v of the previous lane of the group; `first` in the group's first lane (g == 0).
template <int G, typename V>
__device__ __forceinline__ V group_prev(const V& v, const V& first, int g) {
    if constexpr (G == 16) {
        return per_word(first, v, [](int o, int s) { return dpp_i32<kDppRowShr1>(o, s); });
    } else {
        const V p = per_word(first, v, [](int o, int s) { return dpp_i32<kDppRowShr1>(o, s); });
        return g == 0 ? first : p;
    }
}

// v of lane I of the group.
template <int G, int I, typename V>
__device__ __forceinline__ V group_lane(const V& v) {
    return per_word(v, v, [](int, int s) {
        if constexpr (G == 16) return dpp_i32<kDppRowBcast + I>(s, s);
        else if constexpr (G == 8) return dpp_i32<kDppRowBcast + 8 + I, 0xc>(dpp_i32<kDppRowBcast + I, 0x3>(s, s), s);
        else return dpp_i32<I * 0x55>(s, s);  // quad_perm [I,I,I,I]
    });
}

// v0 + v1 + .. + v(D-1) over the group's lanes 0..D-1, left to right.
template <int G, int D, int I = 1, typename V>
__device__ __forceinline__ V group_sum(const V& v, V s) {
    if constexpr (I < D) return group_sum<G, D, I + 1>(v, s + group_lane<G, I>(v));
    else return s;
}

// Bit g: p in lane g of this lane's group, whose first lane is `base`.
template <int G>
__device__ __forceinline__ uint32_t group_ballot(bool p, int base) {
    return (uint32_t)(__ballot(p) >> base) & ((1u << G) - 1u);
}

// ---------------------------------------------------------------------------------------------
// The list of a group: positions 0 .. G*E - 1 in ascending order, lane g holding g*E .. g*E + E - 1.
// The first G*E - k positions hold -inf and never move (as in KBest).  Keys are structured indices
// under the reference policy (insertion after equal distances) and original indices under the
// lower-index policy (ordered by (distance, key)).  Inserting a candidate that the list would
// reject changes nothing.
// ---------------------------------------------------------------------------------------------
template <typename T, int G, int E, bool kLower>
struct GroupList {
    T d[E];
    int32_t x[E];

    __device__ __forceinline__ void init(int k, int g) {
        const int pad = G * E - k;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool is_pad = g * E + e < pad;
            d[e] = is_pad ? -pos_inf<T>() : pos_inf<T>();
            x[e] = kLower && is_pad ? -1 : 0;
        }
    }
    static __device__ __forceinline__ bool after(T de, int32_t xe, T dist, int32_t key) {
        if constexpr (kLower)
            return de > dist || (de == dist && xe > key);
        else
            return de > dist;
    }
    // (dist, key): the same in every lane of the group
    __device__ __forceinline__ void insert(T dist, int32_t key, int g) {
        const T pd = group_prev<G>(d[E - 1], -pos_inf<T>(), g);
        const int32_t px = group_prev<G>(x[E - 1], int32_t(-1), g);
        bool here_next = after(d[E - 1], x[E - 1], dist, key);
#pragma unroll
        for (int e = E - 1; e > 0; --e) {
            const bool shift = after(d[e - 1], x[e - 1], dist, key);
            const bool here = here_next;
            here_next = shift;
            d[e] = KBest<T, 1, false>::med3(d[e - 1], d[e], dist);
            x[e] = shift ? x[e - 1] : (here ? key : x[e]);
        }
        const bool shift = after(pd, px, dist, key);
        d[0] = KBest<T, 1, false>::med3(pd, d[0], dist);
        x[0] = shift ? px : (here_next ? key : x[0]);
    }
};

// ---------------------------------------------------------------------------------------------
// Shape of a group search: U records per lane and chunk (U*G <= 32 candidates staged at a time); with
// record-group boxes a chunk is one group of kGroupRecs records.
// ---------------------------------------------------------------------------------------------
template <typename T, int D, int G, bool kGroups>
struct GroupShape {
    static constexpr int kQueries = kGroupBlock / G;  // per block
    static constexpr bool kWideRec = (int)sizeof(T) * D > 32;
    static constexpr int kU = kGroups ? kGroupRecs / G : G == 16 ? (kWideRec ? 1 : 2) : G == 8 ? (kWideRec ? 2 : 4) : 4;
};

// base[i] through a 32-bit byte offset, for the arrays of nodes and leaves (at most 2^25 entries of at most
// 128 bytes): one shift beside the uniform base address.
template <typename V>
__device__ __forceinline__ V load_at(const V* __restrict__ base, int32_t i) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + (uint32_t)i * (uint32_t)sizeof(V));
}
template <typename T, int D>
__device__ __forceinline__ T node_box_dist(const unsigned char* __restrict__ boxes, int32_t node, const Pt<T, D>& q) {
    return box_dist<T, D>(load_box<T, D>(boxes + (uint32_t)node * (uint32_t)BoxLayout<T, D>::kBytes, 0), q);
}

template <typename T, int D, int G, int E, bool kLower, bool kGroups>
__global__ __launch_bounds__(kGroupBlock) void knn_group_kernel(
    TreeView<T> tv, const T* __restrict__ queries, int64_t nq, const int32_t* __restrict__ order, int k,
    T* __restrict__ out_d, int32_t* __restrict__ out_i, int64_t* __restrict__ out_o) {
    using Shape = GroupShape<T, D, G, kGroups>;
    constexpr int U = Shape::kU;
    constexpr int QB = Shape::kQueries;
    constexpr int K = G * E;
    constexpr int S = G == 16 ? 4 : G == 8 ? 3 : 2;  // levels per descent round
    constexpr int CH = U * G;
    static_assert(CH <= 32 && G - 1 <= kRecPad, "candidate mask and padding records");
    static_assert(D <= G, "a lane per axis");
    static_assert(kMaxLevels <= 24, "32-bit offsets of 2^25 boxes of 128 bytes");
    __shared__ T stage_d[QB * (CH + 1)];
    __shared__ int32_t stage_o[kLower ? QB * (CH + 1) : 1];
    constexpr int kLevelQs = kMaxLevels + 4;  // with the levels that a descent round may look past the last
    static_assert(S <= 4, "levels of a descent round");
    __shared__ T s_q[QB * kLevelQs];

    const int g = (int)(threadIdx.x & (G - 1));
    const int gq = (int)threadIdx.x / G;                  // group of the block
    const int base = (int)(threadIdx.x & 63u & ~(G - 1u));  // first lane of the group in its wavefront
    const int64_t t = xcd_tile(blockIdx.x, gridDim.x) * QB + gq;
    if (t >= nq) return;
    const int64_t qi = order ? (int64_t)order[t] : t;
    Pt<T, D> q;
    load_query<T, D>(queries, qi, q);

    GroupList<T, G, E, kLower> kb;
    kb.init(k, g);
    const int pad = K - k;
    T w = pos_inf<T>();  // the worst entry (k >= 1: the last position is never padding)
    [[maybe_unused]] int32_t wx = 0;
    T* const st_d = stage_d + gq * (CH + 1);
    [[maybe_unused]] int32_t* const st_o = stage_o + (kLower ? gq * (CH + 1) : 0);

    if (has_nan<T, D>(q)) {
        // as nan_fill: the descent's leaf from its end under the reference policy, the empty list
        // under the lower-index policy
        if constexpr (!kLower) {
            int32_t beg = 0, end = 0;
            descent_leaf<T, D>(tv, q, beg, end);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int c = g * E + e - pad;
                const int32_t rec = end - 1 - c;
                if (c >= 0 && rec >= beg) {
                    kb.d[e] = sq_dist<T, D>(q, load_rec<T, D>(tv.recs, rec).c);
                    kb.x[e] = rec;
                }
            }
        }
    } else {
        const int L = tv.levels;
        const int a_lp = axis_of_level<D>(L - 1);
        // q by level, q[l mod D], for the descent (up to S levels past the last)
        T* const s_qg = s_q + gq * kLevelQs;
        for (int l = g; l < kLevelQs; l += G) s_qg[l] = ax_get(q, axis_of_level<D>(l));
        // this lane's place in the descent's subtree (1-based heap index g: depth r, offset g - 2^r)
        const int r = g ? 31 - __builtin_clz(g) : 0;
        const int off = g ? g - (1 << r) : 0;
        // Lane i < D keeps axis i of the reference policy's projected point: pp, q, the levels from the
        // leaf-parents up to the first of that axis, and as a mask the levels c above them of that axis.
        [[maybe_unused]] const int ax_up = (a_lp - g + 2 * D * G) % D;
        [[maybe_unused]] T qv = T(0), pp = T(0);
        [[maybe_unused]] uint32_t ax_mask = 0;
        if constexpr (!kLower) {
            qv = ax_get(q, g < D ? g : 0);
            pp = qv;
            ax_mask = axis_levels<D>(ax_up);
        }
        // Level L - 1 - c is bit c, lane c of batch 0: far_c, the levels entered through their far child.
        uint32_t far_c = 0;
        int32_t node = 0;
        int level = 0;
        // Lanes past the path's levels (and with them the last lane when L < G) take the leaf's own box.
        const int own_sh = g < L ? g : 0, own_xor = g < L ? 1 : 0;
        // Box distances of the far sides on the path, batch b holding the levels c = b*G .. b*G + G - 1, one
        // a lane.  With kKeep they are kept for the levels above the one last entered, where they still
        // hold: batch 0 renews its lanes below `renew`, a later batch is renewed whole, when it is next
        // needed, if its bit in `stale` is set.  For the 64-byte boxes of d = 8, whose loads (a line per
        // lane) bound the search (500K queries, k = 32: 23.2 -> 19.0 ms); at d <= 3 the bookkeeping costs more
        // than the loads (depth-13 tree, k = 8, 1M queries: 0.58 -> 0.63 ms).
        constexpr bool kKeep = D > 3;
        constexpr int NB = (kMaxLevels + G - 1) / G;
        T tb[kKeep ? NB : 1];
#pragma unroll
        for (int b = 0; b < (kKeep ? NB : 1); ++b) tb[b] = T(0);
        [[maybe_unused]] int renew = G;
        [[maybe_unused]] uint32_t stale = ~0u;
        wave_lds_sync();

        // Candidates of the records [c0, min(c0 + CH, end)): distances tested against the worst
        // at the chunk's start, then inserted in scan order (knn_tree.hpp's two-pass scan).
        auto chunk = [&](int32_t c0, int32_t end) {
            Rec<T, D> rec[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // (at most G - 1 records past the last point)
                const int32_t s = c0 + u * G < end ? c0 + u * G + g : c0 + g;
                rec[u] = load_rec<T, D>(tv.recs, s);
            }
            __builtin_amdgcn_sched_barrier(0);
            uint32_t mask = 0;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const T dd = sq_dist<T, D>(q, rec[u].c);
                bool acc = dd < w;
                if constexpr (kLower) {
                    const int32_t s = c0 + u * G + g;
                    const int32_t o = RecLayout<T, D>::kHasIdx ? rec[u].o : load_i32_at(tv.shuffled, min(s, end - 1));
                    acc = acc || (dd == w && o < wx);
                    st_o[u * G + g] = o;
                }
                mask |= group_ballot<G>(acc, base) << (u * G);
                st_d[u * G + g] = dd;
            }
            const int n = end - c0;  // only the leaf's records
            mask &= n >= 32 ? ~0u : (1u << n) - 1u;
            if (mask) {
                wave_lds_sync();
                int j = __builtin_ctz(mask);
                T dj = st_d[j];
                int32_t oj = kLower ? st_o[j] : 0;
                for (;;) {
                    // (the next candidate is read while this one is inserted)
                    mask &= mask - 1u;
                    const int jn = mask ? __builtin_ctz(mask) : j;
                    const T dn = st_d[jn];
                    const int32_t on = kLower ? st_o[jn] : 0;
                    kb.insert(dj, kLower ? oj : c0 + j, g);
                    if (!mask) break;
                    j = jn;
                    dj = dn;
                    oj = on;
                }
                w = group_lane<G, G - 1>(kb.d[E - 1]);
                if constexpr (kLower) wx = group_lane<G, G - 1>(kb.x[E - 1]);
            }
            wave_lds_sync();
        };
        auto passes = [&](T b) { return kLower ? lower_passes(b, w) : b < w; };
        auto scan = [&](int32_t leaf, int32_t beg, int32_t end) {
            if constexpr (kGroups) {
                // the boxes of G record runs at a time; a run is scanned while its box passes
                const int32_t gb = tv.group_base[leaf];
                const int32_t nr = (end - beg + kGroupRecs - 1) / kGroupRecs;
                for (int32_t r0 = 0; r0 < nr; r0 += G) {
                    const T b = aabb_bound<T, D>(tv.group_boxes, gb + min(r0 + g, nr - 1), q);
                    uint32_t left = nr - r0 >= G ? ((1u << G) - 1u) : ((1u << (nr - r0)) - 1u);
                    for (;;) {
                        const uint32_t m = group_ballot<G>(passes(b), base) & left;
                        if (!m) break;
                        const int j = __builtin_ctz(m);
                        left &= ~((2u << j) - 1u);
                        const int32_t c0 = beg + (r0 + j) * kGroupRecs;
                        const int32_t ce = min(end, c0 + kGroupRecs);
                        for (int32_t c = c0; c < ce; c += CH) chunk(c, ce);
                    }
                }
            } else {
                for (int32_t c0 = beg; c0 < end; c0 += CH) chunk(c0, end);
            }
        };
        for (;;) {
            // down the near path to a leaf, S levels per round
            while (level < L) {
                // (lanes of levels past the last read a split value that no step uses)
                const int32_t sub = min(((node + 1) << r) + (off - 1), tv.n_nodes - 1);
                const T m = load_at(tv.split, sub);
                const uint32_t ge = ~group_ballot<G>(s_qg[level + r] < m, base);
                uint32_t idx = 1;
#pragma unroll
                for (int s = 0; s < S; ++s) idx = 2 * idx + ((ge >> idx) & 1u);
                const int steps = min(S, L - level);
                idx >>= S - steps;
                node = (int32_t)(((uint32_t)node << steps) + idx) - 1;
                level += steps;
            }
            const int32_t child1 = node + 1;  // 1-based
            const int32_t lp = (child1 >> 1) - 1;
            const int32_t left_leaf = 2 * lp + 1 - tv.n_nodes;
            const int32_t o0 = load_at(tv.leaf_off, left_leaf), o1 = load_at(tv.leaf_off, left_leaf + 1),
                          o2 = load_at(tv.leaf_off, left_leaf + 2);
            const bool right = child1 & 1;
            [[maybe_unused]] const T m_lp = kLower ? T(0) : load_at(tv.split, lp);
            if (!kKeep || g < renew || g >= L)
                tb[0] = node_box_dist<T, D>(tv.boxes, ((child1 >> own_sh) ^ own_xor) - 1, q);
            const uint32_t levels_here = L < G ? (1u << L) - 1u : (1u << G) - 1u;
            uint32_t near = ~far_c & levels_here;
            bool own;
            if (L < G)
                own = (group_ballot<G>(passes(tb[0]), base) >> (G - 1)) & 1u;
            else
                own = passes(node_box_dist<T, D>(tv.boxes, node, q));
            if (own) scan(left_leaf + (right ? 1 : 0), right ? o1 : o0, right ? o2 : o1);
            uint32_t hit = group_ballot<G>(passes(tb[0]), base) & near;
            // The sibling leaf: there the reference's bound (v = pp - q, v[a] += m - pp[a] on the
            // leaf-parents' axis a) rounds differently from the box distance.
            bool looks = hit & 1u;
            if constexpr (!kLower) {
                if (looks) {
                    T v = pp - qv;
                    v = ax_up == 0 ? v + (m_lp - pp) : v;
                    v = v * v;
                    looks = group_sum<G, D>(v, group_lane<G, 0>(v)) < w;
                }
            }
            if (looks) {
                scan(left_leaf + (right ? 0 : 1), right ? o0 : o1, right ? o1 : o2);
                hit = group_ballot<G>(passes(tb[0]), base) & near;
            }
            hit &= ~1u;
            int cb = 0;  // first level of the batch that hit
            const auto later_batch = [&](T& t, bool renew_it) {
                const int c = g + cb;
                if (renew_it) t = node_box_dist<T, D>(tv.boxes, (c < L ? (child1 >> c) ^ 1 : child1) - 1, q);
                hit = group_ballot<G>(passes(t), base) & ~(far_c >> cb);
                if (L < cb + G) hit &= (1u << (L - cb)) - 1u;
            };
            if constexpr (kKeep) {
#pragma unroll
                for (int b = 1; b < NB; ++b) {
                    if (!hit && L > b * G) {
                        cb = b * G;
                        later_batch(tb[b], (stale >> b) & 1u);
                        stale &= ~(1u << b);
                    }
                }
            } else {
                while (!hit && L > cb + G) {
                    T t;
                    cb += G;
                    later_batch(t, true);
                }
            }
            if (!hit) break;
            // enter the far side of the deepest level that passes
            const int c = __builtin_ctz(hit) + cb;
            const int32_t child = child1 >> c;  // 1-based, on the path below that level
            if constexpr (!kLower) {
                // the c levels left reset pp on their axes, the entered one sets its own
                const T m = load_at(tv.split, (child >> 1) - 1);
                pp = ax_up < c ? qv : pp;
                pp = (ax_mask >> c) & 1u ? m : pp;
            }
            far_c = (far_c & ~((2u << c) - 1u)) | (1u << c);
            if constexpr (kKeep) {
                renew = c;
                stale |= (1u << ((c + G - 1) / G)) - 1u;  // the batches that hold a level below c
            }
            node = (child ^ 1) - 1;
            level = L - c;
        }
    }

    // output: lane g holds entries g*E .. of the row
    const int32_t* map = kLower ? tv.inv_shuffled : tv.shuffled;
    int32_t mo[E];
#pragma unroll
    for (int e = 0; e < E; ++e) mo[e] = load_i32_at(map, max(kb.x[e], 0));
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int p = g * E + e - pad;
        if (p >= 0) {
            out_d[qi * k + p] = kb.d[e];
            out_i[qi * k + p] = kLower ? mo[e] : kb.x[e];
            if (out_o) out_o[qi * k + p] = (int64_t)(kLower ? kb.x[e] : mo[e]);
        }
    }
}

template <typename T, int D, int G, int E>
void launch_group(const TreeView<T>& tv, const T* q, int64_t nq, const int32_t* order, int k, T* dist, int32_t* idx,
                  int64_t* orig, bool lower, hipStream_t s) {
    constexpr int kQueries = kGroupBlock / G;
    const dim3 grid((unsigned)((nq + kQueries - 1) / kQueries)), block(kGroupBlock);
#define TK_GROUP(LOWER, BOXES) \
    hipLaunchKernelGGL((knn_group_kernel<T, D, G, E, LOWER, BOXES>), grid, block, 0, s, tv, q, nq, order, k, dist, idx, orig)
    if (lower) {
        if (tv.group_boxes) TK_GROUP(true, true);
        else TK_GROUP(true, false);
    } else {
        if (tv.group_boxes) TK_GROUP(false, true);
        else TK_GROUP(false, false);
    }
#undef TK_GROUP
    TK_HIP_CHECK(hipGetLastError());
}

// The prebuilt groups: 16 lanes for every list up to 128 entries; 8 and 4 lanes at d <= 3 for lists of
// 2 entries a lane.  search_lanes asks for no other.
template <typename T, int D>
void launch_group_d(const TreeView<T>& tv, const T* q, int64_t nq, const int32_t* order, int k, T* dist, int32_t* idx,
                    int64_t* orig, bool lower, int lanes, hipStream_t s) {
    if constexpr (D <= 3) {
        if (lanes == 4 && k <= 4) return launch_group<T, D, 4, 1>(tv, q, nq, order, k, dist, idx, orig, lower, s);
        if (lanes == 4 && k <= 8) return launch_group<T, D, 4, 2>(tv, q, nq, order, k, dist, idx, orig, lower, s);
        if (lanes == 8 && k <= 8) return launch_group<T, D, 8, 1>(tv, q, nq, order, k, dist, idx, orig, lower, s);
        if (lanes == 8 && k <= 16) return launch_group<T, D, 8, 2>(tv, q, nq, order, k, dist, idx, orig, lower, s);
    }
    if (k <= 16) return launch_group<T, D, 16, 1>(tv, q, nq, order, k, dist, idx, orig, lower, s);
    if (k <= 32) return launch_group<T, D, 16, 2>(tv, q, nq, order, k, dist, idx, orig, lower, s);
    if (k <= 64) return launch_group<T, D, 16, 4>(tv, q, nq, order, k, dist, idx, orig, lower, s);
    if (k <= 128) return launch_group<T, D, 16, 8>(tv, q, nq, order, k, dist, idx, orig, lower, s);
    throw std::runtime_error("list of more than 128 entries in a group search");
}

template <typename T>
void launch_group_search_t(const Tree& t, const T* q, int64_t nq, const int32_t* order, int k, T* dist, int32_t* idx,
                           int64_t* orig, bool lower, int lanes, hipStream_t s) {
    const TreeView<T> tv = tree_view<T>(t);
    switch (t.dims) {
        case 1: launch_group_d<T, 1>(tv, q, nq, order, k, dist, idx, orig, lower, lanes, s); break;
        case 2: launch_group_d<T, 2>(tv, q, nq, order, k, dist, idx, orig, lower, lanes, s); break;
        case 3: launch_group_d<T, 3>(tv, q, nq, order, k, dist, idx, orig, lower, lanes, s); break;
        case 8: launch_group_d<T, 8>(tv, q, nq, order, k, dist, idx, orig, lower, lanes, s); break;
        default: throw std::runtime_error("unsupported dims");
    }
}

}  // namespace tk
