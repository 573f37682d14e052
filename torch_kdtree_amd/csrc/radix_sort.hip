// Stable least-significant-digit radix sort of (uint32 key, uint32 value) pairs, 8 bits per pass.
//
// Up to kSmallItems pairs: one workgroup runs every pass in LDS (one launch).  Up to kLookBackMax:
//   1. radix_count_kernel reads the keys once and counts the digits of every pass, per workgroup;
//   2. one look-back radix_pass_kernel per pass.  Workgroups take tiles of pairs by a ticket, rank
//      their tile, publish its digit counts and find the pairs of each digit in all earlier
//      tiles by looking back over the earlier tiles' published counts (each tile publishes first its
//      own counts, then the sum up to and including it), so a pass is one launch: the single-pass scan of
//      D. Merrill and M. Garland, "Single-pass parallel prefix scan with decoupled look-back", 2016.
// More, per pass:
//   1. radix_hist_kernel counts the digits of every tile;
//   2. radix_scan_kernel scans the counts of each digit over the tiles;
//   3. radix_pass_kernel ranks the tiles and writes them out.
// In a pass every wavefront ranks its quarter of the tile in index order, 64 pairs per round (lanes
// holding the same digit are found with one ballot per digit bit; per-digit running counts live in
// the wavefront's own LDS row).  The tile, rearranged by digit in LDS, is written out slot by slot:
// each digit's run goes to consecutive output positions.  Equal digits keep the input order: the
// sort is stable, and the result does not depend on scheduling.
//
// The look-back ends: a tile's ticket is taken by a workgroup that is already running, which waits
// only for smaller tickets.  A status word holds its flag and its count together, so relaxed
// agent-scope atomics suffice (the XCDs' L2s are not coherent for plain accesses).
// Nothing is cleared with a memset and nothing waits on the host, so the sort can be captured in
// a HIP graph and replayed: radix_count_kernel clears the first pass's status words and the tickets,
// and each pass clears the status words of the next.
//
// Bound: small sorts by the launches (about 4.6 us each), large ones by the passes' memory traffic (8M
// pairs: 47 us to rank and write, 2.9 TB/s, and 14 to count).  The look-back costs a pass more the more tiles are in
// flight (each step back is a load past the L2), which from 512K pairs is more than the two launches it saves.
// Look-back with tiles of 4,096 pairs / three launches, us: 600K pairs of 8 / 24 bits 32 / 31, 62 / 59; 1M 33 / 29,
// 69 / 60; 2M 45 / 30, 96 / 73.  Against a three-kernel scan per pass (five launches a pass): 4,096 pairs of 24-bit
// keys 57 -> 19 us, 65,537 74 -> 37, 1M 87 -> 60, 2M 100 -> 73, 8M of 20 bits 207 -> 178, 16M of 24 bits 414 -> 367.
#include <algorithm>

#include "gpu_common.hpp"
#include "knn_gpu.hpp"

namespace tk {
namespace {

constexpr int kRadixBlock = 256;
constexpr int kRadixItems = 16;  // pairs per thread of a tile, three launches a pass
// Look-back sorts take smaller tiles: 4,096 pairs a tile would leave CUs idle (65,537 pairs 47 -> 37 us, 500K of 32
// bits 78 -> 73).
constexpr int kRadixItemsFew = 8;
constexpr int kRadixTile = kRadixBlock * kRadixItems;
constexpr int kRadixTileFew = kRadixBlock * kRadixItemsFew;
constexpr int64_t kLookBackMax = int64_t(512) << 10;
constexpr int kRadixBins = 256;
constexpr int kMaxPasses = 4;
constexpr int kDirectParts = 32;   // up to this many, the pass kernels sum the workgroups' counts themselves

constexpr int kSmallBlock = 512;
constexpr int kSmallRounds = 8;
constexpr int kSmallItems = kSmallBlock * kSmallRounds;

// Status word of a (tile, digit): the flag above the count (counts < 2^30: n <= 2^28).
constexpr uint32_t kHasCount = 1u << 30;  // the tile's own count
constexpr uint32_t kHasSum = 2u << 30;    // the sum over all tiles up to and including it
constexpr uint32_t kCountMask = (1u << 30) - 1u;

__device__ __forceinline__ uint32_t status_load(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void status_store(uint32_t* p, uint32_t v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Adds one to cnt[dg] for every active lane.  Neighbouring keys often share their high digits: a digit
// that all lanes share is added by one of them.
__device__ __forceinline__ void count_digit(int32_t* cnt, uint32_t dg) {
    const uint32_t f = __builtin_amdgcn_readfirstlane(dg);
    const uint64_t same = __ballot(dg == f), active = __ballot(true);
    if (same != active)
        atomicAdd(&cnt[dg], 1);
    else if ((active & ((1ull << (threadIdx.x & 63)) - 1ull)) == 0)
        atomicAdd(&cnt[f], (int32_t)__popcll(same));
}

// Ranks a wavefront's kRounds * 64 pairs, starting at pair `base` of n, by the 8-bit digit at `shift`:
// rank[s] = pairs of the same digit before this lane's pair of round s; cnt[256], this wavefront's
// own LDS row (zeroed), ends as its digit counts.  One wavefront's LDS accesses take effect in
// program order, so the running counts need no barrier.
template <int kRounds>
__device__ __forceinline__ void rank_pairs(const uint32_t (&key)[kRounds], int64_t base, int64_t n, int shift, int lane,
                                           int32_t* cnt, int32_t (&rank)[kRounds]) {
    const uint64_t lower_lanes = (1ull << lane) - 1ull;
#pragma unroll
    for (int s = 0; s < kRounds; ++s) {
        const bool valid = base + (int64_t)s * 64 + lane < n;
        // invalid slots get digit 256, a group of their own
        const int dg = valid ? (int)((key[s] >> shift) & (kRadixBins - 1)) : kRadixBins;
        uint64_t same = ~0ull;
#pragma unroll
        for (int b = 0; b < 9; ++b) {
            const bool bit = (dg >> b) & 1;
            const uint64_t bal = __ballot(bit);
            same &= bit ? bal : ~bal;
        }
        const int r = __popcll(same & lower_lanes);
        const int prev = valid ? cnt[dg] : 0;
        rank[s] = prev + r;
        if (valid && (same >> lane) == 1ull) cnt[dg] = prev + r + 1;
    }
}

// Exclusive scan of one value per thread over the first 256 threads (4 wavefronts); tmp[4] in LDS.
// Every thread of the workgroup calls it; returns the scan in threads 0..255.
__device__ __forceinline__ int32_t scan_256(int32_t c, int32_t* tmp) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int32_t inc = c;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int32_t y = __shfl_up(inc, off, 64);
        if (lane >= off) inc += y;
    }
    if (w < 4 && lane == 63) tmp[w] = inc;
    __syncthreads();
    int32_t base = 0;
    for (int v = 0; v < min(w, 4); ++v) base += tmp[v];
    return base + inc - c;
}

// Digit counts of all passes, per workgroup (one tile each): part[block][pass][digit].  Also clears the tickets and
// the first pass's status words.
template <int P>
__global__ __launch_bounds__(kRadixBlock) void radix_count_kernel(const uint32_t* __restrict__ keys, int64_t n,
                                                                  uint32_t* __restrict__ part,
                                                                  uint32_t* __restrict__ tickets,
                                                                  uint32_t* __restrict__ status) {
    constexpr int kWaves = kRadixBlock / 64;
    __shared__ int32_t cnt[kWaves][P][kRadixBins];
    const int t = threadIdx.x, w = t >> 6;
#pragma unroll
    for (int p = 0; p < P; ++p)
        for (int v = 0; v < kWaves; ++v) cnt[v][p][t] = 0;
    if (blockIdx.x == 0 && t < kMaxPasses) tickets[t] = 0;
    __syncthreads();
    status[(int64_t)blockIdx.x * kRadixBins + t] = 0;
    const int64_t base = (int64_t)blockIdx.x * kRadixTileFew;
    uint32_t k[kRadixItemsFew];
#pragma unroll
    for (int s = 0; s < kRadixItemsFew; ++s) {
        const int64_t i = base + (int64_t)s * kRadixBlock + t;
        k[s] = i < n ? keys[i] : 0u;
    }
#pragma unroll
    for (int s = 0; s < kRadixItemsFew; ++s) {
        if (base + (int64_t)s * kRadixBlock + t < n) {
#pragma unroll
            for (int p = 0; p < P; ++p) count_digit(cnt[w][p], (k[s] >> (8 * p)) & (kRadixBins - 1));
        }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < P; ++p) {
        int32_t c = 0;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) c += cnt[v][p][t];
        part[((int64_t)blockIdx.x * P + p) * kRadixBins + t] = (uint32_t)c;
    }
}

// base[pass][digit]: the pairs of smaller digits, over all count workgroups.  One workgroup per pass.
constexpr int kBaseBlock = 1024;
__global__ __launch_bounds__(kBaseBlock) void radix_base_kernel(const uint32_t* __restrict__ part, int32_t n_parts,
                                                                int passes, uint32_t* __restrict__ base) {
    constexpr int kSplit = kBaseBlock / kRadixBins;
    __shared__ int32_t sum[kSplit][kRadixBins];
    __shared__ int32_t tmp[4];
    const int t = threadIdx.x, d = t & (kRadixBins - 1), q = t / kRadixBins, p = blockIdx.x;
    int32_t c = 0;
#pragma unroll 8
    for (int32_t b = q; b < n_parts; b += kSplit) c += (int32_t)part[((int64_t)b * passes + p) * kRadixBins + d];
    sum[q][d] = c;
    __syncthreads();
    c = 0;
    if (t < kRadixBins)
        for (int v = 0; v < kSplit; ++v) c += sum[v][t];
    const int32_t e = scan_256(c, tmp);
    if (t < kRadixBins) base[p * kRadixBins + t] = (uint32_t)e;
}

// Digit counts of every tile: hist[digit][tile].
__global__ __launch_bounds__(kRadixBlock) void radix_hist_kernel(const uint32_t* __restrict__ keys, int64_t n, int shift,
                                                                 int32_t n_tiles, uint32_t* __restrict__ hist) {
    constexpr int kWaves = kRadixBlock / 64;
    __shared__ int32_t cnt[kWaves][kRadixBins];
    const int t = threadIdx.x, w = t >> 6;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) cnt[v][t] = 0;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * kRadixTile;
    uint32_t k[kRadixItems];
#pragma unroll
    for (int s = 0; s < kRadixItems; ++s) {
        const int64_t i = base + (int64_t)s * kRadixBlock + t;
        k[s] = i < n ? keys[i] : 0u;
    }
#pragma unroll
    for (int s = 0; s < kRadixItems; ++s)
        if (base + (int64_t)s * kRadixBlock + t < n) count_digit(cnt[w], (k[s] >> shift) & (kRadixBins - 1));
    __syncthreads();
    int32_t c = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) c += cnt[v][t];
    hist[(int64_t)t * n_tiles + blockIdx.x] = (uint32_t)c;
}

// Row `digit` of hist scanned over the tiles (exclusive, in place); total[digit] = its sum.
constexpr int kScanBlock = 1024;
__global__ __launch_bounds__(kScanBlock) void radix_scan_kernel(uint32_t* __restrict__ hist, int32_t n_tiles,
                                                                uint32_t* __restrict__ total) {
    constexpr int kWaves = kScanBlock / 64;
    __shared__ uint32_t wsum[kWaves];
    uint32_t* row = hist + (int64_t)blockIdx.x * n_tiles;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    uint32_t carry = 0;
    for (int32_t b = 0; b < n_tiles; b += kScanBlock) {
        const uint32_t c = b + t < n_tiles ? row[b + t] : 0u;
        uint32_t inc = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t y = __shfl_up(inc, off, 64);
            if (lane >= off) inc += y;
        }
        if (lane == 63) wsum[w] = inc;
        __syncthreads();
        uint32_t lower = 0, all = 0;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            const uint32_t x = wsum[v];
            lower += v < w ? x : 0u;
            all += x;
        }
        if (b + t < n_tiles) row[b + t] = carry + lower + inc - c;
        carry += all;
        __syncthreads();
    }
    if (t == 0) total[blockIdx.x] = carry;
}

// What a pass reads beside its pairs.  With the look-back: the digits' output starts (base), or the
// count workgroups' counts to sum (part: n_parts rows of part_stride values), the ticket and the status
// words of this pass and the next.  Without: the scanned tile counts (hist[digit][tile]) and the totals.
struct PassArgs {
    const uint32_t* base;
    const uint32_t* part;
    int32_t n_parts, part_stride;
    uint32_t *ticket, *status, *status_next;
    const uint32_t *hist, *total;
    int32_t n_tiles;
};

// One pass.  vals_in null: the values are the pairs' indices.
template <bool kLookBack>
__global__ __launch_bounds__(kRadixBlock) void radix_pass_kernel(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, int64_t n, int shift, PassArgs args,
    uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out) {
    constexpr int kWaves = kRadixBlock / 64;
    constexpr int kRounds = kLookBack ? kRadixItemsFew : kRadixItems;
    constexpr int kTile = kRadixBlock * kRounds;
    __shared__ uint32_t tile_k[kTile];           // the tile in digit order (stable)
    __shared__ uint32_t tile_v[kTile];
    __shared__ int32_t tile_start[kRadixBins];        // first tile slot of each digit
    __shared__ int32_t wave_cnt[kWaves][kRadixBins];  // per wavefront: pairs of each digit, then their first slot
    __shared__ int32_t tmp[4];
    __shared__ int32_t blk_off[kRadixBins];  // this tile's output start of each digit, less its tile slot
    __shared__ uint32_t s_tile;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    if (kLookBack && t == 0) s_tile = atomicAdd(args.ticket, 1u);
#pragma unroll
    for (int v = 0; v < kWaves; ++v) wave_cnt[v][t] = 0;
    __syncthreads();
    const int64_t tile = kLookBack ? (int64_t)s_tile : (int64_t)blockIdx.x;
    // output start of digit t (of the pairs of smaller digits) and its pairs in earlier tiles
    uint32_t total = 0, before = 0;
    if constexpr (kLookBack) {
        args.status_next[tile * kRadixBins + t] = 0;
        if (args.part) {
#pragma unroll 8
            for (int32_t b = 0; b < args.n_parts; ++b) total += args.part[(int64_t)b * args.part_stride + t];
        }
    } else {
        total = args.total[t];
        before = args.hist[(int64_t)t * args.n_tiles + tile];
    }
    const int64_t base = tile * kTile + (int64_t)w * kRounds * 64;
    uint32_t key[kRounds], val[kRounds];
    int32_t rank[kRounds];
#pragma unroll
    for (int s = 0; s < kRounds; ++s) {
        const int64_t i = base + (int64_t)s * 64 + lane;
        key[s] = i < n ? keys_in[i] : 0u;
        val[s] = i < n ? (vals_in ? vals_in[i] : (uint32_t)i) : 0u;
    }
    rank_pairs<kRounds>(key, base, n, shift, lane, wave_cnt[w], rank);
    __syncthreads();
    int32_t c = 0;
#pragma unroll
    for (int v = 0; v < kWaves; ++v) c += wave_cnt[v][t];
    uint32_t* const mine = kLookBack ? args.status + tile * kRadixBins + t : nullptr;
    if constexpr (kLookBack) status_store(mine, (tile == 0 ? kHasSum : kHasCount) | (uint32_t)c);
    uint32_t start;
    if (kLookBack && args.base) {
        start = args.base[t];
    } else {
        start = (uint32_t)scan_256((int32_t)total, tmp);
        __syncthreads();
    }
    {
        // first slot of each digit, then of each wavefront's pairs of it, the wavefronts in order
        int32_t run = scan_256(c, tmp);
        tile_start[t] = run;
#pragma unroll
        for (int v = 0; v < kWaves; ++v) {
            const int32_t wc = wave_cnt[v][t];
            wave_cnt[v][t] = run;
            run += wc;
        }
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < kRounds; ++s) {
        if (base + (int64_t)s * 64 + lane < n) {
            const int pos = wave_cnt[w][(key[s] >> shift) & (kRadixBins - 1)] + rank[s];
            tile_k[pos] = key[s];
            tile_v[pos] = val[s];
        }
    }
    // the pairs of digit t in all earlier tiles: back over the published counts, four at a time, until
    // a tile that has published the sum up to it
    if (kLookBack && tile > 0) {
        constexpr int kAhead = 4;
        int64_t j = tile - 1;
        for (bool done = false; !done;) {
            uint32_t st[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) st[u] = status_load(args.status + (j - u > 0 ? j - u : 0) * kRadixBins + t);
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (done || !(st[u] & (kHasCount | kHasSum))) break;  // not published yet: read again from there
                before += st[u] & kCountMask;
                done = (st[u] & kHasSum) != 0;  // (tile 0 always publishes a sum)
                --j;
            }
            if (!done) __builtin_amdgcn_s_sleep(1);
        }
        status_store(mine, kHasSum | (before + (uint32_t)c));
    }
    blk_off[t] = (int32_t)(start + before) - tile_start[t];
    __syncthreads();
    // write out in tile order: each digit's slots go to consecutive output positions
    const int n_tile = (int)min((int64_t)kTile, n - tile * kTile);
    for (int x = t; x < n_tile; x += kRadixBlock) {
        const uint32_t k = tile_k[x];
        const int32_t pos = blk_off[(k >> shift) & (kRadixBins - 1)] + x;
        keys_out[pos] = k;
        vals_out[pos] = tile_v[x];
    }
}

// All passes of up to kSmallItems pairs in one workgroup.
__global__ __launch_bounds__(kSmallBlock) void radix_small_kernel(const uint32_t* __restrict__ keys_in,
                                                                  const uint32_t* __restrict__ vals_in, int32_t n,
                                                                  int passes, uint32_t* __restrict__ keys_out,
                                                                  uint32_t* __restrict__ vals_out) {
    constexpr int kWaves = kSmallBlock / 64;
    __shared__ uint32_t tile_k[kSmallItems];
    __shared__ uint32_t tile_v[kSmallItems];
    __shared__ int32_t wave_cnt[kWaves][kRadixBins];
    __shared__ int32_t tmp[4];
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const int base = w * kSmallRounds * 64;
    uint32_t key[kSmallRounds], val[kSmallRounds];
    int32_t rank[kSmallRounds];
#pragma unroll
    for (int s = 0; s < kSmallRounds; ++s) {
        const int i = base + s * 64 + lane;
        key[s] = i < n ? keys_in[i] : 0u;
        val[s] = i < n ? (vals_in ? vals_in[i] : (uint32_t)i) : 0u;
    }
    for (int p = 0; p < passes; ++p) {
        const int shift = 8 * p;
        for (int x = t; x < kWaves * kRadixBins; x += kSmallBlock) (&wave_cnt[0][0])[x] = 0;
        __syncthreads();
        rank_pairs<kSmallRounds>(key, base, n, shift, lane, wave_cnt[w], rank);
        __syncthreads();
        int32_t c = 0;
        if (t < kRadixBins)
            for (int v = 0; v < kWaves; ++v) c += wave_cnt[v][t];
        int32_t run = scan_256(c, tmp);
        if (t < kRadixBins) {
            for (int v = 0; v < kWaves; ++v) {
                const int32_t wc = wave_cnt[v][t];
                wave_cnt[v][t] = run;
                run += wc;
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kSmallRounds; ++s) {
            if (base + s * 64 + lane < n) {
                const int pos = wave_cnt[w][(key[s] >> shift) & (kRadixBins - 1)] + rank[s];
                tile_k[pos] = key[s];
                tile_v[pos] = val[s];
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kSmallRounds; ++s) {
            const int i = base + s * 64 + lane;
            if (i < n) {
                key[s] = tile_k[i];
                val[s] = tile_v[i];
            }
        }
    }
#pragma unroll
    for (int s = 0; s < kSmallRounds; ++s) {
        const int i = base + s * 64 + lane;
        if (i < n) {
            keys_out[i] = key[s];
            vals_out[i] = val[s];
        }
    }
}

__global__ __launch_bounds__(256) void copy_u32_kernel(const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                                                       int64_t n, uint32_t* __restrict__ oa, uint32_t* __restrict__ ob) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) {
        oa[i] = a[i];
        ob[i] = b ? b[i] : (uint32_t)i;
    }
}

inline size_t a256(size_t b) { return (b + 255) & ~size_t(255); }

struct RadixLayout {
    int32_t n_tiles;
    size_t keys_tmp, vals_tmp, part, base, tickets, status[2], total;
};

RadixLayout radix_layout(int64_t n) {
    RadixLayout l{};
    const bool look_back = n <= kLookBackMax;
    const int64_t tile = look_back ? kRadixTileFew : kRadixTile;
    l.n_tiles = (int32_t)std::max<int64_t>(1, (n + tile - 1) / tile);
    size_t off = 0;
    l.keys_tmp = off; off += a256(4 * (size_t)n);
    l.vals_tmp = off; off += a256(4 * (size_t)n);
    l.part = off; off += look_back ? a256(4 * (size_t)l.n_tiles * kMaxPasses * kRadixBins) : 0;
    l.base = off; off += a256(4 * (size_t)kMaxPasses * kRadixBins);  // (without look-back: the digit totals)
    l.tickets = off; off += a256(4 * (size_t)kMaxPasses);
    // (without look-back the tile counts take the place of the first status words)
    l.status[0] = off; off += a256(4 * (size_t)l.n_tiles * kRadixBins);
    l.status[1] = off; off += look_back ? a256(4 * (size_t)l.n_tiles * kRadixBins) : 0;
    l.total = off;
    return l;
}

}  // namespace

// What any sort of up to n pairs takes (the largest sort of a path can take more than the smallest of the
// next, and a workspace taken for n serves smaller sorts too).
size_t radix_sort_workspace(int64_t n) {
    size_t bytes = radix_layout(n).total;
    if (n > kLookBackMax) bytes = std::max(bytes, radix_layout(kLookBackMax).total);
    return bytes;
}

void radix_sort_pairs(const uint32_t* keys_in, const uint32_t* vals_in, uint32_t* keys_out, uint32_t* vals_out,
                      int64_t n, int key_bits, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (n < 0 || n > (int64_t(1) << 28)) throw std::runtime_error("radix sort: n must be in [0, 2^28]");
    if (key_bits < 0 || key_bits > 32) throw std::runtime_error("radix sort: key_bits must be in [0, 32]");
    if (n == 0) return;
    const RadixLayout l = radix_layout(n);
    if (!workspace || workspace_bytes < l.total) throw std::runtime_error("radix sort: workspace too small");
    const int passes = (key_bits + 7) / 8;
    if (n <= kSmallItems) {  // (no passes: a copy)
        hipLaunchKernelGGL(radix_small_kernel, dim3(1), dim3(kSmallBlock), 0, stream, keys_in, vals_in, (int32_t)n,
                           passes, keys_out, vals_out);
        TK_HIP_CHECK(hipGetLastError());
        return;
    }
    unsigned char* ws = static_cast<unsigned char*>(workspace);
    uint32_t* kt = reinterpret_cast<uint32_t*>(ws + l.keys_tmp);
    uint32_t* vt = reinterpret_cast<uint32_t*>(ws + l.vals_tmp);
    uint32_t* part = reinterpret_cast<uint32_t*>(ws + l.part);
    uint32_t* base = reinterpret_cast<uint32_t*>(ws + l.base);
    uint32_t* tickets = reinterpret_cast<uint32_t*>(ws + l.tickets);
    uint32_t* status[2] = {reinterpret_cast<uint32_t*>(ws + l.status[0]), reinterpret_cast<uint32_t*>(ws + l.status[1])};
    const dim3 grid(l.n_tiles), block(kRadixBlock);
    if (passes == 0) {
        hipLaunchKernelGGL(copy_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, keys_in, vals_in,
                           n, keys_out, vals_out);
        TK_HIP_CHECK(hipGetLastError());
        return;
    }
    const bool look_back = n <= kLookBackMax;
    const bool direct = l.n_tiles <= kDirectParts;
    if (look_back) {
#define TK_COUNT(P)                                                                                               \
    case P:                                                                                                       \
        hipLaunchKernelGGL(radix_count_kernel<P>, grid, block, 0, stream, keys_in, n, part, tickets, status[0]);  \
        break;
        switch (passes) {
            TK_COUNT(1)
            TK_COUNT(2)
            TK_COUNT(3)
            TK_COUNT(4)
        }
#undef TK_COUNT
        TK_HIP_CHECK(hipGetLastError());
        if (!direct) {
            hipLaunchKernelGGL(radix_base_kernel, dim3(passes), dim3(kBaseBlock), 0, stream, part, l.n_tiles, passes,
                               base);
            TK_HIP_CHECK(hipGetLastError());
        }
    }
    // the last pass writes the output: alternate so that it does
    const uint32_t* ks = keys_in;
    const uint32_t* vs = vals_in;
    for (int p = 0; p < passes; ++p) {
        const bool to_out = ((passes - 1 - p) % 2) == 0;
        uint32_t* kd = to_out ? keys_out : kt;
        uint32_t* vd = to_out ? vals_out : vt;
        PassArgs args{};
        args.n_tiles = l.n_tiles;
        if (look_back) {
            args.base = direct ? nullptr : base + p * kRadixBins;
            args.part = direct ? part + p * kRadixBins : nullptr;
            args.n_parts = l.n_tiles;
            args.part_stride = passes * kRadixBins;
            args.ticket = tickets + p;
            args.status = status[p & 1];
            args.status_next = status[(p + 1) & 1];
            hipLaunchKernelGGL(radix_pass_kernel<true>, grid, block, 0, stream, ks, vs, n, 8 * p, args, kd, vd);
        } else {
            args.hist = status[0];
            args.total = base;
            hipLaunchKernelGGL(radix_hist_kernel, grid, block, 0, stream, ks, n, 8 * p, l.n_tiles, status[0]);
            hipLaunchKernelGGL(radix_scan_kernel, dim3(kRadixBins), dim3(kScanBlock), 0, stream, status[0], l.n_tiles,
                               base);
            hipLaunchKernelGGL(radix_pass_kernel<false>, grid, block, 0, stream, ks, vs, n, 8 * p, args, kd, vd);
        }
        TK_HIP_CHECK(hipGetLastError());
        ks = kd;
        vs = vd;
    }
}

}  // namespace tk
