// GPU tree upload and the query driver.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <limits>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "knn_gpu.hpp"
#include "knn_tree.hpp"

namespace tk {

// ------------------------------------------------------------------------------------------
// Small helpers
// ------------------------------------------------------------------------------------------
StreamScratch::StreamScratch(size_t bytes, hipStream_t s) : stream(s) {
    if (bytes) TK_HIP_CHECK(hipMallocAsync(&ptr, bytes, s));
}
StreamScratch::~StreamScratch() {
    if (ptr) (void)hipFreeAsync(ptr, stream);
}

DeviceGuard::DeviceGuard(int device) {
    TK_HIP_CHECK(hipGetDevice(&prev));
    if (device >= 0 && device != prev) TK_HIP_CHECK(hipSetDevice(device));
}
DeviceGuard::~DeviceGuard() {
    int cur = -1;
    if (hipGetDevice(&cur) == hipSuccess && cur != prev && prev >= 0) (void)hipSetDevice(prev);
}

namespace {
struct ProfEntry {
    std::string stage;
    hipEvent_t start, stop;
};
std::mutex g_prof_mu;
std::vector<ProfEntry> g_prof;
std::atomic<bool> g_prof_on{false};
}  // namespace

void prof_enable(bool on) { g_prof_on = on; }

void prof_reset() {
    std::lock_guard<std::mutex> lk(g_prof_mu);
    for (auto& e : g_prof) {
        (void)hipEventDestroy(e.start);
        (void)hipEventDestroy(e.stop);
    }
    g_prof.clear();
}

bool prof_read(const char* stage, double* total_ms, int64_t* launches) {
    std::lock_guard<std::mutex> lk(g_prof_mu);
    double ms = 0;
    int64_t n = 0;
    for (auto& e : g_prof) {
        if (e.stage != stage) continue;
        TK_HIP_CHECK(hipEventSynchronize(e.stop));
        float m = 0;
        TK_HIP_CHECK(hipEventElapsedTime(&m, e.start, e.stop));
        ms += m;
        ++n;
    }
    *total_ms = ms;
    *launches = n;
    return n > 0;
}

ProfScope::ProfScope(const char* st, hipStream_t s) {
    if (!g_prof_on) return;
    stage = st;
    stream = s;
    TK_HIP_CHECK(hipEventCreate(&start));
    TK_HIP_CHECK(hipEventRecord(start, s));
}

ProfScope::~ProfScope() {
    if (!start) return;
    hipEvent_t stop = nullptr;
    if (hipEventCreate(&stop) != hipSuccess || hipEventRecord(stop, stream) != hipSuccess) {
        (void)hipEventDestroy(start);
        if (stop) (void)hipEventDestroy(stop);
        return;
    }
    std::lock_guard<std::mutex> lk(g_prof_mu);
    g_prof.push_back(ProfEntry{stage, start, stop});
}

int rec_bytes_for(int dtype, int dims) {
#define TK_RB(TT)                                  \
    switch (dims) {                                \
        case 1: return RecLayout<TT, 1>::kBytes;   \
        case 2: return RecLayout<TT, 2>::kBytes;   \
        case 3: return RecLayout<TT, 3>::kBytes;   \
        case 8: return RecLayout<TT, 8>::kBytes;   \
    }
    if (dtype == kF32) {
        TK_RB(float)
    } else {
        TK_RB(double)
    }
#undef TK_RB
    throw std::runtime_error("unsupported dims");
}

int box_bytes_for(int dtype, int dims) {
#define TK_BB(TT)                                  \
    switch (dims) {                                \
        case 1: return BoxLayout<TT, 1>::kBytes;   \
        case 2: return BoxLayout<TT, 2>::kBytes;   \
        case 3: return BoxLayout<TT, 3>::kBytes;   \
        case 8: return BoxLayout<TT, 8>::kBytes;   \
    }
    if (dtype == kF32) {
        TK_BB(float)
    } else {
        TK_BB(double)
    }
#undef TK_BB
    throw std::runtime_error("unsupported dims");
}

void free_device_tree(Tree& t) noexcept {
    DeviceTree* d = t.dev;
    if (!d) return;
    int prev = -1;
    (void)hipGetDevice(&prev);
    if (d->device >= 0) (void)hipSetDevice(d->device);
    (void)hipFree(d->arena);
    if (prev >= 0) (void)hipSetDevice(prev);
    delete d;
    t.dev = nullptr;
}

namespace {

// Whether exact distance ties look common among the cloud's neighbours, from up to 256 leaves
// spread over the tree and at most 64 points of each: more than one point in 256 with an exact
// duplicate among its leaf's sampled points, or, on some axis, fewer distinct values than half
// the sampled points (lattices, rounded coordinates).  Finite trees only (NaN has no order).
template <typename TT>
bool cloud_ties_often(const Tree& t) {
    const int D = t.dims;
    const TT* pts = reinterpret_cast<const TT*>(t.points.data());
    const int32_t nl = t.n_leaves;
    const int32_t S = std::min<int32_t>(nl, 256);
    std::vector<std::vector<TT>> vals((size_t)D);
    std::vector<int32_t> idx;
    int64_t sampled = 0, dups = 0;
    for (int32_t i = 0; i < S; ++i) {
        const int32_t l = (int32_t)((int64_t)i * nl / S);
        const int32_t b0 = t.leaf_off[(size_t)l];
        const int32_t b1 = std::min(t.leaf_off[(size_t)l + 1], b0 + 64);
        idx.resize((size_t)(b1 - b0));
        for (int32_t s = b0; s < b1; ++s) idx[(size_t)(s - b0)] = s;
        auto less = [&](int32_t a, int32_t b) {
            for (int c = 0; c < D; ++c) {
                const TT x = pts[(size_t)a * D + c], y = pts[(size_t)b * D + c];
                if (x != y) return x < y;
            }
            return false;
        };
        std::sort(idx.begin(), idx.end(), less);
        for (size_t j = 0; j + 1 < idx.size(); ++j) dups += !less(idx[j], idx[j + 1]) ? 1 : 0;
        for (int32_t s = b0; s < b1; ++s)
            for (int c = 0; c < D; ++c) vals[(size_t)c].push_back(pts[(size_t)s * D + c]);
        sampled += b1 - b0;
    }
    if (sampled < 2) return false;
    if (dups * 256 > sampled) return true;
    for (auto& v : vals) {
        std::sort(v.begin(), v.end());
        const int64_t distinct = std::unique(v.begin(), v.end()) - v.begin();
        if (distinct * 2 < sampled) return true;
    }
    return false;
}

}  // namespace

bool tree_wants_groups(const Tree& t) { return (int64_t)t.n_points >= (int64_t)kGroupMinLeaf * t.n_leaves; }

DeviceTree* alloc_device_tree(const Tree& t, int device, int64_t n_group_boxes) {
    std::unique_ptr<DeviceTree> d(new DeviceTree());
    d->device = device;
    d->rec_bytes = rec_bytes_for(t.dtype, t.dims);
    d->box_bytes = box_bytes_for(t.dtype, t.dims);
    const size_t n = (size_t)t.n_points;
    size_t off = 0;
    const auto take = [&](size_t bytes) {
        const size_t at = off;
        off += (bytes + 255) & ~size_t(255);
        return at;
    };
    const size_t split = take((size_t)t.n_nodes * dtype_size(t.dtype));
    // kRecPad zero records after the last point: chunked leaf scans read them and ignore them
    const size_t recs = take((n + kRecPad) * (size_t)d->rec_bytes);
    const size_t leaf_off = take(4 * ((size_t)t.n_leaves + 1));
    const size_t shuffled = take(4 * n), inv = take(4 * n);
    const size_t boxes = take(((size_t)t.n_nodes + (size_t)t.n_leaves) * (size_t)d->box_bytes);
    const size_t gboxes = take(n_group_boxes ? (size_t)n_group_boxes * (size_t)d->box_bytes : 0);
    const size_t gbase = take(n_group_boxes ? 4 * ((size_t)t.n_leaves + 1) : 0);
    TK_HIP_CHECK(hipMalloc(&d->arena, off));
    unsigned char* base = static_cast<unsigned char*>(d->arena);
    d->split = base + split;
    d->recs = base + recs;
    d->leaf_off = reinterpret_cast<int32_t*>(base + leaf_off);
    d->shuffled = reinterpret_cast<int32_t*>(base + shuffled);
    d->inv_shuffled = reinterpret_cast<int32_t*>(base + inv);
    d->boxes = base + boxes;
    if (n_group_boxes) {
        d->group_boxes = base + gboxes;
        d->group_base = reinterpret_cast<int32_t*>(base + gbase);
    }
    return d.release();
}

void upload_tree(Tree& t, int device) {
    ensure_host(t);
    free_device_tree(t);
    t.tie_prone = !t.finite || (t.dtype == kF32 ? cloud_ties_often<float>(t) : cloud_ties_often<double>(t));
    if (device < 0) TK_HIP_CHECK(hipGetDevice(&device));
    DeviceGuard g(device);
    const int rec_bytes = rec_bytes_for(t.dtype, t.dims), box_bytes = box_bytes_for(t.dtype, t.dims);
    const size_t ts = dtype_size(t.dtype);
    const size_t coord_bytes = ts * (size_t)t.dims;
    const size_t n = (size_t)t.n_points;
    // kRecPad zero records after the last point: chunked leaf scans read them and ignore them
    std::vector<unsigned char> recs((n + kRecPad) * (size_t)rec_bytes, 0);
    std::vector<int32_t> inv(n);
    for (size_t s = 0; s < n; ++s) inv[(size_t)t.shuffled[s]] = (int32_t)s;
    const bool rec_idx = (size_t)rec_bytes >= coord_bytes + 4;  // RecLayout::kHasIdx
    for (size_t s = 0; s < n; ++s) {
        unsigned char* r = &recs[s * (size_t)rec_bytes];
        std::memcpy(r, &t.points[s * coord_bytes], coord_bytes);
        if (rec_idx) std::memcpy(r + coord_bytes, &t.shuffled[s], 4);
    }
    // boxes: lo then hi, each padded from dims to box_bytes / (2 * ts) elements
    const size_t n_boxes = (size_t)t.n_nodes + (size_t)t.n_leaves;
    const size_t half = (size_t)box_bytes / 2;
    std::vector<unsigned char> boxes(n_boxes * (size_t)box_bytes, 0);
    for (size_t b = 0; b < n_boxes; ++b) {
        const unsigned char* src = &t.aabb[b * 2 * coord_bytes];
        unsigned char* dst = &boxes[b * (size_t)box_bytes];
        std::memcpy(dst, src, coord_bytes);
        std::memcpy(dst + half, src + coord_bytes, coord_bytes);
    }
    // Group boxes: min / max of each run of kGroupRecs records of a leaf, in the layout of `boxes`.
    // Only for leaves of several groups on average, where skipping a group pays for its test
    // (plain workload, 4M points: at depth 13, 488 points a leaf, the traversal takes 14.0 instead of
    // 20.1 ms; at depth 17, 30 a leaf, no gain), and only for finite trees, which prune with
    // boxes (a NaN coordinate would be dropped by min / max).
    const bool use_groups = t.finite && tree_wants_groups(t);
    std::vector<int32_t> gbase;
    std::vector<unsigned char> gboxes;
    auto group_box = [&](auto tag) {
        using TT = decltype(tag);
        const TT* pts = reinterpret_cast<const TT*>(t.points.data());
        const int D = t.dims;
        for (int32_t l = 0; l < t.n_leaves; ++l) {
            const int32_t b0 = t.leaf_off[(size_t)l], b1 = t.leaf_off[(size_t)l + 1];
            for (int32_t g = 0; g < gbase[(size_t)l + 1] - gbase[(size_t)l]; ++g) {
                TT lo[8], hi[8];
                for (int a = 0; a < D; ++a) {
                    lo[a] = std::numeric_limits<TT>::infinity();
                    hi[a] = -std::numeric_limits<TT>::infinity();
                }
                for (int32_t s = b0 + g * kGroupRecs; s < std::min(b1, b0 + (g + 1) * kGroupRecs); ++s)
                    for (int a = 0; a < D; ++a) {
                        lo[a] = std::min(lo[a], pts[(size_t)s * D + a]);
                        hi[a] = std::max(hi[a], pts[(size_t)s * D + a]);
                    }
                unsigned char* dst = &gboxes[((size_t)gbase[(size_t)l] + g) * (size_t)box_bytes];
                std::memcpy(dst, lo, sizeof(TT) * D);
                std::memcpy(dst + half, hi, sizeof(TT) * D);
            }
        }
    };
    if (use_groups) {
        gbase.assign((size_t)t.n_leaves + 1, 0);
        for (int32_t l = 0; l < t.n_leaves; ++l) {
            const int32_t nl = t.leaf_off[(size_t)l + 1] - t.leaf_off[(size_t)l];
            gbase[(size_t)l + 1] = gbase[(size_t)l] + (nl + kGroupRecs - 1) / kGroupRecs;
        }
        gboxes.assign(std::max<size_t>((size_t)gbase[(size_t)t.n_leaves], 1) * (size_t)box_bytes, 0);
        if (t.dtype == kF32)
            group_box(float());
        else
            group_box(double());
    }
    std::unique_ptr<DeviceTree> d(alloc_device_tree(t, device, use_groups ? (int64_t)(gboxes.size() / box_bytes) : 0));
    try {
        const auto copy = [](void* dst, const void* src, size_t bytes) {
            TK_HIP_CHECK(hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice));
        };
        copy(d->split, t.split.data(), (size_t)t.n_nodes * ts);
        copy(d->recs, recs.data(), recs.size());
        copy(d->leaf_off, t.leaf_off.data(), sizeof(int32_t) * t.leaf_off.size());
        copy(d->shuffled, t.shuffled.data(), sizeof(int32_t) * n);
        copy(d->inv_shuffled, inv.data(), sizeof(int32_t) * n);
        copy(d->boxes, boxes.data(), boxes.size());
        if (use_groups) {
            copy(d->group_boxes, gboxes.data(), gboxes.size());
            copy(d->group_base, gbase.data(), sizeof(int32_t) * gbase.size());
        }
    } catch (...) {
        (void)hipFree(d->arena);
        throw;
    }
    t.dev = d.release();
}

namespace {

// Device-to-host copies that a stream capture elsewhere in the process does not see: on a stream of their own,
// which waits for no other, with this thread's capture mode relaxed meanwhile (a copy on the null stream would
// fail and end the capture).
class QuietCopies {
public:
    QuietCopies() {
        TK_HIP_CHECK(hipThreadExchangeStreamCaptureMode(&mode_));
        const hipError_t e = hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking);
        if (e != hipSuccess) {
            (void)hipThreadExchangeStreamCaptureMode(&mode_);
            TK_HIP_CHECK(e);
        }
    }
    ~QuietCopies() {
        (void)hipStreamSynchronize(stream_);
        (void)hipStreamDestroy(stream_);
        (void)hipThreadExchangeStreamCaptureMode(&mode_);
    }
    QuietCopies(const QuietCopies&) = delete;
    QuietCopies& operator=(const QuietCopies&) = delete;
    void copy(void* dst, const void* src, size_t bytes) {
        TK_HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream_));
        TK_HIP_CHECK(hipStreamSynchronize(stream_));
    }

private:
    hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
    hipStream_t stream_ = nullptr;
};

}  // namespace

void ensure_host(const Tree& ct) {
    if (ct.host_ready.load(std::memory_order_acquire)) return;
    Tree& t = const_cast<Tree&>(ct);  // the host arrays are a cache of the GPU copy
    std::lock_guard<std::mutex> lk(t.host_mu);
    if (t.host_ready.load(std::memory_order_relaxed)) return;
    if (!t.dev) throw std::runtime_error("the tree has neither host arrays nor a GPU copy");
    DeviceGuard g(t.dev->device);
    const size_t n = (size_t)t.n_points, rb = (size_t)t.dev->rec_bytes;
    const size_t coord_bytes = dtype_size(t.dtype) * (size_t)t.dims;
    // The arrays are made beside the tree and moved in whole: finish_tree also sets `finite` and `split_bounds`,
    // which queries on other threads read meanwhile (the GPU build has set them already).
    Tree h;
    h.dtype = t.dtype;
    h.dims = t.dims;
    h.levels = t.levels;
    h.n_points = t.n_points;
    h.n_nodes = t.n_nodes;
    h.n_leaves = t.n_leaves;
    std::vector<unsigned char> recs(n * rb);
    h.split.resize((size_t)t.n_nodes * dtype_size(t.dtype));
    h.leaf_off.resize((size_t)t.n_leaves + 1);
    h.shuffled.resize(n);
    h.points.resize(n * coord_bytes);
    {
        QuietCopies q;
        q.copy(recs.data(), t.dev->recs, recs.size());
        q.copy(h.split.data(), t.dev->split, h.split.size());
        q.copy(h.leaf_off.data(), t.dev->leaf_off, 4 * h.leaf_off.size());
        q.copy(h.shuffled.data(), t.dev->shuffled, 4 * n);
    }
    for (size_t s = 0; s < n; ++s) std::memcpy(&h.points[s * coord_bytes], &recs[s * rb], coord_bytes);
    finish_tree(h);
    t.axis.swap(h.axis);
    t.split.swap(h.split);
    t.leaf_off.swap(h.leaf_off);
    t.points.swap(h.points);
    t.shuffled.swap(h.shuffled);
    t.aabb.swap(h.aabb);
    t.host_ready.store(true, std::memory_order_release);
}

// out[s] = coordinates of record s (words 32-bit words of each record), idx[s] = its original index.  Threads
// stride over the words, of which a tree can hold more than a launch takes threads.
constexpr int64_t kExportBlocks = int64_t(1) << 22;
__global__ __launch_bounds__(256) void export_kernel(const unsigned char* __restrict__ recs, int rec_words, int words,
                                                     const int32_t* __restrict__ shuffled, int64_t n,
                                                     uint32_t* __restrict__ out, int64_t* __restrict__ idx) {
    const int64_t stride = (int64_t)gridDim.x * 256, total = out ? n * words : n;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += stride) {
        if (out) out[i] = reinterpret_cast<const uint32_t*>(recs)[(i / words) * rec_words + i % words];
        if (idx && i < n) idx[i] = shuffled[i];
    }
}

void export_tree_gpu(const Tree& t, void* points, int64_t* shuffled, hipStream_t stream) {
    if (!t.dev) throw std::runtime_error("The tree has no GPU copy (it was built for the CPU)");
    if (!points && !shuffled) return;
    DeviceGuard g(t.dev->device);
    const int words = (int)(dtype_size(t.dtype) * (size_t)t.dims / 4);
    const int64_t total = (int64_t)t.n_points * (points ? words : 1);
    const int64_t blocks = std::min((total + 255) / 256, kExportBlocks);
    hipLaunchKernelGGL(export_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, t.dev->recs,
                       t.dev->rec_bytes / 4, words, t.dev->shuffled, (int64_t)t.n_points,
                       static_cast<uint32_t*>(points), shuffled);
    TK_HIP_CHECK(hipGetLastError());
    // (complete on return, like the getters: the caller may read the arrays on any stream)
    TK_HIP_CHECK(hipStreamSynchronize(stream));
}

// ------------------------------------------------------------------------------------------
// Streaming copy: 16-byte loads and stores, each thread striding over the array.  Its rate is the
// achievable HBM bandwidth the traversal's roofline is quoted against, and a copy of known size
// scales the FETCH_SIZE / WRITE_SIZE counters.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void stream_copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                          int64_t n16) {
    constexpr int kU = 4;  // loads in flight per thread
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n16; i += kU * stride) {
        uint4 v[kU];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (i + u * stride < n16) v[u] = src[i + u * stride];
#pragma unroll
        for (int u = 0; u < kU; ++u)
            if (i + u * stride < n16) dst[i + u * stride] = v[u];
    }
}

void stream_copy_gpu(void* dst, const void* src, size_t bytes, hipStream_t stream) {
    if (bytes % 16 != 0 || (((uintptr_t)dst | (uintptr_t)src) & 15u) != 0)
        throw std::runtime_error("stream copy: 16-byte aligned pointers and a multiple of 16 bytes needed");
    const int64_t n16 = (int64_t)(bytes / 16);
    if (n16 == 0) return;
    const unsigned blocks = (unsigned)std::min<int64_t>((n16 + 255) / 256, 256 * 16);
    hipLaunchKernelGGL(stream_copy_kernel, dim3(blocks), dim3(256), 0, stream, static_cast<const uint4*>(src),
                       static_cast<uint4*>(dst), n16);
    TK_HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------------------------------------------------
// VALU issue probe: 8 independent chains per lane of 32-bit VALU operations (no FMA under
// -ffp-contract=off).  Mode 0: a v_mul_f32 and a v_add_f32 per chain, mode 1: two v_med3_f32 per
// chain (16 VALU instructions per loop iteration); mode 2: a compare, a select and an add per chain
// (v_cmp_gt_f32, v_cndmask_b32, v_add_f32: 24 per iteration), the mix of the searches' list and
// pruning code.  Launched over every CU, mode 0's rate is the issue ceiling of 4-cycle
// instructions (one wave instruction per SIMD every 4 cycles); compares and selects issue faster,
// which mode 2 shows.  The traversal's VALU instruction count is quoted against both.
// ------------------------------------------------------------------------------------------
template <int MODE>
__global__ __launch_bounds__(256) void valu_probe_kernel(float* __restrict__ out, int iters, float a, float b) {
    float x[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = (float)threadIdx.x * 0.001f + (float)i;
    for (int it = 0; it < iters; ++it) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (MODE == 0) {
                x[i] = x[i] * a;
                x[i] = x[i] + b;
            } else if constexpr (MODE == 1) {
                x[i] = __builtin_amdgcn_fmed3f(x[i], a, b);
                x[i] = __builtin_amdgcn_fmed3f(x[i], b, a);
            } else {
                x[i] = x[i] + (x[i] < a ? b : -b);
            }
        }
    }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) s += x[i];
    out[(int64_t)blockIdx.x * 256 + threadIdx.x] = s;
}

int64_t valu_probe_gpu(float* out, int64_t threads, int iters, int mode, hipStream_t stream) {
    if (threads <= 0 || threads % 256 != 0 || threads / 256 > INT32_MAX || iters <= 0)
        throw std::runtime_error("VALU probe: threads must be a positive multiple of 256, iters positive");
    if (mode < 0 || mode > 2) throw std::runtime_error("VALU probe: mode 0 (mul + add), 1 (med3) or 2 (compare + select)");
    const dim3 grid((unsigned)(threads / 256));
    if (mode == 0)
        hipLaunchKernelGGL(valu_probe_kernel<0>, grid, dim3(256), 0, stream, out, iters, 0.999f, 0.001f);
    else if (mode == 1)
        hipLaunchKernelGGL(valu_probe_kernel<1>, grid, dim3(256), 0, stream, out, iters, 0.999f, 0.001f);
    else
        hipLaunchKernelGGL(valu_probe_kernel<2>, grid, dim3(256), 0, stream, out, iters, 0.999f, 0.001f);
    TK_HIP_CHECK(hipGetLastError());
    return threads / 64 * (int64_t)iters * (mode == 2 ? 24 : 16);
}

// ------------------------------------------------------------------------------------------
// Query driver
// ------------------------------------------------------------------------------------------
// Lanes per query, measured on MI355X (whole queries in us or ms; "/" separates the forms, "s" marks one
// with the presort, which one lane always has).
// * k > 32, and d = 8 but on few points: 16 lanes at every size.  One lane's list does not fit its registers (100K
//   queries, k = 100: 0.85 ms; 19.3 ms with one lane's list in LDS), and at d = 8 the walks of 64 lanes part (500K
//   queries, k = 32: 19 ms against 45).
// * few queries leave the chip idle with one lane each, and a search is then one chain of dependent
//   loads, which more lanes shorten.  d = 3, k = 8, 16 / 8 / 4 / 1 lanes: cloud of 100K points, 1,000 queries
//   19 / 25 / 37 / 100 us; 30,000 32 / 31 / 35 / 146; 120,000 84 / 73 / 74 / 176; 300,000 188 / 160 / 150 / 223;
//   600,000 355 / 294 / 274 / 308.  Larger calls, 4s / 1 lanes: 1M 421 / 402 (100K points), 526 / 514 (1M,
//   uniform), 584 / 611 (4M), 611 / 683 (1M on a surface), 624 / 816 (1M, clustered); 2M 1,017 / 886, 1,139 / 1,053,
//   1,109 / 1,051, 1,117 / 1,257 (clustered); 4M 2,238 / 1,789.
// * k = 16: 30,000 41 / 42 / - / 186; 120,000 108 / 111 / - / 219; 300,000 249 / 229 / - / 284.  8s / 1 lanes, 1M:
//   650 / 567, 735 / 717, 838 / 820, 858 / 934, 836 / 1,105; 2M 1,317 / 1,172, 1,568 / 1,375, 1,524 / 1,450, 1,531 / 1,663.
// * k = 32, 16 / 1: 120,000 201 / 344; 300,000 456 / 566; 16s / 1: 600,000 911 / 1,020; 1M 1,419 / 1,503; 2M 2,646 /
//   2,578.
// * d = 1 and 2, 4 / 1: d = 2, k = 8: 300,000 84 / 140; 1M 244 / 231; 2M 468 / 398; k = 4: 1M 194 / 207, 2M 371 / 314.
//   d = 1, 4M: 559 / 629.
// * doubles, a lane's list being twice the registers: k = 16, 16 / 8 / 1: 150,000 302 / 321 / 912; 16s / 8s / 1: 500,000
//   777 / 788 / 1,450; 1.5M 1,937 / 1,890 / 2,428; 2M of a uniform cloud - / 2.11 / 1.96 ms.
// * trees of big leaves (record-group boxes), k <= 8: 4s at every larger size (depth 13, k = 8: 1M of 1M points
//   588 / 658; 4M of 4M points 3.48 / 3.92 ms, 16M 11.7 / 11.9).
// * from some size on one lane is faster, the sooner the shorter the walks (few axes, few points) and the longer
//   the list.  Where the two cross, in thousands of queries (clustered clouds of 1M points in brackets; "l" the
//   lower-index policy):
//     one axis     16 entries 515-595 (595), "l" 350-730 (435);  32: 310-380 (360), "l" 240-320 (280)
//     two axes     8: 635-810 (2,330);  16: 310-540 (1,220), "l" 250-370 (800);  32: 160-325 (890), "l" 160-240
//     three axes   8: 500-910 (3,000);  16: 255-350 below 10K points, 580-850 (1,970) above, "l" 250-480 (1,010);
//                  32: 165-370, 640-1,320 (2,530), "l" 125-340 (800)
//   A list that k does not fill costs one lane more (its rows go out in 4-byte stores): 12 of 16 entries, one axis none
//   up to 3M, two 810 and more, three 470 and more; 24 of 32, one none, two 305-455 (1,500), three 235-475, 880 and more.
//   So does the (distance, index) list, of doubles and of clouds that tie often: doubles "l", 16 and 32, two axes
//   500-520 at 300 points, 1,430 and more above.  Doubles: two axes, 8: 545-820 (1,920), 16: 250-395 (970), 32: 165-360 (1,630);
//   three axes, 16: 220 at 300 points, 830 at 100K, 2,000 at 1M; 32: 165, 1,430, 2,000.
// * big leaves on one axis or two: presorted lanes scan the same records, groups each their own, so the line is a number
//   of records scanned; on few queries one lane each leaves the chip idle, so it is never below the floors.  Best group / 1,
//   (s) presorted: d = 1, 64K points, leaves of 500, k = 1, 100K queries 118 / 116, 300K 253 (s) / 146, k = 32, 300K 677 (s) / 650;
//   1M, leaves of 122, k = 1, 700K 176 / 146, 1.5M 354 (s) / 218; 50K, leaves of 3,125, k = 1, 30K 307 / 356, 60K, k = 8, 565 / 625;
//   d = 2, 64K, leaves of 250, k = 8, 300K 186 (s) / 196, 700K 304 (s) / 263; 50K, leaves of 3,125, k = 8, 100K 464 / 569, "l" 661 /
//   1,934.  f64, d = 1, leaves of 250, k = 1, 30K, 16 / 4 lanes 71 / 34.
// * one pair of leaves (levels 1, no walk; one lane takes no presort): 150 points, d = 1, k = 1, 30K 14.8 / 14.6, 100K 22.3 /
//   15.0; d = 3, k = 8, 60K 23 / 28, 80K 26 / 29, 100K 33 / 29, k = 16, 60K 35 / 41, 100K 50 / 42; d = 1, k = 32, 80K 60 / 84, 300K 190 /
//   161; "l", d = 3, k = 8, 80K 35 / 51, 300K 95 / 64; doubles "l", k = 32, 80K 138 / 278, 300K 450 / 634.
// * leaves of a few points, which a chunk of a group's records exceeds: leaves of 4, d = 3, k = 16, 300K 425 / 416, 700K 897
//   (s) / 705; f64, k = 8, 8 lanes, 300K 530 / 532, 700K 1,105 (s) / 861, k = 16 1,593 (s) / 1,226; leaves of 2, d = 2, k = 32, 100K 218 /
//   257, 300K 620 / 406.
// * doubles on one axis or two, k <= 8, 16 / 8 / 4 / 1 lanes: d = 2, 100K points, k = 4, 120K 54 / 46 / 39 / 95; 1M 379 / 299 /
//   223 / 222; k = 8, 120K 67 / 56 / 49 / 105; 1M 472 / 371 / 290 / 266; d = 1, k = 4, 1M 212 / 162 / 114 / 168.
// * d = 8 on few points: with hundreds of queries a point, presorted neighbours take the same walk and the 64 lanes
//   of a wavefront stay together.  16 / 1 lanes, k = 16: 500 points, 120K 144 / 155, 250K 278 / 236, 1M 1,046 / 743; 2,000 points, 600K
//   1,853 / 1,835, 1M 3,039 / 2,865; 10,000 points, 1M 8.3 / 10.3 ms.  f64: 500 points, 60K 164 / 181, 120K 319 / 235, 1M 2,473 / 1,457;
//   2,000 points, 250K 2,054 / 1,670, 1M 7,987 / 6,240; 10,000 points, 1M 18.4 / 24.6 ms; k = 32 no gain.  "l", 500 points, k = 16, 250K
//   316 / 367, 600K 719 / 581; f64 640 / 646, 1,470 / 1,440.  Lists of one or two entries gain only on fewer points
//   (2,000 points, k = 1, 1M 1.74 / 2.18 ms).
namespace {

constexpr int32_t kFewPoints = 10000, kManyPoints = 500000;

// Queries up to which a group search at d <= 3 and k <= 32 is taken.  keyed: the (distance, index) list; flagged: the
// lower-index policy's list with tie flags, cheaper beside a group's (distance, index) list.
int64_t group_search_to(const Tree& t, int k, bool keyed, bool flagged) {
    const bool f64 = t.dtype == kF64, few = t.n_points < kFewPoints, many = t.n_points >= kManyPoints;
    const bool wide = k > 16, full = k == 16 || k == 32;
    const int d = t.dims;
    if (!f64 && d == 3 && k <= 8 && t.dev && t.dev->group_boxes) return INT64_MAX;
    const int64_t most = f64 ? 1750000 : wide ? 1200000 : 1000000;
    int64_t to;
    if (k <= 8) {
        if (k > 4 && (few ? flagged || (keyed && d > 1) : flagged && d == 2 && !many))
            to = few ? 600000 : 800000;
        else if (d == 1)
            to = f64 ? 1750000 : 4000000;
        else
            to = few || (d == 2 && !(f64 && many)) ? 1000000 : f64 ? 1750000 : 1500000;
    } else if (keyed) {
        to = !full || !(few || d == 1) ? most : d > 1 || f64 ? 1000000 : wide ? 300000 : 600000;
    } else {
        if (d == 1)
            to = wide ? 300000 : 600000;
        else if (d == 2)
            to = wide ? (few ? 165000 : !many ? 320000 : f64 ? most : 900000) : few ? 300000 : !many ? 450000 : 1000000;
        else
            to = few ? (wide ? 200000 : 250000) : wide && !f64 && !many ? 650000 : most;
        if (!full) to = !wide && !f64 ? most : std::min(most, d == 1 ? 3 * to : wide ? to * 3 / 2 : 2 * to);
        if (flagged && (wide || !many)) to = to * 3 / 5;
    }
    const int64_t leaf = t.n_points >> t.levels;  // points of a leaf
    if (leaf < 8) {
        if (f64 && d == 3 && !keyed && k > 2)
            to = std::min<int64_t>(to, 600000);
        else if (d == 1 && k <= 8)
            to = k > 4 ? std::min<int64_t>(to, 1200000) : to;
        else if (k > 8 || (flagged && k > 4))
            to /= 2;
    }
    if (d <= 2 && leaf >= 32) {
        const bool listed = keyed || flagged;
        const int64_t scans = !many ? (k <= 8 ? 60000000 : 40000000) : d == 1 || (listed && k > 8) ? 80000000 : 175000000;
        const int64_t least = d == 1 ? (k > 1 ? 75000 : f64 ? 24000 : 45000) : listed && k > 4 ? 250000 : 150000;
        to = std::min(to, std::max(least, scans / leaf));
    }
    return to;
}

}  // namespace

int search_lanes(const Tree& t, int64_t nq, int k, bool lower) {
    const auto prebuilt = [&](int lanes) {
        return lanes == 16 || (lanes == 1 ? k <= 32 : t.dims <= 3 && (lanes == 4 ? k <= 8 : k <= 16));
    };
    if (t.lanes && prebuilt(t.lanes)) return t.lanes;
    if (k > 32) return 16;
    const bool f64 = t.dtype == kF64, few = t.n_points < kFewPoints, many = t.n_points >= kManyPoints;
    if (t.dims == 8) {
        const int32_t points = k <= (f64 && !lower ? 2 : 4) ? 1000 : 5000;
        const int64_t a_point = f64 ? (lower ? 400 : k > 8 ? 50 : 100) : lower ? 800 : 250;
        return t.n_points < points && (!f64 || k <= 16) && nq > a_point * t.n_points ? 1 : 16;
    }
    if (nq <= 24000) return 16;
    const bool keyed = lower && (f64 || t.lower_keyed());
    if (t.levels == 1 && !(f64 && keyed && k > 4) && nq > (k == 1 ? 24000 : k > 16 || (lower && k > 4) ? 100000 : 70000)) return 1;
    if (nq > group_search_to(t, k, keyed, lower && !keyed)) return 1;
    if (k > 16) return 16;
    const bool deep = f64 && !few && (t.dims == 3 || (t.dims == 2 && many && lower));
    if (deep) return nq <= 500000 ? 16 : k > 8 || nq <= 1000000 || lower || (t.dev && t.dev->group_boxes) ? 8 : 4;
    if (k > 8) return nq <= 60000 ? 16 : 8;
    const bool scanned = t.dims == 1 && (t.n_points >> t.levels) >= 32;
    if (f64) return !scanned && nq <= (few ? 30000 : 60000) ? 16 : 4;
    return t.dims == 3 && nq <= (few ? 100000 : 250000) ? 8 : 4;
}

namespace {

constexpr int64_t kPresortMinQueries = 4096;
constexpr int kMaxBucketBits = 22;

inline size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Queries from which a group search gains more from the presort than the sort costs.  One lane per query
// always needs the order, to keep its wavefront's walks together; groups gain cache hits.  Without / with:
// d = 8, k = 32, 500K queries 27.4 / 23.6 ms, equal at 100K; k = 100, 1M 7.6 / 6.4 ms, equal at 100K; d = 3, k = 8: 600K
// 384 / 365 us (1M points), 274 / 303 (100K points), 1M 618 / 533; k = 16: 300K 276 / 300, 600K 528 / 486; k = 32: 300K
// 515 / 519, 600K 1,003 / 900; doubles, k = 16: 150K 302 / 320, 500K 835 / 777; d = 2, k = 8, 1M 243 / 267, doubles, 100K
// points, k = 4, 1M 223 / 263.  d = 8 on trees of few points, k = 16, without / leaf / curve: 2,000 points, 250K 795 / 861 /
// 855, 1M 2,980 / 3,049 / 2,899 (k = 1: 1,632 / 1,730 / 1,522); 10,000 points, 250K 2,197 / 2,324 / 2,095.
int64_t group_presort_from(const Tree& t, int k) {
    if (t.dims == 8) return t.n_points < kFewPoints ? 750000 : 65536;
    if (k > 32) return 131072;
    if (t.dims <= 2 && k <= 8 && !(t.dtype == kF64 && t.n_points >= kManyPoints)) return INT64_MAX;
    if (t.dtype == kF64) return 400000;
    return k > 16 ? 400000 : k > 8 ? 550000 : 700000;
}

// The presort of a call.  Asked for by name it always runs.  Auto: from kPresortMinQueries queries, and for
// groups from group_presort_from.  The order: the space-filling curve at d <= 3 and, for groups, on trees of
// few points; the near-leaf order at d = 8, where the curve over a 3-bit-per-axis grid groups queries more
// coarsely.
int presort_mode(const Tree& t, int64_t nq, int k, const QueryOpts& o) {
    if (nq <= 0) return kPresortOff;
    if (o.presort == kPresortAuto) {
        if (nq < kPresortMinQueries || t.levels <= 1) return kPresortOff;
        const bool exact = o.tie != kTieLowerIndex && !(t.finite && t.split_bounds);
        const bool groups = !exact && search_lanes(t, nq, k, o.tie == kTieLowerIndex) > 1;
        if (groups && nq < group_presort_from(t, k)) return kPresortOff;
        return t.dims == 8 && !(groups && t.n_points < kFewPoints) ? kPresortLeaf : kPresortMorton;
    }
    if (o.presort != kPresortOff && o.presort != kPresortMorton && o.presort != kPresortLeaf)
        throw std::runtime_error("unknown presort mode");
    return o.presort;
}

int bucket_shift(const Tree& t) { return std::max(0, t.levels - kMaxBucketBits); }

struct PresortLayout {
    size_t key, key_s, order, box, radix, radix_bytes, total;
    int key_bits;
};

int bits_for(int64_t n) {
    int b = 1;
    while (b < 32 && (int64_t(1) << b) < n) ++b;
    return b;
}

PresortLayout presort_layout(const Tree& t, int64_t nq, int mode) {
    PresortLayout l{};
    l.key_bits = mode == kPresortMorton ? bits_for(morton_bucket_count(t.dims)) : bits_for(t.n_leaves >> bucket_shift(t));
    size_t off = 0;
    l.key = off; off += align256(sizeof(int32_t) * (size_t)nq);
    l.key_s = off; off += align256(sizeof(int32_t) * (size_t)nq);
    l.order = off; off += align256(sizeof(int32_t) * (size_t)nq);
    l.box = off; off += align256(box_scratch_bytes(t.dims, t.dtype));
    l.radix = off;
    l.radix_bytes = radix_sort_workspace(nq);
    off += align256(l.radix_bytes);
    l.total = off;
    return l;
}

}  // namespace

size_t box_scratch_bytes(int dims, int dtype) { return (size_t)kMaxBoxParts * 2 * (size_t)dims * dtype_size(dtype); }

int canonical_morton_bits(int64_t nq, int dims) {
    int maxb = 0;
    switch (dims) {
        case 1: maxb = MortonBits<1>::kBits; break;
        case 2: maxb = MortonBits<2>::kBits; break;
        case 3: maxb = MortonBits<3>::kBits; break;
        case 8: maxb = MortonBits<8>::kBits; break;
        default: throw std::runtime_error("unsupported dims");
    }
    int b = 0;
    while (b < maxb && (int64_t(8) << ((b + 1) * dims)) <= nq) ++b;
    return b;
}

// Queries are presorted and searched in slices of at most this many: the presort's radix sort orders at most
// 2^28 pairs, and a launch takes fewer than 2^32 threads, of which a group search uses up to 16 a query.  Queries
// are independent, so slicing changes no result.
constexpr int64_t kQuerySlice = int64_t(1) << 27;
static_assert(16 * kQuerySlice + kGroupBlock < (int64_t(1) << 32), "threads of a group search's launch");

size_t query_gpu_workspace(const Tree& t, int64_t nq, const QueryOpts& o) {
    nq = std::min(nq, kQuerySlice);
    // (auto: what a call of this size takes if it presorts, which depends on k; either order takes the same)
    const int mode = o.presort != kPresortAuto                  ? presort_mode(t, nq, 1, o)
                     : nq < kPresortMinQueries || t.levels <= 1 ? kPresortOff
                                                                : kPresortMorton;
    if (mode == kPresortOff) return 0;
    return presort_layout(t, nq, mode).total;
}

void query_gpu(const Tree& t, const void* queries, int64_t nq, int k, void* dist, int32_t* idx, int64_t* orig,
               const QueryOpts& o, hipStream_t stream, void* workspace, size_t workspace_bytes) {
    if (!t.dev) throw std::runtime_error("The tree has no GPU copy (it was built for the CPU)");
    if (k < 1) throw std::runtime_error("nr_nns_searches must be >= 1");
    if (k > t.n_points) throw std::runtime_error("You requested more nearest neighbors than there are in the KD-Tree");
    if (k > kMaxGpuK)
        throw std::runtime_error("nr_nns_searches > " + std::to_string(kMaxGpuK) + " is not supported on the GPU");
    if (o.tie != kTieReference && o.tie != kTieLowerIndex) throw std::runtime_error("unknown tie policy");
    if (nq < 0) throw std::runtime_error("negative query count");
    if (nq == 0) return;
    if (nq >= (int64_t(1) << 31)) throw std::runtime_error("Only 32 bit signed query indexing implemented");
    if (nq > kQuerySlice) {
        const size_t ts = dtype_size(t.dtype);
        for (int64_t s0 = 0; s0 < nq; s0 += kQuerySlice) {
            const int64_t n1 = std::min(kQuerySlice, nq - s0);
            query_gpu(t, static_cast<const unsigned char*>(queries) + (size_t)s0 * t.dims * ts, n1, k,
                      static_cast<unsigned char*>(dist) + (size_t)s0 * k * ts, idx + s0 * k,
                      orig ? orig + s0 * k : nullptr, o, stream, workspace, workspace_bytes);
        }
        return;
    }
    // (a workspace is one for calls of this size, whether or not this k presorts)
    if (workspace && workspace_bytes < query_gpu_workspace(t, nq, o)) throw std::runtime_error("query workspace too small");
    DeviceGuard g(t.dev->device);
    const int32_t* order = nullptr;
    std::unique_ptr<StreamScratch> own;
    const int mode = presort_mode(t, nq, k, o);
    if (mode != kPresortOff) {
        ProfScope ps("presort", stream);
        const PresortLayout l = presort_layout(t, nq, mode);
        unsigned char* ws = static_cast<unsigned char*>(workspace);
        if (!ws) {
            own.reset(new StreamScratch(l.total, stream));
            ws = static_cast<unsigned char*>(own->ptr);
        }
        uint32_t* key = reinterpret_cast<uint32_t*>(ws + l.key);
        uint32_t* key_s = reinterpret_cast<uint32_t*>(ws + l.key_s);
        int32_t* ord = reinterpret_cast<int32_t*>(ws + l.order);
        if (mode == kPresortMorton) {
            if (t.dtype == kF32)
                launch_morton_bucket_f32(t, static_cast<const float*>(queries), nq, ws + l.box, key, stream);
            else
                launch_morton_bucket_f64(t, static_cast<const double*>(queries), nq, ws + l.box, key, stream);
        } else if (t.dtype == kF32) {
            launch_leaf_bucket_f32(t, static_cast<const float*>(queries), nq, bucket_shift(t), key, stream);
        } else {
            launch_leaf_bucket_f64(t, static_cast<const double*>(queries), nq, bucket_shift(t), key, stream);
        }
        radix_sort_pairs(key, nullptr, key_s, reinterpret_cast<uint32_t*>(ord), nq, l.key_bits, ws + l.radix,
                         l.radix_bytes, stream);
        order = ord;
    }
    ProfScope pt("traverse", stream);
    if (t.dtype == kF32)
        launch_tree_search_f32(t, static_cast<const float*>(queries), nq, order, k, static_cast<float*>(dist), idx, orig,
                               o.tie, stream);
    else
        launch_tree_search_f64(t, static_cast<const double*>(queries), nq, order, k, static_cast<double*>(dist), idx,
                               orig, o.tie, stream);
}

// ------------------------------------------------------------------------------------------
// The query that allocates nothing: its presort workspace is a static device array.  `scratch`
// below names the host-side stand-in of that array; the device address of each GPU's copy comes
// from hipGetSymbolAddress, taken once per device on the first call there (with that device
// current), and only that address is ever handed to kernels.
// ------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// The device address of `scratch` on the current device.
void* scratch_on_current_device() {
    int dev = -1;
    TK_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxScratchDevices) throw std::runtime_error("no-allocation query: device out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p)
            throw std::runtime_error(std::string("no-allocation query: hipGetSymbolAddress failed: ") +
                                     hipGetErrorString(e));
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}
}  // namespace

void query_gpu_noalloc(const Tree& t, const void* queries, int64_t nq, int k, void* dist, int32_t* idx, int64_t* orig,
                       const QueryOpts& o, hipStream_t stream) {
    if (!t.dev) throw std::runtime_error("The tree has no GPU copy (it was built for the CPU)");
    if (nq > kNoAllocMaxQueries)
        throw std::runtime_error("no-allocation query: " + std::to_string(nq) + " queries exceed the limit of " +
                                 std::to_string(kNoAllocMaxQueries) + " per call (static scratch of " +
                                 std::to_string(kNoAllocScratchBytes >> 20) + " MiB per GPU)");
    const size_t need = query_gpu_workspace(t, nq, o);
    if (need > kNoAllocScratchBytes) throw std::runtime_error("no-allocation query: workspace exceeds the static scratch");
    DeviceGuard g(t.dev->device);
    void* ws = need ? scratch_on_current_device() : nullptr;
    query_gpu(t, queries, nq, k, dist, idx, orig, o, stream, ws, need ? kNoAllocScratchBytes : 0);
}

}  // namespace tk
