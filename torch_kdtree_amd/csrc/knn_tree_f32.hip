// float32 instantiations of the traversal and presort kernels.
#include <algorithm>

#include "knn_tree_launch.hpp"

namespace tk {

void launch_tree_search_f32(const Tree& t, const float* q, int64_t nq, const int32_t* order, int k, float* dist,
                            int32_t* idx, int64_t* orig, int tie, hipStream_t s) {
    if (tie != kTieLowerIndex && !(t.finite && t.split_bounds)) {
        launch_exact_search_t<float>(t, q, nq, order, k, dist, idx, orig, s);
        return;
    }
    const int lanes = search_lanes(t, nq, k, tie == kTieLowerIndex);
    if (lanes > 1) {
        launch_group_search_f32(t, q, nq, order, k, dist, idx, orig, tie == kTieLowerIndex, lanes, s);
        return;
    }
    int kb = 1;
    while (kb < k) kb <<= 1;
    // a tuned launch variant, where one is prebuilt (trees without record-group boxes)
    if (t.variant > 0 && t.finite && !t.dev->group_boxes &&
        launch_tree_variant_f32_d3(t, q, nq, order, k, kb, dist, idx, orig, tie == kTieLowerIndex, t.variant, s))
        return;
    launch_lane_search_t<float>(t, q, nq, order, k, dist, idx, orig, tie, s);
}

void launch_leaf_bucket_f32(const Tree& t, const float* q, int64_t nq, int shift, uint32_t* key, hipStream_t s) {
    launch_leaf_bucket_t<float>(t, q, nq, shift, key, s);
}

void launch_morton_bucket_f32(const Tree& t, const float* q, int64_t nq, void* box, uint32_t* key, hipStream_t s) {
    launch_morton_bucket_t<float>(t, q, nq, box, key, s);
}

int morton_bucket_count(int dims) { return morton_buckets(dims); }

}  // namespace tk
