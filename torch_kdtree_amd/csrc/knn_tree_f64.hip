// float64 instantiations of the traversal and presort kernels.
#include <algorithm>

#include "knn_tree_launch.hpp"

namespace tk {

void launch_tree_search_f64(const Tree& t, const double* q, int64_t nq, const int32_t* order, int k, double* dist,
                            int32_t* idx, int64_t* orig, int tie, hipStream_t s) {
    if (tie != kTieLowerIndex && !(t.finite && t.split_bounds)) {
        launch_exact_search_t<double>(t, q, nq, order, k, dist, idx, orig, s);
        return;
    }
    const int lanes = search_lanes(t, nq, k, tie == kTieLowerIndex);
    if (lanes > 1)
        launch_group_search_f64(t, q, nq, order, k, dist, idx, orig, tie == kTieLowerIndex, lanes, s);
    else
        launch_lane_search_t<double>(t, q, nq, order, k, dist, idx, orig, tie, s);
}

void launch_leaf_bucket_f64(const Tree& t, const double* q, int64_t nq, int shift, uint32_t* key, hipStream_t s) {
    launch_leaf_bucket_t<double>(t, q, nq, shift, key, s);
}

void launch_morton_bucket_f64(const Tree& t, const double* q, int64_t nq, void* box, uint32_t* key, hipStream_t s) {
    launch_morton_bucket_t<double>(t, q, nq, box, key, s);
}

}  // namespace tk
