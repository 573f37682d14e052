// float32 instantiations of the group search (several lanes per query).
#include "knn_group.hpp"

namespace tk {

void launch_group_search_f32(const Tree& t, const float* q, int64_t nq, const int32_t* order, int k, float* dist,
                             int32_t* idx, int64_t* orig, bool lower, int lanes, hipStream_t s) {
    launch_group_search_t<float>(t, q, nq, order, k, dist, idx, orig, lower, lanes, s);
}

}  // namespace tk
