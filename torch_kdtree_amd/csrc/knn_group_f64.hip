// float64 instantiations of the group search (several lanes per query).
#include "knn_group.hpp"

namespace tk {

void launch_group_search_f64(const Tree& t, const double* q, int64_t nq, const int32_t* order, int k, double* dist,
                             int32_t* idx, int64_t* orig, bool lower, int lanes, hipStream_t s) {
    launch_group_search_t<double>(t, q, nq, order, k, dist, idx, orig, lower, lanes, s);
}

}  // namespace tk
