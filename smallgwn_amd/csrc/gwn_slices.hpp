// gwn_slices.hpp - batches in launches that HIP accepts: one dimension of a launch holds fewer than 2^32
// work-items, which several lanes per query reach at sizes that one lane per query serves.
#pragma once

#include <cstddef>

namespace gwn {

// Queries per launch with four lanes each: 2^30 work-items.
constexpr std::size_t k_quad_slice = std::size_t(1) << 28;

// launch(first, count) over consecutive slices of at most `slice` of the n queries.
template <class Launch> void for_each_slice(std::size_t n, std::size_t slice, Launch &&launch) {
    for (std::size_t first = 0; first < n; first += slice)
        launch(first, n - first < slice ? n - first : slice);
}

} // namespace gwn
