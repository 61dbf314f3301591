// gwn_quad.hpp - four lanes per query: exchange within a quad and a row of 16, and the near-first order of a
// BVH4 node's children, shared by the distance, ray and winding batches.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#pragma clang fp contract(off)

namespace gwn {
namespace {

// Every lane of a quad (lanes 4k..4k+3) receives lane S's value.
template <int S, class T> __device__ inline T quad_bcast(T v) {
    if constexpr (sizeof(T) == 8) {
        std::uint64_t const b = __builtin_bit_cast(std::uint64_t, v);
        std::uint64_t const lo = quad_bcast<S>(static_cast<std::uint32_t>(b));
        std::uint64_t const hi = quad_bcast<S>(static_cast<std::uint32_t>(b >> 32));
        return __builtin_bit_cast(T, (hi << 32) | lo);
    } else {
        return __builtin_bit_cast(
            T, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), S * 0x55, 0xf, 0xf, false));  // quad_perm [S, S, S, S]
    }
}

// The other lane's value: quad_perm [1, 0, 3, 2] and [2, 3, 0, 1].
__device__ inline std::uint32_t quad_swap1(std::uint32_t v) {
    return static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xb1, 0xf, 0xf, false));
}
__device__ inline std::uint32_t quad_swap2(std::uint32_t v) {
    return static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4e, 0xf, 0xf, false));
}
__device__ inline std::uint32_t quad_or(std::uint32_t v) {
    v |= quad_swap1(v);
    return v | quad_swap2(v);
}
__device__ inline float quad_min(float v) {  // no NaN
    v = fminf(v, __uint_as_float(quad_swap1(__float_as_uint(v))));
    return fminf(v, __uint_as_float(quad_swap2(__float_as_uint(v))));
}
__device__ inline std::uint32_t quad_min(std::uint32_t v) {
    v = min(v, quad_swap1(v));
    return min(v, quad_swap2(v));
}

__device__ inline std::uint32_t quad_sum(std::uint32_t v) {
    return quad_bcast<0>(v) + quad_bcast<1>(v) + quad_bcast<2>(v) + quad_bcast<3>(v);
}

// Over the 16 lanes of a row: row_half_mirror joins quads 0-1 and 2-3, row_mirror the two halves.
__device__ inline std::uint32_t row_or(std::uint32_t v) {
    v = quad_or(v);
    v |= static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xf, 0xf, false));
    return v | static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x140, 0xf, 0xf, false));
}
__device__ inline std::uint32_t row_min(std::uint32_t v) {
    v = quad_min(v);
    v = min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xf, 0xf, false)));
    return min(v, static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x140, 0xf, 0xf, false)));
}
__device__ inline std::uint32_t row_sum(std::uint32_t v) {
    v = quad_sum(v);
    v += static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x141, 0xf, 0xf, false));
    return v + static_cast<std::uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x140, 0xf, 0xf, false));
}

// Slot lists of the 16 passing masks: bits 2t..2t+1 hold the t-th slot, the passing ones first, each
// kind in slot order.
constexpr std::uint32_t quad_slots(std::uint32_t mask) {
    std::uint32_t list = 0, t = 0;
    for (int pass = 1; pass >= 0; --pass)
        for (std::uint32_t s = 0; s < 4; ++s)
            if (static_cast<int>((mask >> s) & 1u) == pass)
                list |= s << (2 * t++);
    return list;
}
constexpr std::uint32_t quad_slots4(std::uint32_t first) {
    return quad_slots(first) | (quad_slots(first + 1) << 8) | (quad_slots(first + 2) << 16) | (quad_slots(first + 3) << 24);
}

// By value: through a closure's references the selects became indexed scratch loads.
__device__ inline float pick4(std::uint32_t i, float k0, float k1, float k2, float k3) {
    float const a = i & 1u ? k1 : k0;
    float const b = i & 1u ? k3 : k2;
    return i & 2u ? b : a;
}
__device__ inline void compare_swap(float &a, float &b, std::uint32_t &ia, std::uint32_t &ib) {
    bool const gt = a > b;
    float const ka = gt ? b : a, kb = gt ? a : b;
    std::uint32_t const xa = gt ? ib : ia, xb = gt ? ia : ib;
    a = ka;
    b = kb;
    ia = xa;
    ib = xb;
}

// Position of this lane's slot in the per-lane traversals' near-first order of a node's surviving children
// (those past the survivors are in no order).  `d` is the lane's box distance, `mask` the slots that the
// traversal's compaction keeps (all four where it has none).  Distinct distances have one order; with equal ones (or NaN) anywhere in the wave it
// is that of the compaction in slot order and the five-comparator network, which is not stable, run on
// (distance, slot) pairs.
// `ties`: the wave's lanes that share a distance with another survivor of their node.
__device__ inline std::uint32_t near_first_position(
    float d, bool pass, std::uint32_t mask, std::uint32_t j, std::uint64_t &ties
) {
    float const k = pass ? d : INFINITY;
    std::uint32_t const kb = __float_as_uint(k);
    float const n1 = __uint_as_float(quad_swap1(kb)), n2 = __uint_as_float(quad_swap2(kb));
    float const n3 = __uint_as_float(quad_swap2(quad_swap1(kb)));
    bool const apart = (n1 < k || n1 > k) && (n2 < k || n2 > k) && (n3 < k || n3 > k);
    std::uint32_t pos = (n1 < k ? 1u : 0u) + (n2 < k ? 1u : 0u) + (n3 < k ? 1u : 0u);
    ties = __ballot(pass && !apart);
    if (ties != 0ull) {
        float const k0 = __uint_as_float(quad_bcast<0>(kb)), k1 = __uint_as_float(quad_bcast<1>(kb)),
                    k2 = __uint_as_float(quad_bcast<2>(kb)), k3 = __uint_as_float(quad_bcast<3>(kb));
        std::uint32_t const lo = mask & 4u ? quad_slots4(4) : quad_slots4(0);
        std::uint32_t const hi = mask & 4u ? quad_slots4(12) : quad_slots4(8);
        std::uint32_t const list = (mask & 8u ? hi : lo) >> ((mask & 3u) * 8u);
        std::uint32_t i0 = list & 3u, i1 = (list >> 2) & 3u, i2 = (list >> 4) & 3u, i3 = (list >> 6) & 3u;
        float c0 = pick4(i0, k0, k1, k2, k3), c1 = pick4(i1, k0, k1, k2, k3), c2 = pick4(i2, k0, k1, k2, k3),
              c3 = pick4(i3, k0, k1, k2, k3);
        compare_swap(c0, c1, i0, i1);
        compare_swap(c2, c3, i2, i3);
        compare_swap(c0, c2, i0, i2);
        compare_swap(c1, c3, i1, i3);
        compare_swap(c1, c2, i1, i2);
        pos = i0 == j ? 0u : (i1 == j ? 1u : (i2 == j ? 2u : 3u));
    }
    return pos;
}

} // namespace
} // namespace gwn
