// gwn_ray.hip - nearest ray-triangle hit batch on gfx950.
//
// Reference: include/gwn/detail/gwn_query_ray_impl.cuh:20-595, include/gwn/gwn_query.cuh:182-290.
//
// Four lanes per ray (ray_quad_kernel; one per lane for the work counters, a leaf root and many rays of a few
// triangles).  Two traversals, chosen per batch exactly as the reference's launcher does:
//   packed    (internal root, fewer than 2^29 nodes, packed_stack_bound within the stack): leaf
//             and internal children share one near-ordered sequence of 32-bit payloads (leaf =
//             bit 31 | parent << 2 | slot); the nearest child is entered, the others pushed;
//   canonical (otherwise): leaves of a node are intersected in near order before its internal
//             children are queued; only internal node ids occupy the stack.
// A hit replaces the current best only with a strictly smaller t, so ties resolve by traversal
// order -- the same order as the reference's traversal of the same tree.
//
// Arithmetic is unfused with correctly rounded division, so every record equals the CPU
// oracle's replay bit for bit.
#include <algorithm>
#include <type_traits>

#include "gwn_core.hpp"
#include "gwn_quad.hpp"
#include "../../include/gwn/detail/gwn_device_ray.hpp"

#include <cfloat>

#pragma clang fp contract(off)

namespace gwn {
namespace {

using namespace ::gwn::detail::ray;
constexpr int k_block = 256;
// With Count, only the work counters (slab tests, triangle tests) are written, two per ray.
template <bool Packed, int Cap, bool Count = false>
__global__ __launch_bounds__(k_block) void ray_kernel(
    ray_scene sc, std::uint64_t root_ref, float const *__restrict__ ox, float const *__restrict__ oy,
    float const *__restrict__ oz, float const *__restrict__ dx, float const *__restrict__ dy,
    float const *__restrict__ dz, ray_hit *__restrict__ out, std::size_t n, float t_min, float t_max,
    std::uint32_t *__restrict__ counters = nullptr
) {
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_block + threadIdx.x;
    if (i >= n)
        return;
    traversal_work w;
    ray_hit const res = ray_first_hit_lane<Packed, Cap>(sc, root_ref, ox[i], oy[i], oz[i], dx[i], dy[i], dz[i], t_min,
                                                        t_max, Count ? &w : nullptr);
    if constexpr (Count) {
        counters[2 * i] = w.boxes;
        counters[2 * i + 1] = w.tris;
    } else {
        out[i] = res;
    }
}

constexpr int k_ray_stride = k_block / 4 + 1;  // entry e of quad k's stack at [e * k_ray_stride + k]

// The quads' stacks of a block: per entry a node and the t beyond which it is dropped.  Whole: both words of an
// entry side by side, one 8-byte access.  Half: the nodes, then the upper 16 bits of the largest floats that
// have no others and are not above t (t is not NaN), 6 bytes an entry.
template <bool Half> struct ray_stack;
template <> struct ray_stack<false> {
    static constexpr std::size_t k_entry = sizeof(uint2);
    uint2 *at;
    __device__ ray_stack(std::uint32_t *lds, int, int quad) : at(reinterpret_cast<uint2 *>(lds) + quad) {}
    __device__ void put(int e, std::uint32_t node, float t) { at[e * k_ray_stride] = make_uint2(node, __float_as_uint(t)); }
    __device__ std::uint32_t get(int e, float &t) const {
        uint2 const v = at[e * k_ray_stride];
        t = __uint_as_float(v.y);
        return v.x;
    }
};
template <> struct ray_stack<true> {
    static constexpr std::size_t k_entry = sizeof(std::uint32_t) + sizeof(std::uint16_t);
    std::uint32_t *node;
    std::uint16_t *bound;
    __device__ ray_stack(std::uint32_t *lds, int entries, int quad)
        : node(lds + quad), bound(reinterpret_cast<std::uint16_t *>(lds + entries * k_ray_stride) + quad) {}
    __device__ void put(int e, std::uint32_t n, float t) {
        std::uint32_t const b = __float_as_uint(t);
        node[e * k_ray_stride] = n;
        bound[e * k_ray_stride] = static_cast<std::uint16_t>((b + (b >> 31 != 0u ? 0xffffu : 0u)) >> 16);
    }
    __device__ std::uint32_t get(int e, float &t) const {
        t = __uint_as_float(static_cast<std::uint32_t>(bound[e * k_ray_stride]) << 16);
        return node[e * k_ray_stride];
    }
};
constexpr std::size_t ray_stack_bytes(int entries, bool half) {
    return static_cast<std::size_t>(entries) * k_ray_stride * (half ? ray_stack<true>::k_entry : ray_stack<false>::k_entry);
}

// intersect_triangle's result before it meets the best hit: whether the ray meets the triangle at t >= t_min.
__device__ inline bool triangle_candidate(
    ray_state const &r, tri_record const &tr, float t_min, float &t, float &bu, float &bv, float (&ng)[3]
) {
    best_hit h{INFINITY, 0.0f, 0.0f, {0.0f, 0.0f, 0.0f}, 0u, false};
    intersect_triangle(r, tr, 0u, t_min, h);
    t = h.t;
    bu = h.u;
    bv = h.v;
    ng[0] = h.n[0];
    ng[1] = h.n[1];
    ng[2] = h.n[2];
    return h.found;
}

// Four lanes per ray, lane j of the quad owning child slot j of each node, with the hits of
// ray_first_hit_lane bit for bit.  The four slab tests, and the triangles of the leaf children (one per
// leaf in this library's trees; a triangle's hit does not depend on the best found before it), are
// evaluated side by side, and the quad takes the traversal's steps on them together:
//   canonical: every leaf near first, then the internal children far to near onto the stack, the nearest
//     entered.  A hit nearer than its leaf's box is a rounding case that goes leaf by leaf; without one
//     the smallest t wins, and among equal ones the first in order, whichever leaves the best excludes;
//   packed: the leaves before the first internal child in near-first order, that child entered, the rest
//     (leaves too) onto the stack; up to four leaves from the top of the stack are settled at a time.
// The stack (the quad's column of an LDS array) keeps the slab entry t of each child or a 16-bit lower bound of
// it, and an internal child beyond the best hit is dropped when popped: its children's boxes lie inside its
// own and every operation of the slab test is monotone in the bounds, so they would all have missed.  The
// packed test is not where a direction component's reciprocal is infinite: a side of a child's box in the
// origin's plane gives 0 * inf, and that child is met at any t.  Such rays drop nothing.  (The canonical test
// skips an axis with such a product, so a child's entry is still no nearer than its parent's.)  A wave hands
// its next ray to a quad that has finished (18 nodes a ray on average, 500 at most on the 1M-triangle mesh).
//
// One ray per lane was bound by the gathers: each of a node's eight 16-byte loads touched 64 lines a
// wave, and its stack lived in scratch memory; a quad reads a node's 128 bytes in two.  Measured, one lane per
// ray against this form: 4,194,304 rays on 1,048,576 triangles 5.3 / 3.1 ms (canonical), 4.3 / 3.5 ms
// (packed), on 5,120 1.91 / 1.69 ms; 1,000 rays on 1,048,576 285 / 91 us.
template <bool Packed, bool Half>
__global__ __launch_bounds__(k_block) void ray_quad_kernel(
    ray_scene sc, std::uint32_t root, int cap, float const *__restrict__ ox, float const *__restrict__ oy,
    float const *__restrict__ oz, float const *__restrict__ dx, float const *__restrict__ dy,
    float const *__restrict__ dz, ray_hit *__restrict__ out, std::size_t n, float t_min, float t_max
) {
    extern __shared__ __align__(8) std::uint32_t s_stack[];
    std::uint32_t const lane = threadIdx.x & 63u;
    std::uint32_t const j = lane & 3u;
    std::uint32_t const shift = lane & 60u;
    ray_stack<Half> stack(s_stack, cap, static_cast<int>(threadIdx.x >> 2));
    // The wave's t-th ray: 16 consecutive ones, then 16 one grid further on.
    std::size_t const wave = static_cast<std::size_t>(blockIdx.x) * (k_block / 64) + (threadIdx.x >> 6);
    std::size_t const waves = static_cast<std::size_t>(gridDim.x) * (k_block / 64);
    auto const nth = [=](std::size_t k) { return ((k >> 4) * waves + wave) * 16 + (k & 15); };
    std::size_t taken = 16;  // rays handed out so far, wave-uniform
    std::size_t i = nth(lane >> 2);
    bool live = i < n;
    ray_state r{};
    best_hit best{};
    int sp = 0;
    [[maybe_unused]] bool keep = false;  // packed: a reciprocal is infinite
    bvh_child slot{};
    auto const begin_ray = [&] {
        r.o[0] = ox[i];
        r.o[1] = oy[i];
        r.o[2] = oz[i];
        r.d[0] = dx[i];
        r.d[1] = dy[i];
        r.d[2] = dz[i];
        best = best_hit{t_max, 0.0f, 0.0f, {0.0f, 0.0f, 0.0f}, 0xffffffffu, false};
        sp = 0;
        slot = sc.nodes[root].children[j];
        float const len2 = r.d[0] * r.d[0] + r.d[1] * r.d[1] + r.d[2] * r.d[2];
        if (!(len2 > 0.0f))
            slot.reference = 0;  // a zero direction meets nothing
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            r.zero[k] = r.d[k] == 0.0f;
            r.inv[k] = r.zero[k] ? 0.0f : 1.0f / r.d[k];
        }
        r.parallel = r.zero[0] || r.zero[1] || r.zero[2];
        if constexpr (Packed)
            keep = fmaxf(fmaxf(fabsf(r.inv[0]), fabsf(r.inv[1])), fabsf(r.inv[2])) == INFINITY;
    };
    if (live)
        begin_ray();
    while (__ballot(live) != 0ull) {
        bool finished = false;
        bool overflow = false;
        if (live) {
            // Takes the lane marked by `mine` (at most one a quad) as the best hit.
            auto const take = [&](bool mine, float t, float u, float v, float const (&ng)[3], std::uint32_t rec) {
                auto const share = [&](float x) { return __uint_as_float(quad_or(mine ? __float_as_uint(x) : 0u)); };
                best.t = share(t);
                best.u = share(u);
                best.v = share(v);
                best.n[0] = share(ng[0]);
                best.n[1] = share(ng[1]);
                best.n[2] = share(ng[2]);
                best.prim = sc.prim[quad_or(mine ? rec : 0u)];
                best.found = true;
            };
            // Settles the quad's leaf triangles (this lane's: record `rec`, order `at`, entry t `tn`).
            auto const settle = [&](bool leaf, std::uint32_t rec, std::uint32_t at, float tn) {
                if (__ballot(leaf) == 0ull)
                    return;
                tri_record tr{};
                if (leaf)
                    tr = sc.tris[rec];
                float t, u, v, ng[3];
                bool const hit = triangle_candidate(r, tr, t_min, t, u, v, ng) && leaf;
                if (!Packed && __ballot(hit && t < tn) != 0ull) {
                    for (std::uint32_t s = 0; s < 4; ++s) {
                        bool const mine =
                            hit && at == s && tn <= best.t && (best.found ? t < best.t : t <= best.t);
                        if (quad_or(mine ? 1u : 0u) != 0u)
                            take(mine, t, u, v, ng, rec);
                    }
                } else {
                    float const m = quad_min(hit ? t : INFINITY);
                    bool const any = quad_or(hit ? 1u : 0u) != 0u;
                    if (any && (best.found ? m < best.t : m <= best.t)) {
                        std::uint32_t const key = hit && t == m ? at : 4u;
                        take(key == quad_min(key) && key < 4u, t, u, v, ng, rec);
                    }
                }
            };
            std::uint32_t const child = static_cast<std::uint32_t>(ref_offset(slot.reference));
            float tn = INFINITY;
            bool hit = ref_valid(slot.reference);
            if constexpr (Packed)
                hit = hit && box_packed(r, slot.bounds, t_min, best.t, tn) && tn != INFINITY;
            else
                hit = hit && box_canonical(r, slot.bounds, t_min, best.t, tn);
            bool const is_leaf = ref_leaf(slot.reference);
            std::uint32_t const mask = Packed ? 15u : static_cast<std::uint32_t>(__ballot(hit) >> shift) & 15u;
            std::uint64_t ties;
            std::uint32_t const pos = near_first_position(tn, hit, mask, j, ties);
            std::uint32_t const inner = quad_or(hit && !is_leaf ? 1u << pos : 0u);
            // Positions that go onto the stack or, the first internal one, are entered.
            std::uint32_t const first = inner != 0u ? static_cast<std::uint32_t>(__builtin_ctz(inner)) : 4u;
            std::uint32_t behind = inner;
            if constexpr (Packed)
                behind = quad_or(hit && pos >= first ? 1u << pos : 0u);
            bool found = inner != 0u;
            int const count = __popc(behind);
            int const to = sp + count - 1 - __popc(behind & ((1u << pos) - 1u));
            // The t beyond which the child is dropped.
            float const bound = Packed && keep ? -INFINITY : tn;
            bool const stacked = hit && (Packed ? pos > first : !is_leaf && pos > first);
            if (stacked && to < cap)
                stack.put(to, is_leaf ? (k_payload_leaf | child) : child, bound);
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            std::uint32_t next = quad_or(hit && pos == first ? child : 0u);
            float next_t = __uint_as_float(quad_or(hit && pos == first ? __float_as_uint(bound) : 0u));
            if (found) {
                sp += count - 1;
                overflow = sp > cap;
            }
            // Requested before the leaf triangles are evaluated.
            bvh_child ahead = slot;
            if (found)
                ahead = sc.nodes[next].children[j];
            settle(hit && is_leaf && (!Packed || pos < first), child, pos, tn);
            found = found && !(next_t > best.t);
            bool popped = false;
            while (!found && sp > 0 && !overflow) {
                // The four topmost entries: leaves are settled and excluded nodes dropped up to the first
                // node that is neither.
                int const e = sp - 1 - static_cast<int>(j);
                float et = 0.0f;
                std::uint32_t const en = e >= 0 ? stack.get(e, et) : 0u;
                bool const entry_leaf = Packed && e >= 0 && (en & k_payload_leaf) != 0u;
                std::uint32_t const open =
                    static_cast<std::uint32_t>(__ballot(e >= 0 && !entry_leaf && !(et > best.t)) >> shift) & 15u;
                std::uint32_t const run = open != 0u ? static_cast<std::uint32_t>(__builtin_ctz(open)) : 4u;
                if constexpr (Packed)
                    settle(entry_leaf && j < run, en & ~k_payload_leaf, j, et);
                if (open != 0u) {
                    next = quad_or(j == run ? en : 0u);
                    next_t = __uint_as_float(quad_or(j == run ? __float_as_uint(et) : 0u));
                    found = !(next_t > best.t);
                    popped = found;
                    sp -= static_cast<int>(run) + 1;
                } else {
                    sp = sp > 4 ? sp - 4 : 0;
                }
            }
            if (popped)
                ahead = sc.nodes[next].children[j];
            slot = ahead;
            finished = !found || overflow;
        }
        std::uint64_t const ended = __ballot(finished);
        if (ended != 0ull) {
            if (finished) {
                std::uint32_t const status = overflow ? 2u : (best.found ? 1u : 0u);
                // Each lane writes two of the record's eight words.
                std::uint32_t const lo =
                    j == 0u ? __float_as_uint(best.found ? best.t : -1.0f)
                            : __float_as_uint(j == 1u ? best.v : best.n[1]);
                std::uint32_t const hi = j == 0u   ? __float_as_uint(best.u)
                                         : j == 3u ? status
                                                   : __float_as_uint(j == 1u ? best.n[0] : best.n[2]);
                reinterpret_cast<uint2 *>(out + i)[j] = make_uint2(j == 3u ? best.prim : lo, hi);
                i = nth(taken + static_cast<std::size_t>(__popcll(ended & ((1ull << shift) - 1ull)) >> 2));
                live = i < n;
                if (live)
                    begin_ray();
            }
            taken += static_cast<std::size_t>(__popcll(ended) >> 2);
        }
    }
}

// Blocks of the quad traversal: 16,384 waves where at most 6,144 fit the chip, so that the last ones even out,
// fewer where every quad has its ray at once (4M rays on 1M triangles 3.8-3.9 ms with 2,048 to 4,096 blocks,
// 5.4 ms with a quad per ray; on 5,120 triangles 1.88 ms with 2,048, 1.73 ms with 4,096).
inline unsigned ray_quad_grid(std::size_t n) { return std::min(grid_for(4 * n, k_block), 4096u); }

constexpr std::size_t k_lds_per_cu = std::size_t(160) << 10, k_lds_per_block = std::size_t(64) << 10;

// Whether the stacks keep 16-bit bounds: where LDS with whole floats holds fewer blocks per CU than registers
// do (6) and the grid has more than those.  The arrays are as long as the tree's own stack bound.  4,194,304
// rays, H-PLOC trees, one lane per ray / whole floats at a compiled 64 or 128 entries / this: 1,048,576
// triangles canonical (59 entries) 5.34 / 3.52 / 3.06 ms, packed (94) 4.29 / 5.51 / 3.47 ms; 4,194,304 packed
// (108) 6.32 / 6.44 / 5.18 ms.  Where few blocks run, the conversions only lengthen the chain: 1,000 rays of
// 1,048,576 triangles 93.7 us with 16 bits, 90.5 us without.
bool ray_half_bounds(int entries, unsigned grid) {
    std::size_t const bytes = ray_stack_bytes(entries, false);
    return bytes > k_lds_per_block || (6 * bytes > k_lds_per_cu && grid > 256 * (k_lds_per_cu / bytes));
}

// Large batches over a few nodes keep one ray per lane: nearly every ray meets all of them, so there is no chain
// to shorten and the lanes' work is even.  One lane against four, 4,194,304 rays of 24 triangles 591 / 721 us, of
// 50 775 / 889, of 500 1,291 / 1,243; 1,000,003 of 24 166 / 186; 65,536 of 24 41 / 23.
bool ray_lanes(std::size_t triangles, std::size_t n) { return triangles <= 64 && n >= (std::size_t(1) << 19); }

template <bool Packed, int Cap>
void launch_ray(
    gwn_bvh_handle const &bvh, int need, float const *ox, float const *oy, float const *oz, float const *dx,
    float const *dy, float const *dz, void *out, std::size_t n, float t_min, float t_max,
    std::uint32_t *counters, hipStream_t stream
) {
    ray_scene const sc{bvh.nodes.ptr, bvh.node_count, bvh.triangles.ptr, bvh.primitive_indices.ptr, bvh.triangle_count};
    if (counters != nullptr)
        ray_kernel<Packed, Cap, true><<<grid_for(n, k_block), k_block, 0, stream>>>(
            sc, bvh.root.reference, ox, oy, oz, dx, dy, dz, nullptr, n, t_min, t_max, counters);
    else if (ref_internal(bvh.root.reference) && !ray_lanes(bvh.triangle_count, n)) {
        unsigned const grid = ray_quad_grid(n);
        std::uint32_t const root = static_cast<std::uint32_t>(ref_offset(bvh.root.reference));
        if (ray_half_bounds(need, grid))
            ray_quad_kernel<Packed, true><<<grid, k_block, ray_stack_bytes(need, true), stream>>>(
                sc, root, need, ox, oy, oz, dx, dy, dz, static_cast<ray_hit *>(out), n, t_min, t_max);
        else
            ray_quad_kernel<Packed, false><<<grid, k_block, ray_stack_bytes(need, false), stream>>>(
                sc, root, need, ox, oy, oz, dx, dy, dz, static_cast<ray_hit *>(out), n, t_min, t_max);
    } else
        ray_kernel<Packed, Cap><<<grid_for(n, k_block), k_block, 0, stream>>>(
            sc, bvh.root.reference, ox, oy, oz, dx, dy, dz, static_cast<ray_hit *>(out), n, t_min, t_max);
    GWN_LAUNCH_CHECK();
}

template <bool Packed>
void launch_ray_cap(
    gwn_bvh_handle const &bvh, int need, float const *ox, float const *oy, float const *oz, float const *dx,
    float const *dy, float const *dz, void *out, std::size_t n, float t_min, float t_max, std::uint32_t *counters,
    hipStream_t stream
) {
    if (need <= 32)
        launch_ray<Packed, 32>(bvh, need, ox, oy, oz, dx, dy, dz, out, n, t_min, t_max, counters, stream);
    else if (need <= 64)
        launch_ray<Packed, 64>(bvh, need, ox, oy, oz, dx, dy, dz, out, n, t_min, t_max, counters, stream);
    else if (need <= 128)
        launch_ray<Packed, 128>(bvh, need, ox, oy, oz, dx, dy, dz, out, n, t_min, t_max, counters, stream);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
}

void dispatch_ray(
    gwn_bvh_handle const &bvh, float const *ox, float const *oy, float const *oz, float const *dx,
    float const *dy, float const *dz, void *out, std::size_t n, float t_min, float t_max,
    query_launch const &cfg, std::uint32_t *counters, hipStream_t stream
) {
    if (n == 0)
        return;
    // gwn_query.cuh:276-289: packed payloads hold a 29-bit parent offset.
    bool const packed = ref_internal(bvh.root.reference) && bvh.node_count < (std::size_t(1) << 29) &&
                        static_cast<int>(bvh.packed_stack_bound) <= cfg.stack_capacity;
    if (packed)
        launch_ray_cap<true>(bvh, static_cast<int>(bvh.packed_stack_bound), ox, oy, oz, dx, dy, dz, out, n, t_min,
                             t_max, counters, stream);
    else
        launch_ray_cap<false>(bvh, static_cast<int>(bvh.internal_stack_bound), ox, oy, oz, dx, dy, dz, out, n,
                              t_min, t_max, counters, stream);
}

} // namespace

void ray_first_hit(
    gwn_bvh_handle const &bvh, float const *ox, float const *oy, float const *oz, float const *dx,
    float const *dy, float const *dz, void *out, std::size_t n, float t_min, float t_max,
    query_launch const &cfg, hipStream_t stream
) {
    dispatch_ray(bvh, ox, oy, oz, dx, dy, dz, out, n, t_min, t_max, cfg, nullptr, stream);
}

void ray_first_hit_work(
    gwn_bvh_handle const &bvh, float const *ox, float const *oy, float const *oz, float const *dx,
    float const *dy, float const *dz, std::size_t n, float t_min, float t_max, query_launch const &cfg,
    std::uint32_t *counters, hipStream_t stream
) {
    dispatch_ray(bvh, ox, oy, oz, dx, dy, dz, nullptr, n, t_min, t_max, cfg, counters, stream);
}

} // namespace gwn
