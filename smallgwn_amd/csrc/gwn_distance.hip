// gwn_distance.hip - unsigned point-to-mesh distance batch on gfx950.
//
// Reference: include/gwn/detail/gwn_query_distance_impl.cuh:20-192,
// include/gwn/detail/gwn_query_geometry_impl.cuh:46-114, include/gwn/gwn_query.cuh:109-180.
//
// Near-first culled traversal of the canonical BVH4 (one lane per point in distance_kernel, four or
// 16 in distance_quad_kernel, the default, with the same results): the culling band
// (clamped at zero) is the initial squared bound and the result when nothing is closer; children
// whose box is no closer than the current best are skipped; the survivors are ordered by box
// distance with a five-comparator network; leaves of a node are evaluated before its internal
// children are queued, the nearest internal child is entered directly and the others are pushed
// far-to-near.  A query that reaches distance zero stops (zero is the global lower bound).
// Queries may be visited through a Hilbert-order permutation so that a wave's lanes walk nearby
// paths; results land at the input positions.  With sort_queries = 2 the Hilbert-ordered batch
// uses a wave-cooperative traversal instead (distance_wave_traverse).
//
// Arithmetic is unfused and the square root correctly rounded, so every result equals the CPU
// oracle's replay bit for bit.
#include <algorithm>

#include "gwn_core.hpp"
#include "gwn_quad.hpp"
#include "../../include/gwn/detail/gwn_device_distance.hpp"

#pragma clang fp contract(off)

namespace gwn {
namespace {

using namespace ::gwn::detail::distance;
constexpr int k_block = 256;


// Wave-cooperative form of distance_traverse (sort_queries = 2).  The wave walks one node at a
// time (node records are wave-uniform loads); every lane computes its own box distances and prunes
// by its own best, so a lane's result is its minimum over the triangles it reaches.  A child is
// entered when any lane still needs it; leaves of a node are evaluated before its internal
// children, children in the order of the first needing lane's box distances (near first).
// Pruning compares FP32 box and triangle distances, and a box's distance can round above that of
// a triangle inside it, so which of two equally near triangles survives depends on visiting
// order: results can differ from the reference-order traversal in the last bits.  `s_node` is
// this wave's LDS stack.  Returns the lane's status (k_dist_overflow for every lane when the
// shared stack overflows).
template <int StackCap>
__device__ inline int distance_wave_traverse(
    distance_scene const &sc, bool active, float x, float y, float z, float &best, std::uint32_t *best_rec,
    std::uint32_t *s_node
) {
    int status = k_dist_done;
    if (ref_leaf(sc.root_ref)) {
        if (active && !visit_leaf(sc.tris, sc.nt, sc.root_ref, x, y, z, best, best_rec))
            status = k_dist_zero;
        return status;
    }
    if (!ref_internal(sc.root_ref))
        return status;
    constexpr std::uint32_t k_none = 0xffffffffu;
    int sp = 0;
    bool overflow = false;  // wave-uniform
    std::uint32_t node = static_cast<std::uint32_t>(ref_offset(sc.root_ref));
    while (node != k_none && !overflow) {
        node = __builtin_amdgcn_readfirstlane(node);
        std::uint32_t next = k_none;
        if (node < sc.node_count) {
            bvh_node4 const &nd = sc.nodes[node];
            float cd[4], key[4];
            std::uint64_t cr[4], need[4];
            int idx[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                bvh_child const ch = nd.children[s];
                cr[s] = ch.reference;
                cd[s] = box_distance2(x, y, z, ch.bounds);
                bool const want = active && status == k_dist_done && ref_valid(ch.reference) && cd[s] < best;
                need[s] = __ballot(want);
                key[s] = INFINITY;
                if (need[s] != 0ull) {
                    int const first = __builtin_ctzll(need[s]);
                    key[s] = __builtin_bit_cast(
                        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cd[s]), first));
                }
                idx[s] = s;
            }
            sort4(key, idx);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                int const s = idx[k];
                if (need[s] == 0ull || !ref_leaf(cr[s]))
                    continue;
                if (active && status == k_dist_done && cd[s] < best &&
                    !visit_leaf(sc.tris, sc.nt, cr[s], x, y, z, best, best_rec))
                    status = k_dist_zero;
            }
#pragma unroll
            for (int k = 3; k >= 0; --k) {
                int const s = idx[k];
                if (need[s] == 0ull || !ref_internal(cr[s]) || overflow)
                    continue;
                // Re-check after the leaves: some lanes may no longer need this child.
                if (__ballot(active && status == k_dist_done && cd[s] < best) == 0ull)
                    continue;
                if (next != k_none) {
                    if (sp < StackCap)
                        s_node[sp++] = next;
                    else
                        overflow = true;
                }
                next = static_cast<std::uint32_t>(ref_offset(cr[s]));
            }
        }
        if (next == k_none && sp > 0)
            next = s_node[--sp];
        node = next;
    }
    return overflow ? k_dist_overflow : status;
}

template <int StackCap>
__global__ __launch_bounds__(k_block) void distance_wave_kernel(
    distance_scene sc, float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, float *__restrict__ out, std::size_t n, float culling_band,
    std::uint32_t *__restrict__ nearest
) {
    __shared__ std::uint32_t s_node[k_block / 64][StackCap];
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_block + threadIdx.x;
    bool const active = i < n;
    if (__ballot(active) == 0ull)
        return;
    std::size_t const q = active ? order[i] : 0;
    float const x = active ? qx[q] : 0.0f, y = active ? qy[q] : 0.0f, z = active ? qz[q] : 0.0f;
    float const band = culling_band < 0.0f ? 0.0f : culling_band;
    float best = band * band;
    std::uint32_t rec = k_nearest_none;
    int const st = distance_wave_traverse<StackCap>(sc, active, x, y, z, best, nearest ? &rec : nullptr,
                                                    s_node[threadIdx.x >> 6]);
    if (active) {
        out[q] = st == k_dist_zero ? 0.0f : (st == k_dist_overflow ? __builtin_nanf("") : sqrtf(best));
        if (nearest != nullptr)
            nearest[q] = nearest_code(st, rec);
    }
}

// box_distance2 for a child's box (min <= max): at most one of the two excesses of an axis is positive,
// so their sum is the larger of them and zero.
__device__ inline float child_box_distance2(float x, float y, float z, aabb const &b) {
    float const dx = fmaxf(fmaxf(b.min_x - x, x - b.max_x), 0.0f);
    float const dy = fmaxf(fmaxf(b.min_y - y, y - b.max_y), 0.0f);
    float const dz = fmaxf(fmaxf(b.min_z - z, z - b.max_z), 0.0f);
    return dx * dx + dy * dy + dz * dz;
}

// point_triangle_distance2 of a record without branches: the region (vertex, edge or face) is decided
// by the same comparisons in the same order, one quotient serves every region, and the closest point is
// formed by the region's own operations, so the result is the same bits.  64 lanes over 16 points meet
// every region, and the branched form then runs all of them one after the other with four quotients.
__device__ inline float record_distance2(tri_record const &t, float px, float py, float pz) {
    float const ax = t.v0x, ay = t.v0y, az = t.v0z;
    float const bx = t.v0x + (t.v1x - t.v0x), by = t.v0y + (t.v1y - t.v0y), bz = t.v0z + (t.v1z - t.v0z);
    float const cx = t.v0x + (t.v2x - t.v0x), cy = t.v0y + (t.v2y - t.v0y), cz = t.v0z + (t.v2z - t.v0z);
    float const abx = bx - ax, aby = by - ay, abz = bz - az;
    float const acx = cx - ax, acy = cy - ay, acz = cz - az;
    float const apx = px - ax, apy = py - ay, apz = pz - az;
    float const bpx = px - bx, bpy = py - by, bpz = pz - bz;
    float const cpx = px - cx, cpy = py - cy, cpz = pz - cz;
    float const d1 = dot3(abx, aby, abz, apx, apy, apz), d2 = dot3(acx, acy, acz, apx, apy, apz);
    float const d3 = dot3(abx, aby, abz, bpx, bpy, bpz), d4 = dot3(acx, acy, acz, bpx, bpy, bpz);
    float const d5 = dot3(abx, aby, abz, cpx, cpy, cpz), d6 = dot3(acx, acy, acz, cpx, cpy, cpz);
    float const vc = d1 * d4 - d3 * d2, vb = d5 * d2 - d1 * d6, va = d3 * d6 - d5 * d4;
    float const d43 = d4 - d3, d56 = d5 - d6;
    bool const at_a = d1 <= 0.0f && d2 <= 0.0f;
    bool const at_b = !at_a && d3 >= 0.0f && d4 <= d3;
    bool const on_ab = !at_a && !at_b && vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f;
    bool const at_c = !at_a && !at_b && !on_ab && d6 >= 0.0f && d5 <= d6;
    bool const before = at_a || at_b || on_ab || at_c;
    bool const on_ac = !before && vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f;
    bool const on_bc = !before && !on_ac && va <= 0.0f && d43 >= 0.0f && d56 >= 0.0f;
    bool const edge = on_ab || on_ac || on_bc;
    bool const vertex = at_a || at_b || at_c;
    float const num = on_ab ? d1 : (on_ac ? d2 : (on_bc ? d43 : 1.0f));
    float const den = on_ab ? d1 - d3 : (on_ac ? d2 - d6 : (on_bc ? d43 + d56 : va + vb + vc));
    float const quo = num / den;
    // Edges: base + quo * e; face: (a + (vb quo) ab) + (vc quo) ac.
    float const s = edge ? quo : vb * quo;
    bool const base_b = at_b || on_bc;
    float const ox = at_c ? cx : (base_b ? bx : ax), oy = at_c ? cy : (base_b ? by : ay),
                oz = at_c ? cz : (base_b ? bz : az);
    float const ex = on_bc ? cx - bx : (on_ac ? acx : abx), ey = on_bc ? cy - by : (on_ac ? acy : aby),
                ez = on_bc ? cz - bz : (on_ac ? acz : abz);
    float const w = vc * quo;
    float const hx = ox + s * ex, hy = oy + s * ey, hz = oz + s * ez;
    float const fx = hx + w * acx, fy = hy + w * acy, fz = hz + w * acz;
    float const rx = px - (vertex ? ox : (edge ? hx : fx)), ry = py - (vertex ? oy : (edge ? hy : fy)),
                rz = pz - (vertex ? oz : (edge ? hz : fz));
    return dot3(rx, ry, rz, rx, ry, rz);
}

constexpr int k_stack_stride = k_block / 4 + 1;  // entry e of quad k's stack at [e * k_stack_stride + k]

// The rest of a point's traversal with a row of 16 lanes: quad g of the row tests the g-th entry from the
// top of the stack.  Entries are settled in stack order up to the first whose node has internal children
// to enter; those are pushed, and what the quads behind it found is dropped (their entries stay on the
// stack).  So the nodes, and the leaves of each, take effect in the quad traversal's order; an entry
// excluded by a leaf of one before it needs no undoing, as none of its leaves is below the best then (the
// rounding case goes leaf by leaf).  The order among equal box distances depends on which children
// survive, so an entry with such children waits until it is the top one and the best is settled.  A long
// traversal is mostly nodes with only leaves near its best
// distance, of which this settles up to four at a time.
template <int StackCap, bool WantRec, class Finish>
__device__ inline void distance_row_tail(
    distance_scene const &sc, bool alive, std::size_t q, float x, float y, float z, float best, std::uint32_t rec,
    int sp, std::uint32_t *st_node, float *st_dist, Finish const &finish
) {
    std::uint32_t const lane = threadIdx.x & 63u;
    std::uint32_t const j = lane & 3u;
    std::uint32_t const g = (lane >> 2) & 3u;
    std::uint32_t const shift = lane & 60u, row_shift = lane & 48u;
    bool held = false;      // `slot` is this lane's child of the quad's entry
    float entry_d = 0.0f;
    bvh_child slot{};
    auto const fetch = [&] {
        int const e = sp - 1 - static_cast<int>(g);
        held = e >= 0;
        if (held) {
            entry_d = st_dist[e * k_stack_stride];
            held = !(entry_d >= best);
            if (held)
                slot = sc.nodes[st_node[e * k_stack_stride]].children[j];
        }
    };
    if (alive)
        fetch();
    while (__ballot(alive) != 0ull) {
        if (alive) {
            int status = k_dist_done;
            bool const test = held && !(entry_d >= best);
            float const node_d = entry_d;
            float const d = child_box_distance2(x, y, z, slot.bounds);
            bool const pass = test && ref_valid(slot.reference) && !(d >= best);
            bool const inner = pass && ref_internal(slot.reference);
            std::uint32_t const mask = static_cast<std::uint32_t>(__ballot(pass) >> shift) & 15u;
            std::uint64_t ties;
            std::uint32_t const pos = near_first_position(d, pass, mask, j, ties);
            std::uint32_t const inners = static_cast<std::uint32_t>(__ballot(inner) >> row_shift) & 0xffffu;
            std::uint32_t last = inners != 0u ? static_cast<std::uint32_t>(__builtin_ctz(inners)) >> 2 : 3u;
            std::uint32_t const tied = static_cast<std::uint32_t>(ties >> row_shift) & 0xfff0u;
            if (tied != 0u)
                last = min(last, (static_cast<std::uint32_t>(__builtin_ctz(tied)) >> 2) - 1u);
            bool const enter = inner && g == last;
            bool const leaf = pass && g <= last && ref_leaf(slot.reference) && d < best && ref_offset(slot.reference) < sc.nt;
            std::uint32_t const child = static_cast<std::uint32_t>(ref_offset(slot.reference));
            bool const many = leaf && ref_count(slot.reference) > 1u;
            std::uint64_t const leaf_ref = slot.reference;
            tri_record t{};
            if (leaf)
                t = sc.tris[child];
            sp = sp > static_cast<int>(last) + 1 ? sp - static_cast<int>(last) - 1 : 0;
            std::uint32_t const at = row_or(enter ? 1u << pos : 0u);
            int const count = __popc(at);
            int const to = sp + count - 1 - __popc(at & ((1u << pos) - 1u));
            if (enter && to <= StackCap) {
                st_node[to * k_stack_stride] = child;
                st_dist[to * k_stack_stride] = d;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            sp += count;
            if (sp > StackCap + 1)
                status = k_dist_overflow;
            else
                fetch();  // requested before the leaf triangles are evaluated
            if (__ballot(leaf) != 0ull) {
                float cm = INFINITY;
                std::uint32_t crec = child;
                float const td = record_distance2(t, x, y, z);
                if (leaf && td < cm)
                    cm = td;
                if (many) {
                    cm = INFINITY;
                    visit_leaf(sc.tris, sc.nt, leaf_ref, x, y, z, cm, &crec);
                }
                if (__ballot(leaf && cm < d) != 0ull) {
                    for (std::uint32_t k = 0; k < 16; ++k) {
                        bool const take = leaf && g * 4 + pos == k && !(node_d >= best) && d < best && cm < best;
                        if (row_or(take ? 1u : 0u) != 0u) {
                            best = __uint_as_float(row_or(take ? __float_as_uint(cm) : 0u));
                            if constexpr (WantRec)
                                rec = row_or(take ? crec : 0u);
                        }
                    }
                } else {
                    float const m = __uint_as_float(row_min(__float_as_uint(cm)));  // not negative
                    if (m < best) {
                        best = m;
                        if constexpr (WantRec) {
                            std::uint32_t const first = cm == m ? g * 4 + pos : 16u;
                            rec = row_or(first == row_min(first) ? crec : 0u);
                        }
                    }
                }
                if (!(best > 0.0f) && status == k_dist_done)
                    status = k_dist_zero;
            }
            if (sp == 0 || status != k_dist_done) {
                alive = false;
                if ((lane & 15u) == 0u) {
                    float const p[3] = {x, y, z};
                    finish(q, status, best, rec, p);
                }
            }
        }
    }
}

// Quad form of distance_traverse: four lanes per point, lane j of the quad owning child slot j of
// each node, with distances, nearest records (kept where WantRec) and statuses equal to
// distance_traverse's bit for bit.  Lane j computes its child's box distance and, for a surviving
// leaf child, its triangle's distance (which does not depend on the best found before it); the quad
// then takes distance_traverse's steps together:
//   - leaves, near first, each against the running best.  A leaf distance below its box's is a rounding
//     case that needs the order; without one in the wave the smallest distance wins, and among equal
//     ones the first in order, whichever leaves the running best would have skipped;
//   - internal children far to near onto the stack (the quad's column of an LDS array), the nearest
//     entered.  The stack keeps each entry's box distance, and an entry no closer than the best is
//     dropped when popped: its children's boxes lie inside its own, and every operation of
//     box_distance2 is monotone in the bounds, so none of them would have survived.  So children can be
//     pushed before the node's leaves are evaluated, and the next node's read overlaps them.
// Each wave hands its next point to a quad that has finished: queries' work spreads over two orders of
// magnitude (240 nodes on average, 7,000 at most, on the 1M-triangle mesh), and a wave of 16 fixed points
// lasts as long as its longest.  A wave's points are runs of 4 neighbours from places spread over the
// whole visiting order, since the long ones lie together (1M points of 1M triangles: 14.3 ms, runs of 16
// 16.8 ms, all of a wave's points in a row 42 ms).
// When a wave has no further point to hand out and at most four left, each of them gets a row of 16
// lanes (distance_row_tail).  A batch of no more points than the grid has rows starts that way.
//
// VALU bound from some million points on (84 % of the issue slots at 4M), below that by the instructions
// of the longest point's chain.  Measured against 16 fixed points a wave with the box of every popped node
// tested: 1,000 points of 5,120 triangles 653 -> 160 us; of 1,048,576 8.4 -> 1.8 ms; 1,000,003 of
// 1,048,576 28.5 -> 14.3 ms; 4,000,000 55 -> 41 ms.
//
// `finish(q, status, best, rec, point)` is called by one lane per point.
template <int StackCap, bool WantRec, class Finish>
__device__ inline void distance_quad_range(
    distance_scene const &sc, float const *__restrict__ qx, float const *__restrict__ qy,
    float const *__restrict__ qz, std::uint32_t const *__restrict__ order, std::size_t n, float best0,
    std::uint32_t *s_node, float *s_dist, Finish const &finish
) {
    constexpr int k_stride = k_stack_stride;
    std::uint32_t const lane = threadIdx.x & 63u;
    std::uint32_t const j = lane & 3u;
    std::uint32_t const shift = lane & 60u;
    std::uint32_t *const st_node = s_node + (threadIdx.x >> 2);
    float *const st_dist = s_dist + (threadIdx.x >> 2);
    // The wave's t-th point: 4 consecutive ones of the visiting order, then 4 one grid further on.
    std::size_t const wave = static_cast<std::size_t>(blockIdx.x) * (k_block / 64) + (threadIdx.x >> 6);
    std::size_t const waves = static_cast<std::size_t>(gridDim.x) * (k_block / 64);
    auto const point = [=](std::size_t t) { return ((t >> 2) * waves + wave) * 4 + (t & 3); };
    bool const rows = n <= waves * 4;  // a row per point from the start
    if (!ref_internal(sc.root_ref)) {  // a leaf (or nothing) for a root: one lane per point
        for (std::size_t i = wave * 64 + lane; i < n; i += waves * 64) {
            std::size_t const q = order ? order[i] : i;
            float const p[3] = {qx[q], qy[q], qz[q]};
            float best = best0;
            std::uint32_t rec = k_nearest_none;
            int const status = ref_leaf(sc.root_ref) &&
                                       !visit_leaf(sc.tris, sc.nt, sc.root_ref, p[0], p[1], p[2], best, &rec)
                                   ? k_dist_zero
                                   : k_dist_done;
            finish(q, status, best, rec, p);
        }
        return;
    }
    std::size_t taken = 16;  // points handed out so far, wave-uniform
    std::size_t i = rows ? ((lane & 12u) == 0u ? wave * 4 + (lane >> 4) : n) : point(lane >> 2);
    bool live = i < n;
    bool more = !rows;  // the wave may have further points
    std::size_t q = 0;
    float x = 0.0f, y = 0.0f, z = 0.0f, best = best0;
    std::uint32_t rec = k_nearest_none;
    int sp = 0;
    bvh_child slot{};            // this lane's child of `node`
    std::uint32_t node = 0;
    float node_d = 0.0f;         // the box distance it was entered with
    std::uint32_t const root = static_cast<std::uint32_t>(ref_offset(sc.root_ref));
    auto const begin_point = [&] {
        q = order ? order[i] : i;
        x = qx[q];
        y = qy[q];
        z = qz[q];
        best = best0;
        rec = k_nearest_none;
        sp = 0;
        node = root;
        node_d = -1.0f;
        slot = sc.nodes[root].children[j];
    };
    if (live)
        begin_point();
    for (;;) {
        std::uint64_t const alive = __ballot(live);
        if (alive == 0ull)
            return;
        if (!more && __popcll(alive) <= 16)
            break;
        bool finished = false;
        int status = k_dist_done;
        if (live) {
            float const d = child_box_distance2(x, y, z, slot.bounds);
            bool const pass = ref_valid(slot.reference) && !(d >= best);
            bool const leaf = pass && ref_leaf(slot.reference) && d < best && ref_offset(slot.reference) < sc.nt;
            bool const enter = pass && ref_internal(slot.reference);
            std::uint32_t const child = static_cast<std::uint32_t>(ref_offset(slot.reference));
            tri_record t{};
            if (leaf)
                t = sc.tris[child];
            std::uint32_t const mask = static_cast<std::uint32_t>(__ballot(pass) >> shift) & 15u;
            std::uint64_t ties;
            std::uint32_t const pos = near_first_position(d, pass, mask, j, ties);
            // Internal children far to near onto the stack, the nearest next.
            std::uint32_t const at = quad_or(enter ? 1u << pos : 0u);
            int const count = __popc(at);
            int const rank = __popc(at & ((1u << pos) - 1u));
            std::uint32_t next = quad_or(enter && rank == 0 ? child : 0u);
            float next_d = __uint_as_float(quad_or(enter && rank == 0 ? __float_as_uint(d) : 0u));
            int const to = sp + count - 1 - rank;
            if (enter && rank > 0 && to < StackCap) {
                st_node[to * k_stride] = child;
                st_dist[to * k_stride] = d;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            bool found = count > 0;
            if (found) {
                sp += count - 1;
                status = sp > StackCap ? k_dist_overflow : k_dist_done;
            }
            // The nearest stack entry that the best does not exclude, four at a time.
            auto const pop = [&] {
                while (!found && sp > 0) {
                    int const e = sp - 1 - static_cast<int>(j);
                    float const ed = e >= 0 ? st_dist[e * k_stride] : 0.0f;
                    std::uint32_t const en = e >= 0 ? st_node[e * k_stride] : 0u;
                    std::uint32_t const keep = static_cast<std::uint32_t>(__ballot(e >= 0 && !(ed >= best)) >> shift) & 15u;
                    if (keep != 0u) {
                        std::uint32_t const top = static_cast<std::uint32_t>(__builtin_ctz(keep));
                        next = quad_or(j == top ? en : 0u);
                        next_d = __uint_as_float(quad_or(j == top ? __float_as_uint(ed) : 0u));
                        sp -= static_cast<int>(top) + 1;
                        found = true;
                    } else {
                        sp = sp > 4 ? sp - 4 : 0;
                    }
                }
            };
            if (status == k_dist_done)
                pop();
            // The next node is requested before the leaf triangles are evaluated, and given up if they
            // bring the best below its box.
            bvh_child ahead = slot;
            if (found && status == k_dist_done)
                ahead = sc.nodes[next].children[j];
            if (__ballot(leaf) != 0ull) {
                float cm = INFINITY;
                std::uint32_t crec = child;
                float const td = record_distance2(t, x, y, z);
                if (leaf && td < cm)
                    cm = td;
                if (leaf && ref_count(slot.reference) > 1u) {
                    cm = INFINITY;
                    visit_leaf(sc.tris, sc.nt, slot.reference, x, y, z, cm, &crec);
                }
                if (__ballot(leaf && cm < d) != 0ull) {
                    for (std::uint32_t s = 0; s < 4; ++s) {
                        bool const take = leaf && pos == s && d < best && cm < best;
                        if (quad_or(take ? 1u : 0u) != 0u) {
                            best = __uint_as_float(quad_or(take ? __float_as_uint(cm) : 0u));
                            if constexpr (WantRec)
                                rec = quad_or(take ? crec : 0u);
                            if (!(best > 0.0f) && status == k_dist_done)
                                status = k_dist_zero;
                        }
                    }
                } else {
                    float const m = quad_min(cm);
                    if (m < best) {
                        best = m;
                        if constexpr (WantRec) {
                            std::uint32_t const first = cm == m ? pos : 4u;
                            rec = quad_or(first == quad_min(first) ? crec : 0u);
                        }
                        if (!(best > 0.0f) && status == k_dist_done)
                            status = k_dist_zero;
                    }
                }
                if (found && next_d >= best && status == k_dist_done) {
                    found = false;
                    pop();
                    if (found)
                        ahead = sc.nodes[next].children[j];
                }
            }
            slot = ahead;
            node = next;
            node_d = next_d;
            finished = !found || status != k_dist_done;
        }
        std::uint64_t const ended = __ballot(finished);
        if (ended != 0ull) {
            if (finished) {
                if (j == 0u) {
                    float const p[3] = {x, y, z};
                    finish(q, status, best, rec, p);
                }
                i = point(taken + static_cast<std::size_t>(__popcll(ended & ((1ull << shift) - 1ull)) >> 2));
                live = i < n;
                if (live)
                    begin_point();
            }
            taken += static_cast<std::size_t>(__popcll(ended) >> 2);
            more = more && __ballot(finished && !live) == 0ull;
        }
    }
    // The k-th point left goes to row k, its next node on top of its stack.
    if (live && j == 0u) {
        st_node[sp * k_stride] = node;
        st_dist[sp * k_stride] = node_d;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    std::uint64_t left = __ballot(live) & 0x1111111111111111ull;
    for (std::uint32_t k = 0; k < 3; ++k)
        left = k < (lane >> 4) ? left & (left - 1ull) : left;
    bool const has = left != 0ull;
    int const from = has ? static_cast<int>(__builtin_ctzll(left)) : static_cast<int>(lane);
    distance_row_tail<StackCap, WantRec>(
        sc, has, static_cast<std::size_t>(__shfl(static_cast<unsigned long long>(q), from)), __shfl(x, from),
        __shfl(y, from), __shfl(z, from), __shfl(best, from), static_cast<std::uint32_t>(__shfl(static_cast<int>(rec), from)),
        __shfl(sp, from) + 1, s_node + (threadIdx.x >> 6) * 16 + (from >> 2), s_dist + (threadIdx.x >> 6) * 16 + (from >> 2),
        finish);
}

// Up to this many points every point has a row of 16 lanes from the start: their rows hardly fill the chip, and
// the batch lasts as long as its longest point.  Beyond, quads that hand out points (and rows for the last
// ones) do less in all.  Measured, a row per point / quads: 16,384 points of 500 triangles 83 / 98 us, of
// 1,048,576 2.8 / 3.4 ms; 65,536 of 12 90 / 87 us, of 5,120 301 / 332 us, of 131,072 1.21 / 1.50 ms, of 1,048,576
// 3.6 / 4.0 ms; 131,072 of 500 240 / 194 us, of 5,120 457 / 388 us, of 131,072 2.02 / 2.01 ms, of 1,048,576 6.2 /
// 6.2 ms; 262,144 of 12 165 / 120 us, of 131,072 2.41 / 2.20 ms, of 1,048,576 7.3 / 7.5 ms; 1,000,003 of 1,048,576
// 18.1 / 13.9 ms.
constexpr std::size_t k_row_points = std::size_t(1) << 16;

// Blocks of the quad traversal.  Quads: 16,384 waves where 2,048 to 6,144 fit the chip, as the stacks' LDS lets
// them (half or twice as many measured 5-25 % slower from 1M points on).
inline unsigned distance_quad_grid(std::size_t n) {
    return n <= k_row_points ? grid_for(16 * n, k_block) : std::min(grid_for(4 * n, k_block), 4096u);
}

template <int StackCap, bool WantRec>
__global__ __launch_bounds__(k_block) void distance_quad_kernel(
    distance_scene sc, float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, float *__restrict__ out, std::size_t n, float culling_band,
    std::uint32_t *__restrict__ nearest
) {
    __shared__ std::uint32_t s_node[(StackCap + 1) * k_stack_stride];
    __shared__ float s_dist[(StackCap + 1) * k_stack_stride];
    float const band = culling_band < 0.0f ? 0.0f : culling_band;
    distance_quad_range<StackCap, WantRec>(
        sc, qx, qy, qz, order, n, band * band, s_node, s_dist,
        [&](std::size_t q, int st, float best, std::uint32_t rec, float const (&)[3]) {
            out[q] = st == k_dist_zero ? 0.0f : (st == k_dist_overflow ? __builtin_nanf("") : sqrtf(best));
            if constexpr (WantRec)
                nearest[q] = nearest_code(st, rec);
        });
}

template <int StackCap>
__global__ __launch_bounds__(k_block) void distance_kernel(
    distance_scene sc, float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, float *__restrict__ out, std::size_t n, float culling_band,
    std::uint32_t *__restrict__ nearest
) {
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_block + threadIdx.x;
    if (i >= n)
        return;
    std::size_t const q = order ? order[i] : i;
    float const band = culling_band < 0.0f ? 0.0f : culling_band;
    float best = band * band;
    std::uint32_t rec = k_nearest_none;
    int const st = distance_traverse<StackCap>(sc, qx[q], qy[q], qz[q], best, nearest ? &rec : nullptr);
    out[q] = st == k_dist_zero ? 0.0f : (st == k_dist_overflow ? __builtin_nanf("") : sqrtf(best));
    if (nearest != nullptr)
        nearest[q] = nearest_code(st, rec);
}

// The one-lane traversal in input order, writing only its work counters (box tests, triangle
// tests) per query.
template <int StackCap>
__global__ __launch_bounds__(k_block) void distance_work_kernel(
    distance_scene sc, float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::size_t n, float culling_band, std::uint32_t *__restrict__ counters
) {
    std::size_t const q = static_cast<std::size_t>(blockIdx.x) * k_block + threadIdx.x;
    if (q >= n)
        return;
    float const band = culling_band < 0.0f ? 0.0f : culling_band;
    float best = band * band;
    traversal_work w;
    (void)distance_traverse<StackCap>(sc, qx[q], qy[q], qz[q], best, nullptr, &w);
    counters[2 * q] = w.boxes;
    counters[2 * q + 1] = w.tris;
}

// Barycentric coordinates (of b and c) of the closest point of triangle (a, b, c) to p: the
// Voronoi-region cases of point_triangle_distance2.
__device__ inline void closest_barycentrics(
    float const (&p)[3], float const (&a)[3], float const (&b)[3], float const (&c)[3], float &v, float &w
) {
    float const ab[3] = {b[0] - a[0], b[1] - a[1], b[2] - a[2]};
    float const ac[3] = {c[0] - a[0], c[1] - a[1], c[2] - a[2]};
    float const ap[3] = {p[0] - a[0], p[1] - a[1], p[2] - a[2]};
    float const d1 = dot3(ab[0], ab[1], ab[2], ap[0], ap[1], ap[2]);
    float const d2 = dot3(ac[0], ac[1], ac[2], ap[0], ap[1], ap[2]);
    v = w = 0.0f;
    if (d1 <= 0.0f && d2 <= 0.0f)
        return;
    float const bp[3] = {p[0] - b[0], p[1] - b[1], p[2] - b[2]};
    float const d3 = dot3(ab[0], ab[1], ab[2], bp[0], bp[1], bp[2]);
    float const d4 = dot3(ac[0], ac[1], ac[2], bp[0], bp[1], bp[2]);
    if (d3 >= 0.0f && d4 <= d3) {
        v = 1.0f;
        return;
    }
    float const vc = d1 * d4 - d3 * d2;
    if (vc <= 0.0f && d1 >= 0.0f && d3 <= 0.0f) {
        v = d1 / (d1 - d3);
        return;
    }
    float const cp[3] = {p[0] - c[0], p[1] - c[1], p[2] - c[2]};
    float const d5 = dot3(ab[0], ab[1], ab[2], cp[0], cp[1], cp[2]);
    float const d6 = dot3(ac[0], ac[1], ac[2], cp[0], cp[1], cp[2]);
    if (d6 >= 0.0f && d5 <= d6) {
        w = 1.0f;
        return;
    }
    float const vb = d5 * d2 - d1 * d6;
    if (vb <= 0.0f && d2 >= 0.0f && d6 <= 0.0f) {
        w = d2 / (d2 - d6);
        return;
    }
    float const va = d3 * d6 - d5 * d4;
    if (va <= 0.0f && (d4 - d3) >= 0.0f && (d5 - d6) >= 0.0f) {
        w = (d4 - d3) / ((d4 - d3) + (d5 - d6));
        v = 1.0f - w;
        return;
    }
    float const denom = 1.0f / (va + vb + vc);
    v = vb * denom;
    w = vc * denom;
}

// Per-point part of the distance adjoint once the nearest record is known.
__device__ inline void distance_adjoint_finish(
    distance_scene const &sc, float const (&p)[3], std::size_t q, int st, std::uint32_t rec, float uq,
    std::uint32_t const *__restrict__ prim, std::uint32_t const *__restrict__ i0, std::uint32_t const *__restrict__ i1,
    std::uint32_t const *__restrict__ i2, float *dvx, float *dvy, float *dvz, float *__restrict__ dpx,
    float *__restrict__ dpy, float *__restrict__ dpz
) {
    float g[3] = {0.0f, 0.0f, 0.0f};
    if (st == k_dist_overflow) {
        g[0] = g[1] = g[2] = __builtin_nanf("");
    } else if (st == k_dist_done && rec != 0xffffffffu) {
        tri_record const t = sc.tris[rec];
        float const a[3] = {t.v0x, t.v0y, t.v0z};
        float const b[3] = {t.v0x + (t.v1x - t.v0x), t.v0y + (t.v1y - t.v0y), t.v0z + (t.v1z - t.v0z)};
        float const c[3] = {t.v0x + (t.v2x - t.v0x), t.v0y + (t.v2y - t.v0y), t.v0z + (t.v2z - t.v0z)};
        float v, w;
        closest_barycentrics(p, a, b, c, v, w);
        float const bary[3] = {1.0f - v - w, v, w};
        float r[3];
        for (int k = 0; k < 3; ++k)
            r[k] = p[k] - (bary[0] * a[k] + bary[1] * b[k] + bary[2] * c[k]);
        float const len = sqrtf(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
        if (len > 0.0f) {
            float const su = uq / len;
            std::uint32_t const pr = prim[rec];
            std::uint32_t const ids[3] = {i0[pr], i1[pr], i2[pr]};
            for (int k = 0; k < 3; ++k)
                g[k] = su * r[k];
            for (int vtx = 0; vtx < 3; ++vtx) {
                atomicAdd(dvx + ids[vtx], -bary[vtx] * g[0]);
                atomicAdd(dvy + ids[vtx], -bary[vtx] * g[1]);
                atomicAdd(dvz + ids[vtx], -bary[vtx] * g[2]);
            }
        }
    }
    if (dpx != nullptr) {
        dpx[q] = g[0];
        dpy[q] = g[1];
        dpz[q] = g[2];
    }
}

// Adjoint of sum_p u_p d_p: the forward traversal (same decisions) remembers the nearest record;
// with c = sum b_i v_i its closest point and n = (p - c) / |p - c|, d d/dp = n and
// d d/dv_i = -b_i n (the closest point moves with the triangle).  Points on the surface, beyond the
// band or overflowing the stack contribute nothing (NaN dp on overflow).
template <int StackCap>
__global__ __launch_bounds__(k_block) void distance_adjoint_kernel(
    distance_scene sc, float const *__restrict__ px, float const *__restrict__ py, float const *__restrict__ pz,
    float const *__restrict__ u, std::uint32_t const *__restrict__ order, std::size_t n,
    float culling_band, std::uint32_t const *__restrict__ prim, std::uint32_t const *__restrict__ i0, std::uint32_t const *__restrict__ i1,
    std::uint32_t const *__restrict__ i2, float *dvx, float *dvy, float *dvz, float *__restrict__ dpx,
    float *__restrict__ dpy, float *__restrict__ dpz
) {
    // Four lanes per point (the nearest record of distance_traverse); the quad's first lane finishes
    // the point.
    __shared__ std::uint32_t s_node[(StackCap + 1) * k_stack_stride];
    __shared__ float s_dist[(StackCap + 1) * k_stack_stride];
    float const band = culling_band < 0.0f ? 0.0f : culling_band;
    distance_quad_range<StackCap, true>(
        sc, px, py, pz, order, n, band * band, s_node, s_dist,
        [&](std::size_t q, int st, float, std::uint32_t rec, float const (&p)[3]) {
            distance_adjoint_finish(sc, p, q, st, rec, u[q], prim, i0, i1, i2, dvx, dvy, dvz, dpx, dpy, dpz);
        });
}


// Distance adjoint from the forward's nearest records: no traversal.
__global__ __launch_bounds__(k_block) void distance_adjoint_nearest_kernel(
    distance_scene sc, float const *__restrict__ px, float const *__restrict__ py, float const *__restrict__ pz,
    float const *__restrict__ u, std::uint32_t const *__restrict__ nearest, std::size_t n,
    std::uint32_t const *__restrict__ prim, std::uint32_t const *__restrict__ i0, std::uint32_t const *__restrict__ i1,
    std::uint32_t const *__restrict__ i2, float *dvx, float *dvy, float *dvz, float *__restrict__ dpx,
    float *__restrict__ dpy, float *__restrict__ dpz
) {
    std::size_t const q = static_cast<std::size_t>(blockIdx.x) * k_block + threadIdx.x;
    if (q >= n)
        return;
    std::uint32_t const code = nearest[q];
    bool const valid = code < sc.nt;
    int const st = code == k_nearest_overflow ? k_dist_overflow : (valid ? k_dist_done : k_dist_zero);
    float const p[3] = {px[q], py[q], pz[q]};
    distance_adjoint_finish(sc, p, q, st, valid ? code : k_nearest_none, u[q], prim, i0, i1, i2, dvx, dvy, dvz,
                            dpx, dpy, dpz);
}

template <int Cap>
void launch_distance(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, std::uint32_t const *order,
    float *out, std::size_t n, float band, bool wave, bool quad, std::uint32_t *nearest, hipStream_t stream
) {
    distance_scene const sc{bvh.nodes.ptr, bvh.node_count, bvh.triangles.ptr, bvh.triangle_count, bvh.root.reference};
    if (wave && order != nullptr)
        distance_wave_kernel<Cap><<<grid_for(n, k_block), k_block, 0, stream>>>(sc, qx, qy, qz, order, out, n, band,
                                                                                  nearest);
    else if (quad && nearest != nullptr)
        distance_quad_kernel<Cap, true><<<distance_quad_grid(n), k_block, 0, stream>>>(
            sc, qx, qy, qz, order, out, n, band, nearest);
    else if (quad)
        distance_quad_kernel<Cap, false><<<distance_quad_grid(n), k_block, 0, stream>>>(
            sc, qx, qy, qz, order, out, n, band, nullptr);
    else
        distance_kernel<Cap><<<grid_for(n, k_block), k_block, 0, stream>>>(sc, qx, qy, qz, order, out, n, band,
                                                                             nearest);
    GWN_LAUNCH_CHECK();
}

} // namespace

void unsigned_distance(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, float *out, std::size_t n,
    float culling_band, query_launch const &cfg, std::uint32_t *nearest, hipStream_t stream
) {
    if (n == 0)
        return;
    bool const sort = cfg.sort_queries > 0 || (cfg.sort_queries < 0 && n >= (1u << 16));
    bool const wave = cfg.sort_queries == 2;
    // Four lanes per point (or 16, distance_quad_range) unless one is asked for: the results are the same.
    bool const quad = cfg.lanes_per_point != 1;
    device_buffer<std::uint32_t> order;
    if (sort) {
        order.allocate(n, stream);
        query_order(bvh, qx, qy, qz, order.ptr, n, stream);
    }
    int const need = static_cast<int>(bvh.internal_stack_bound);
    if (need <= 32)
        launch_distance<32>(bvh, qx, qy, qz, order.ptr, out, n, culling_band, wave, quad, nearest, stream);
    else if (need <= 64)
        launch_distance<64>(bvh, qx, qy, qz, order.ptr, out, n, culling_band, wave, quad, nearest, stream);
    else if (need <= 128)
        launch_distance<128>(bvh, qx, qy, qz, order.ptr, out, n, culling_band, wave, quad, nearest, stream);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
}

void unsigned_distance_work(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, std::size_t n, float culling_band,
    std::uint32_t *counters, hipStream_t stream
) {
    if (n == 0)
        return;
    distance_scene const sc{bvh.nodes.ptr, bvh.node_count, bvh.triangles.ptr, bvh.triangle_count, bvh.root.reference};
    int const need = static_cast<int>(bvh.internal_stack_bound);
    unsigned const grid = grid_for(n, k_block);
    if (need <= 32)
        distance_work_kernel<32><<<grid, k_block, 0, stream>>>(sc, qx, qy, qz, n, culling_band, counters);
    else if (need <= 64)
        distance_work_kernel<64><<<grid, k_block, 0, stream>>>(sc, qx, qy, qz, n, culling_band, counters);
    else if (need <= 128)
        distance_work_kernel<128><<<grid, k_block, 0, stream>>>(sc, qx, qy, qz, n, culling_band, counters);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
    GWN_LAUNCH_CHECK();
}

void unsigned_distance_adjoint(
    gwn_geometry_handle const &g, gwn_bvh_handle const &bvh, float const *px, float const *py, float const *pz,
    float const *u, std::size_t n, float culling_band, std::uint32_t const *nearest, float *dvx, float *dvy,
    float *dvz, float *dpx, float *dpy, float *dpz, hipStream_t stream
) {
    if (n == 0 || bvh.triangle_count == 0)
        return;
    if (nearest != nullptr) {
        distance_scene const sc{bvh.nodes.ptr, bvh.node_count, bvh.triangles.ptr, bvh.triangle_count,
                                bvh.root.reference};
        distance_adjoint_nearest_kernel<<<grid_for(n, k_block), k_block, 0, stream>>>(
            sc, px, py, pz, u, nearest, n, bvh.primitive_indices.ptr, g.i0.ptr, g.i1.ptr, g.i2.ptr, dvx, dvy, dvz,
            dpx, dpy, dpz);
        GWN_LAUNCH_CHECK();
        return;
    }
    device_buffer<std::uint32_t> order;
    if (n >= (1u << 16)) {
        order.allocate(n, stream);
        query_order(bvh, px, py, pz, order.ptr, n, stream);
    }
    distance_scene const sc{bvh.nodes.ptr, bvh.node_count, bvh.triangles.ptr, bvh.triangle_count, bvh.root.reference};
    int const need = static_cast<int>(bvh.internal_stack_bound);
#define GWN_DADJ(C)                                                                                            \
    distance_adjoint_kernel<C><<<distance_quad_grid(n), k_block, 0, stream>>>(                                \
        sc, px, py, pz, u, order.ptr, n, culling_band, bvh.primitive_indices.ptr, g.i0.ptr, g.i1.ptr, g.i2.ptr, \
        dvx, dvy, dvz, dpx, dpy, dpz)
    if (need <= 32)
        GWN_DADJ(32);
    else if (need <= 64)
        GWN_DADJ(64);
    else if (need <= 128)
        GWN_DADJ(128);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
#undef GWN_DADJ
    GWN_LAUNCH_CHECK();
}

} // namespace gwn
