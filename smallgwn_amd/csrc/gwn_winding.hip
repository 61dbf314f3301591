// gwn_winding.hip - exact and Taylor winding-number batches on gfx950.
//
// Reference: include/gwn/detail/gwn_query_winding_impl.cuh:102-443,
// include/gwn/detail/gwn_query_geometry_impl.cuh:16-45, include/gwn/gwn_query.cuh:296-445.
//
// Exact batch: one query per lane; the block streams the leaf-ordered triangle records through
// LDS in 256-record tiles, so every record is read from HBM/L2 once per block and broadcast to
// all 256 lanes.  VALU bound (solid angle: 3 sqrt, 3 div, 1 atan2 per pair).
//
// Taylor batch: 16 or four lanes per query, or 64 queries per wave where Hilbert-ordered queries are dense
// (results are written back in input order).  A stack of internal node ids; the last internal child
// of a node is entered directly, the others are pushed, leaves are evaluated in slot order --
// the reference's traversal order, so float sums are formed in the same sequence.  The node
// data is one traversal record per node (compact child refs + field-SoA coefficients), so a
// node visit touches 2-3 consecutive 128-byte lines and no separate hierarchy array.
//
// Precision split: traversal and far-field Taylor terms in FP32; a leaf triangle within four edge
// lengths of the query in FP64 on the exact vertices, farther leaf triangles in FP32; every term
// accumulated in FP64.
//
// Products are contracted into FMAs only within one source expression (contract(on), not the
// default across statements), so every kernel that evaluates a term -- per-lane, wave, gradient,
// batched -- rounds it identically and their results agree bit for bit.
#include <mutex>
#include <type_traits>

#include "gwn_core.hpp"
#include "gwn_slices.hpp"
#include "../../include/gwn/detail/gwn_device_winding.hpp"
#include "gwn_quad.hpp"

#include <algorithm>
#include <cmath>

#pragma clang fp contract(on)

namespace gwn {
namespace {

using namespace ::gwn::detail::winding;
constexpr std::uint32_t k_invalid = 0xffffffffu;

// ------------------------------------------------------------------------------------------
// Exact batch
// ------------------------------------------------------------------------------------------

constexpr int k_exact_block = 256;

// What one triangle contributes to every query's solid angle, formed once per tile while the
// record is staged: 64 bytes, so a lane's broadcast reads are four aligned 16-byte LDS reads.
// Plain: the reference's corners v0, v0 + (v1 - v0), v0 + (v2 - v0).  Split: v0, the edges
// e1, e2, their cross product n, |e1|^2, |e2|^2, e1 . e2 and the squared near-field radius.
struct __align__(16) exact_item {
    float f[16];
    __device__ static exact_item load(exact_item const &src) {
        exact_item t;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            reinterpret_cast<float4 *>(t.f)[j] = reinterpret_cast<float4 const *>(src.f)[j];
        return t;
    }
};

template <int Prec>
__device__ inline void stage_exact_item(tri_record const &t, exact_item &o) {
    float const e1x = t.v1x - t.v0x, e1y = t.v1y - t.v0y, e1z = t.v1z - t.v0z;
    float const e2x = t.v2x - t.v0x, e2y = t.v2y - t.v0y, e2z = t.v2z - t.v0z;
    float4 *const d = reinterpret_cast<float4 *>(o.f);
    d[0] = {t.v0x, t.v0y, t.v0z, Prec == GWN_PRECISION_PLAIN ? t.v0x + e1x : e1x};
    if constexpr (Prec == GWN_PRECISION_PLAIN) {
        d[1] = {t.v0y + e1y, t.v0z + e1z, t.v0x + e2x, t.v0y + e2y};
        d[2] = {t.v0z + e2z, 0.0f, 0.0f, 0.0f};
    } else {
        float const s1 = e1x * e1x + e1y * e1y + e1z * e1z;
        float const s2 = e2x * e2x + e2y * e2y + e2z * e2z;
        d[1] = {e1y, e1z, e2x, e2y};
        d[2] = {e2z, e1y * e2z - e1z * e2y, e1z * e2x - e1x * e2z, e1x * e2y - e1y * e2x};
        d[3] = {s1, s2, e1x * e2x + e1y * e2y + e1z * e2z, k_split_near_scale2 * fmaxf(s1, s2)};
    }
}

// solid_angle_plain on the staged corners.
__device__ inline float solid_angle_plain_staged(exact_item const &t, float qx, float qy, float qz) {
    return solid_angle_corners(t.f[0] - qx, t.f[1] - qy, t.f[2] - qz, t.f[3] - qx, t.f[4] - qy, t.f[5] - qz,
                               t.f[6] - qx, t.f[7] - qy, t.f[8] - qz);
}

// half_angle_far of a staged triangle.
__device__ inline float half_angle_far_staged(exact_item const &t, float ax, float ay, float az, float aa, bool far) {
    return half_angle_far(aa, ax * t.f[3] + ay * t.f[4] + az * t.f[5], ax * t.f[6] + ay * t.f[7] + az * t.f[8],
                          ax * t.f[9] + ay * t.f[10] + az * t.f[11], t.f[12], t.f[13], t.f[14], far);
}

// Adds the values of a group's Lanes lanes to its running sum in lane order (the group's lanes are
// Lanes consecutive lanes of a 16-lane row; every one ends with the same sum).
template <int Lanes, int J = 0> __device__ inline void add_in_lane_order(float &sum, float v) {
    if constexpr (Lanes == 1) {
        sum += v;
    } else if constexpr (J < Lanes) {
        constexpr int k_ctrl = Lanes == 4 ? J * 0x55 : 0x150 + J;  // quad_perm [J, J, J, J] / row_newbcast:J
        sum += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), k_ctrl, 0xf, 0xf, false));
        add_in_lane_order<Lanes, J + 1>(sum, v);
    }
}

// Plain exact batch, Lanes (1, 4 or 16) lanes per query: lane j of a query's group evaluates
// triangles j, j + Lanes, ... of each 256-record tile, and the group adds each round's angles in
// record order, so every query's float sum is formed over the records in the reference's order
// whatever Lanes is (a lane past the tile's end adds zero, which changes no sum).
//
// VALU bound: about 165 issue slots a pair (nine correctly rounded quotients, three square roots,
// one arctangent), one to sixteen for the ordered add.  One lane per query leaves the chip idle
// below some hundred thousand queries.  Measured with one lane and the general quotients, square roots and
// arctangent (220 slots) against this form: 131,044 triangles x 1,000 queries 74.0 against 5.6 ms (the groups
// alone), 100,000 x 65,536 56.5 against 22.0 ms.
template <int Lanes, class Out>
__global__ __launch_bounds__(k_exact_block) void exact_plain_kernel(
    tri_record const *__restrict__ tris, std::size_t nt, float const *__restrict__ qx,
    float const *__restrict__ qy, float const *__restrict__ qz, Out *__restrict__ out, std::size_t nq
) {
    static_assert(Lanes == 1 || Lanes == 4 || Lanes == 16, "groups are a lane, a quad or a row");
    __shared__ exact_item tile[k_exact_block];
    std::size_t const qi = (static_cast<std::size_t>(blockIdx.x) * k_exact_block + threadIdx.x) / Lanes;
    int const j = static_cast<int>(threadIdx.x) % Lanes;
    bool const active = qi < nq;
    float const x = active ? qx[qi] : 0.0f;
    float const y = active ? qy[qi] : 0.0f;
    float const z = active ? qz[qi] : 0.0f;
    float sum = 0.0f;
    for (std::size_t base = 0; base < nt; base += k_exact_block) {
        int const count = static_cast<int>((nt - base) < k_exact_block ? (nt - base) : k_exact_block);
        __syncthreads();
        if (static_cast<int>(threadIdx.x) < count)
            stage_exact_item<GWN_PRECISION_PLAIN>(tris[base + threadIdx.x], tile[threadIdx.x]);
        __syncthreads();
        for (int k = 0; k < count; k += Lanes) {
            float v = 0.0f;
            if (Lanes == 1 || k + j < count)
                v = solid_angle_plain_staged(tile[k + j], x, y, z);
            add_in_lane_order<Lanes>(sum, v);
        }
    }
    if (active && j == 0)
        out[qi] = static_cast<Out>(sum / (4.0f * k_pi_f));
}

// Split and FP64 exact batches: one query per lane; the block streams its share of the leaf-ordered
// records through LDS in 256-record tiles.  blockIdx.y is the share: tiles [y, y + 1) *
// tiles_per_share.  With one share the winding number goes to `out`; with more, the share's FP64 sum
// goes to part[y * nq + q] and exact_combine_kernel adds the shares in order.
//
// VALU bound (a far split pair costs 49 issue slots), so what counts is that every SIMD has waves: a
// launch of nq / 256 blocks alone left 32,749 queries on half of the CUs with one wave per SIMD.
// Measured, split, one share with per-pair edges and arctangents against this form: 100,000 triangles
// x 32,749 queries 38.1 against 4.7 ms, 131,044 x 1,000 52.3 against 0.48 ms, 25,600 x 600,000 (one
// share in both) 56.9 against 37.0 ms.
//
// OneTile: at most 256 triangles, most of them near most queries.  Waves without a far pair skip its arithmetic,
// and near triangles come from LDS (elsewhere the test costs 2 % and the larger tile 3-5 %): 4,000,000 queries of 24
// triangles 365 us without, 293 with, 1,000 of 24 15.8 and 11.9 us.
template <int Prec, bool OneTile>
__global__ __launch_bounds__(k_exact_block) void exact_kernel(
    tri_record const *__restrict__ tris, std::size_t nt, float const *__restrict__ qx,
    float const *__restrict__ qy, float const *__restrict__ qz, double *__restrict__ out, double *__restrict__ part,
    std::size_t nq, std::size_t tiles_per_share
) {
    static_assert(Prec == GWN_PRECISION_SPLIT || Prec == GWN_PRECISION_FP64, "FP64 sums");
    constexpr bool k_raw = Prec == GWN_PRECISION_FP64;
    __shared__ std::conditional_t<k_raw, tri_record, exact_item> tile[k_exact_block];
    __shared__ tri_record raw[OneTile && !k_raw ? k_exact_block : 1];
    std::size_t const qi = static_cast<std::size_t>(blockIdx.x) * k_exact_block + threadIdx.x;
    bool const active = qi < nq;
    float const x = active ? qx[qi] : 0.0f;
    float const y = active ? qy[qi] : 0.0f;
    float const z = active ? qz[qi] : 0.0f;
    double sum = 0.0;
    std::size_t const share = tiles_per_share * k_exact_block;
    std::size_t const first = static_cast<std::size_t>(blockIdx.y) * share;
    std::size_t const last = nt - first < share ? nt : first + share;
    for (std::size_t base = first; base < last; base += k_exact_block) {
        int const count = static_cast<int>((last - base) < k_exact_block ? (last - base) : k_exact_block);
        __syncthreads();
        if (static_cast<int>(threadIdx.x) < count) {
            if constexpr (k_raw)
                tile[threadIdx.x] = tris[base + threadIdx.x];
            else
                stage_exact_item<Prec>(tris[base + threadIdx.x], tile[threadIdx.x]);
            if constexpr (OneTile && !k_raw)
                raw[threadIdx.x] = tris[base + threadIdx.x];
        }
        __syncthreads();
        if constexpr (k_raw) {
            for (int k = 0; k < count; ++k)
                sum += solid_angle_f64(tile[k], x, y, z);
        } else {
            // Per-tile FP32 partial sums of the far triangles, folded into the FP64 total.
            float far = 0.0f;
            for (int k = 0; k < count; ++k) {
                exact_item const t = exact_item::load(tile[k]);
                float const ax = t.f[0] - x, ay = t.f[1] - y, az = t.f[2] - z;
                float const aa = ax * ax + ay * ay + az * az;
                bool const near = !(aa > t.f[15]);
                if (!OneTile || __ballot(!near) != 0ull) {
                    float const h = half_angle_far_staged(t, ax, ay, az, aa, !near);
                    far += near ? 0.0f : h;
                }
                if (near)
                    sum += solid_angle_split_near(OneTile ? raw[k] : tris[base + k], x, y, z);
            }
            sum += 2.0 * double(far);
        }
    }
    if (!active)
        return;
    if (part != nullptr)
        part[static_cast<std::size_t>(blockIdx.y) * nq + qi] = sum;
    else
        out[qi] = sum / (4.0 * k_pi_d);
}

// Winding numbers from the shares' sums, added in share order (the same bits on every run).
__global__ __launch_bounds__(256) void exact_combine_kernel(
    double const *__restrict__ part, std::size_t shares, double *__restrict__ out, std::size_t nq
) {
    std::size_t const q = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (q >= nq)
        return;
    double s = 0.0;
    for (std::size_t k = 0; k < shares; ++k)
        s += part[k * nq + q];
    out[q] = s / (4.0 * k_pi_d);
}

// Shares of the triangles per query block.  Up to 8 blocks of 256 fit a CU (LDS and registers), so
// 16 per CU give every SIMD eight waves and a second round to even out the last one.  A share is at
// least one tile (256 pairs a lane, beside which its staging and its sum are small), and the shares'
// sums take at most 64 MiB.
std::size_t exact_shares(std::size_t nt, std::size_t nq) {
    std::size_t const blocks = (nq + k_exact_block - 1) / k_exact_block;
    std::size_t const tiles = (nt + k_exact_block - 1) / k_exact_block;
    std::size_t const target = 16 * 256;
    if (blocks >= target)
        return 1;
    std::size_t s = (target + blocks - 1) / blocks;
    std::size_t const by_bytes = (std::size_t(64) << 20) / (nq * sizeof(double));
    s = s < tiles ? s : tiles;
    s = s < by_bytes ? s : by_bytes;
    return s == 0 ? 1 : s;
}

template <int Prec>
void launch_exact(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, double *out, std::size_t nq,
    hipStream_t stream
) {
    std::size_t const nt = bvh.triangle_count;
    std::size_t const tiles = (nt + k_exact_block - 1) / k_exact_block;
    std::size_t shares = exact_shares(nt, nq);
    if (shares > 1 && stream_capturing(stream))  // a captured batch stays one launch without an allocation
        shares = 1;
    std::size_t tiles_per_share = tiles == 0 ? 1 : (tiles + shares - 1) / shares;
    shares = tiles == 0 ? 1 : (tiles + tiles_per_share - 1) / tiles_per_share;  // none is empty
    device_buffer<double> part;
    if (shares > 1 && !part.try_allocate(shares * nq, stream)) {  // no memory for the sums: no shares
        shares = 1;
        tiles_per_share = tiles;
    }
    dim3 const grid(grid_for(nq, k_exact_block), static_cast<unsigned>(shares));
    auto const kernel = tiles <= 1 && Prec == GWN_PRECISION_SPLIT ? exact_kernel<Prec, Prec == GWN_PRECISION_SPLIT>
                                                                  : exact_kernel<Prec, false>;
    kernel<<<grid, k_exact_block, 0, stream>>>(bvh.triangles.ptr, nt, qx, qy, qz, out, part.ptr, nq, tiles_per_share);
    GWN_LAUNCH_CHECK();
    if (shares > 1) {
        exact_combine_kernel<<<grid_for(nq, 256), 256, 0, stream>>>(part.ptr, shares, out, nq);
        GWN_LAUNCH_CHECK();
    }
}

// Plain: the widest groups whose launch still holds eight waves per SIMD, since the ordered add costs
// up to 16 issue slots a pair with 16 lanes against one with one lane.
template <class Out>
void launch_exact_plain(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, Out *out, std::size_t nq,
    hipStream_t stream
) {
    std::size_t const full = std::size_t(256) * 8 * k_exact_block;  // lanes of eight waves on every SIMD
#define GWN_EXACT_PLAIN(L)                                                                        \
    exact_plain_kernel<L, Out><<<grid_for(nq * L, k_exact_block), k_exact_block, 0, stream>>>(    \
        bvh.triangles.ptr, bvh.triangle_count, qx, qy, qz, out, nq)
    if (nq >= full)
        GWN_EXACT_PLAIN(1);
    else if (nq * 4 >= full)
        GWN_EXACT_PLAIN(4);
    else
        GWN_EXACT_PLAIN(16);
#undef GWN_EXACT_PLAIN
    GWN_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------------------
// Taylor batch
// ------------------------------------------------------------------------------------------

constexpr int k_taylor_block = 256;

__device__ inline std::uint32_t spread10(std::uint32_t v) {
    std::uint32_t x = v & 0x3ffu;
    x = (x | (x << 16)) & 0x030000ffu;
    x = (x | (x << 8)) & 0x0300f00fu;
    x = (x | (x << 4)) & 0x030c30c3u;
    x = (x | (x << 2)) & 0x09249249u;
    return x;
}

// Position of a cell of the 1024^3 grid along the 3-D Hilbert curve (30 bits), by Skilling's
// transpose method ("Programming the Hilbert curve", AIP Conf. Proc. 707, 2004): undo the
// excess work on the axes' bits from the top down, Gray-encode, then interleave the transposed
// bits (axis 0 most significant in each triple).  Consecutive keys are face-adjacent cells, so a
// wave of consecutive queries is more compact than along the Morton curve, whose keys jump.
__device__ inline std::uint32_t hilbert_key10(std::uint32_t x0, std::uint32_t x1, std::uint32_t x2) {
    std::uint32_t X[3] = {x0 & 0x3ffu, x1 & 0x3ffu, x2 & 0x3ffu};
    for (std::uint32_t Q = 1u << 9; Q > 1u; Q >>= 1) {
        std::uint32_t const P = Q - 1u;
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            if (X[i] & Q) {
                X[0] ^= P;
            } else {
                std::uint32_t const t = (X[0] ^ X[i]) & P;
                X[0] ^= t;
                X[i] ^= t;
            }
        }
    }
    X[1] ^= X[0];
    X[2] ^= X[1];
    std::uint32_t t = 0;
    for (std::uint32_t Q = 1u << 9; Q > 1u; Q >>= 1)
        if (X[2] & Q)
            t ^= Q - 1u;
    X[0] ^= t;
    X[1] ^= t;
    X[2] ^= t;
    return (spread10(X[0]) << 2) | (spread10(X[1]) << 1) | spread10(X[2]);
}

// Sort keys of the query presort: each query's Hilbert position on the 1024^3 grid over the
// BVH's root box (points outside are clamped onto it).
__global__ __launch_bounds__(256) void query_key_kernel(
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::size_t n, aabb box, std::uint32_t *__restrict__ keys, std::uint32_t *__restrict__ ids
) {
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (i >= n)
        return;
    float const sx = box.max_x > box.min_x ? 1.0f / (box.max_x - box.min_x) : 1.0f;
    float const sy = box.max_y > box.min_y ? 1.0f / (box.max_y - box.min_y) : 1.0f;
    float const sz = box.max_z > box.min_z ? 1.0f / (box.max_z - box.min_z) : 1.0f;
    // NaN coordinates compare false and land in cell 0; order only affects performance.
    float const fx = fminf(fmaxf((qx[i] - box.min_x) * sx, 0.0f), 1.0f) * 1023.0f;
    float const fy = fminf(fmaxf((qy[i] - box.min_y) * sy, 0.0f), 1.0f) * 1023.0f;
    float const fz = fminf(fmaxf((qz[i] - box.min_z) * sz, 0.0f), 1.0f) * 1023.0f;
    keys[i] = hilbert_key10(static_cast<std::uint32_t>(fx), static_cast<std::uint32_t>(fy),
                            static_cast<std::uint32_t>(fz));
    ids[i] = static_cast<std::uint32_t>(i);
}


// A wave-uniform value in scalar registers (one read back from LDS otherwise lives in vector ones, and
// every mask formed from it with it).
__device__ inline std::uint64_t uniform_u64(std::uint64_t v) {
    std::uint32_t const lo = __builtin_amdgcn_readfirstlane(static_cast<std::uint32_t>(v));
    std::uint32_t const hi = __builtin_amdgcn_readfirstlane(static_cast<std::uint32_t>(v >> 32));
    return (static_cast<std::uint64_t>(hi) << 32) | lo;
}

// Wave-cooperative traversal (defined below; the batched kernel uses it too).
template <int Order, int Prec, bool Grad, bool Count>
__device__ inline bool taylor_wave_traverse(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node, bool active,
    float x, float y, float z, float beta2, taylor_sums<Prec, Grad> &acc, std::uint32_t &n_tests,
    std::uint32_t &n_accept, std::uint32_t &n_leaf, std::uint32_t *s_node, std::uint64_t *s_mask, int cap
);

// Four lanes per query (defined below; the batched kernel uses it too).
template <int Order, int Prec, bool Grad, int StackCap>
__device__ inline bool taylor_quad_traverse(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node, float x, float y,
    float z, float beta2, taylor_sums<Prec, Grad> &acc, std::uint32_t &n_tests, std::uint32_t &n_accept,
    std::uint32_t &n_leaf, std::uint32_t *stack, int stride, int cap
);

// Batched persistent traversal: many meshes, one launch.  Work is a list of chunks of consecutive
// queries of one mesh (the mesh's `chunk` of them); every block takes chunks from a global counter
// until none is left (no wave waits for another) and evaluates them with that mesh's records and the
// traversals of the single-mesh batch, so each result equals that batch's.  A mesh whose `wave` flag
// is set is walked by whole waves, any other with four lanes per query (a wave walks the union of its
// lanes' paths, which pays where a mesh's queries are dense and costs where a few queries are spread
// over a large tree: one such wave alone can last as long as the rest of the launch).  Waves, Quads:
// whether any mesh may be walked either way.  A block walks one way at a time, so both kinds of stacks share
// its LDS, batch_lds_bytes of it for `cap` entries (both at a compiled 128 entries and a block of 256 held four
// blocks a CU: 20M queries of 200 meshes of 1,000 triangles 5.92 ms, 4.92 now; in blocks of 64 15.3, 4.6).  Rebuild and query of 128 meshes of up to 100,000 triangles, recorded:
// 8.04 ms with whole waves for every mesh, 4.16 now (2.36M queries in all); of 8 meshes with 174,131:
// 4.69, 1.28; of 512 with 9.0M: 14.2, 11.5.
template <int Order, bool Waves, bool Quads>
__global__ __launch_bounds__(256) void taylor_batch_kernel(
    batch_mesh const *__restrict__ meshes, std::uint32_t mesh_count, std::uint64_t total_chunks, float beta2, int cap,
    std::uint64_t *counter
) {
    __shared__ std::uint64_t s_chunk;
    extern __shared__ std::uint64_t s_stacks[];
    int const wave = threadIdx.x >> 6;
    int const quads = static_cast<int>(blockDim.x >> 2);
    std::uint64_t *const s_mask = s_stacks + wave * cap;
    std::uint32_t *const s_node = reinterpret_cast<std::uint32_t *>(s_stacks + static_cast<int>(blockDim.x >> 6) * cap) + wave * cap;
    std::uint32_t *const s_quad = reinterpret_cast<std::uint32_t *>(s_stacks) + (threadIdx.x >> 2);  // entry e at [e * quads]
    for (;;) {
        if (threadIdx.x == 0)
            s_chunk = atomicAdd(reinterpret_cast<unsigned long long *>(counter), 1ull);
        __syncthreads();
        std::uint64_t const c = s_chunk;
        __syncthreads();
        if (c >= total_chunks)
            return;
        // Mesh of this chunk: last mesh whose first_chunk <= c (binary search).
        std::uint32_t lo = 0, hi = mesh_count;
        while (hi - lo > 1) {
            std::uint32_t const mid = (lo + hi) >> 1;
            if (meshes[mid].first_chunk <= c)
                lo = mid;
            else
                hi = mid;
        }
        batch_mesh const m = meshes[lo];
        std::uint32_t const chunk = m.chunk;
        std::uint64_t const base = (c - m.first_chunk) * chunk;
        if (Quads && !ref_leaf(m.root) && !(Waves && m.wave != 0u)) {  // uniform over the block
            for (std::uint32_t t = threadIdx.x >> 2; t < chunk; t += blockDim.x >> 2) {  // whole quads
                std::uint64_t const p = base + t;
                if (p >= m.count)
                    break;
                std::uint64_t const q = m.order ? m.order[p] : p;
                taylor_sums<GWN_PRECISION_PLAIN, false> acc;
                std::uint32_t n_tests = 0, n_accept = 0, n_leaf = 0;
                bool const overflow = taylor_quad_traverse<Order, GWN_PRECISION_PLAIN, false, 0>(
                    m.records, m.tris, static_cast<std::uint32_t>(ref_offset(m.root)), m.qx[q], m.qy[q], m.qz[q], beta2,
                    acc, n_tests, n_accept, n_leaf, s_quad, quads, cap);
                if ((threadIdx.x & 3u) == 0u)
                    acc.store(overflow, q, m.out, nullptr, nullptr, nullptr);
            }
            continue;
        }
        // Whole waves step through the chunk together, so the wave traversal sees uniform meshes.
        for (std::uint32_t t = threadIdx.x; t - (threadIdx.x & 63u) < chunk; t += blockDim.x) {
            std::uint64_t const p = base + t;
            bool const active = t < chunk && p < m.count;
            std::uint64_t const q = active ? (m.order ? m.order[p] : p) : 0;
            float const x = active ? m.qx[q] : 0.0f, y = active ? m.qy[q] : 0.0f, z = active ? m.qz[q] : 0.0f;
            taylor_sums<GWN_PRECISION_PLAIN, false> acc;
            bool overflow = false;
            if (ref_leaf(m.root)) {
                if (!active)
                    continue;
                std::uint64_t const off = ref_offset(m.root);
                std::uint32_t const cnt = ref_count(m.root);
                for (std::uint32_t k = 0; k < cnt; ++k)
                    acc.leaf(m.tris[off + k], x, y, z);
            } else if constexpr (Waves) {
                if (__ballot(active) == 0ull)
                    continue;
                std::uint32_t n_tests = 0, n_accept = 0, n_leaf = 0;
                overflow = taylor_wave_traverse<Order, GWN_PRECISION_PLAIN, false, false>(
                    m.records, m.tris, static_cast<std::uint32_t>(ref_offset(m.root)), active, x, y, z, beta2, acc,
                    n_tests, n_accept, n_leaf, s_node, s_mask, cap);
                if (!active)
                    continue;
            }
            acc.store(overflow, q, m.out, nullptr, nullptr, nullptr);
        }
    }
}

// Wave-cooperative traversal for spatially sorted queries.  The 64 lanes of a wave walk the union
// of their traversal paths together: the wave-uniform stack holds (node, lane mask) pairs, every
// node record is fetched once per wave from a wave-uniform address, and each lane only tests the
// children of nodes its own traversal reaches.  A lane's descended internal children are pushed
// and entered in the same slot / last-in-first-out order as in the per-lane kernel, so every lane
// forms its sum over exactly the same terms in exactly the same order; the stack depth is bounded
// by internal_stack_bound for the same reason.
// The wave-cooperative traversal of one wave's queries (lanes with `active`); s_node / s_mask are
// this wave's LDS stack.  The wave must hold at least one active lane.  Returns true on overflow.
// `records` are evaluation records for the value alone and traversal records with the gradient,
// as for the per-lane traversal.  The work tallies are kept where Count (three adds a slot otherwise).
template <int Order, int Prec, bool Grad, bool Count>
__device__ inline bool taylor_wave_traverse(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node, bool active,
    float x, float y, float z, float beta2, taylor_sums<Prec, Grad> &acc, std::uint32_t &n_tests,
    std::uint32_t &n_accept, std::uint32_t &n_leaf, std::uint32_t *s_node, std::uint64_t *s_mask, int cap
) {
    constexpr int RV = Grad ? moment_record_vec4(Order) : eval_record_vec4(Order);
    constexpr int B = eval_slot_floats(Order);
    std::uint64_t mask = __ballot(active);
    std::uint64_t const my_bit = 1ull << (threadIdx.x & 63);
    std::uint32_t node = root_node;
    int sp = 0;
    bool overflow = false;  // wave-uniform
    // In a vector register: a product of two scalar ones takes a move first, once per acceptance test.
    float scale2 = beta2;
    asm("" : "+v"(scale2));
    while (node != k_invalid && !overflow) {
        node = __builtin_amdgcn_readfirstlane(node);
        mask = uniform_u64(mask);
        float4 const *rec = records + static_cast<std::size_t>(node) * RV;
        float4 const refs = rec[0];
        float4 const mp = rec[1], px = rec[2], py = rec[3], pz = rec[4];
        float const *fields = reinterpret_cast<float const *>(rec + 1);
        std::uint32_t const cref[4] = {__float_as_uint(refs.x), __float_as_uint(refs.y),
                                       __float_as_uint(refs.z), __float_as_uint(refs.w)};
        float const mpd[4] = {mp.x, mp.y, mp.z, mp.w};
        float const cx[4] = {px.x, px.y, px.z, px.w};
        float const cy[4] = {py.x, py.y, py.z, py.w};
        float const cz[4] = {pz.x, pz.y, pz.z, pz.w};
        // All of the header at once: left to itself the compiler moves a slot's part past the check of the
        // slot's reference, a second wait on the node-to-node chain.
        asm volatile("" ::"s"(mp.x), "s"(mp.y), "s"(mp.z), "s"(mp.w), "s"(px.x), "s"(px.y), "s"(px.z), "s"(px.w),
                     "s"(py.x), "s"(py.y), "s"(py.z), "s"(py.w), "s"(pz.x), "s"(pz.y), "s"(pz.z), "s"(pz.w));
        [[maybe_unused]] bool const in = (mask & my_bit) != 0ull;
        std::uint32_t next = k_invalid;
        std::uint64_t next_mask = 0ull;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            std::uint32_t const c = __builtin_amdgcn_readfirstlane(cref[s]);
            if (c == k_invalid || overflow)
                continue;
            // Every lane tests and evaluates; the masks, in scalar registers, say whose result counts.
            // (Masked instructions issue no faster, and the branches' masks cost vector instructions.)
            constexpr int k_less = 4, k_less_equal = 5;  // ordered
            float const qrx = x - cx[s], qry = y - cy[s], qrz = z - cz[s];
            float const ql2 = squared_norm_unfused(qrx, qry, qrz);
            // A zero or NaN ql2 descends here or by the test on w below.
            std::uint64_t dmask = __builtin_amdgcn_fcmpf(ql2, product_unfused(mpd[s], scale2), k_less_equal) & mask;
            std::uint64_t const fmask = mask & ~dmask;
            if constexpr (Count)
                n_tests += in ? 1u : 0u;
            if (fmask != 0ull) {
                float g[3];
                float w;
                if constexpr (Grad)
                    w = taylor_term<Order, true>(fields, s, qrx, qry, qrz, ql2, g);
                else
                    w = taylor_value<Order>(reinterpret_cast<float const *>(rec + 5) + s * B, qrx, qry, qrz, ql2);
                std::uint64_t const amask = __builtin_amdgcn_fcmpf(fabsf(w), INFINITY, k_less) & fmask;
                dmask |= fmask & ~amask;
                // A lane without a term adds zero, which leaves its sum as it is (never -0).
                bool const accepted = __builtin_amdgcn_inverse_ballot_w64(amask);
                w = accepted ? w : 0.0f;
                if constexpr (Grad) {
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        g[k] = accepted ? g[k] : 0.0f;
                } else {
                    asm("" : "+v"(w));  // one select on the term, not two on its FP64 value
                }
                acc.far_term(w, g);
                if constexpr (Count)
                    n_accept += accepted ? 1u : 0u;
            }
            if (dmask == 0ull)
                continue;
            if (c & k_cref_leaf) {
                tri_record const t = tris[c & ~k_cref_leaf];
                if (__builtin_amdgcn_inverse_ballot_w64(dmask)) {
                    if constexpr (Count)
                        ++n_leaf;
                    acc.leaf(t, x, y, z);
                }
                continue;
            }
            if (next != k_invalid) {
                if (sp < cap) {
                    s_node[sp] = next;
                    s_mask[sp] = next_mask;
                    ++sp;
                } else {
                    overflow = true;
                }
            }
            next = c;
            next_mask = dmask;
        }
        if (next == k_invalid && sp > 0) {
            --sp;
            next = s_node[sp];
            next_mask = s_mask[sp];
        }
        node = next;
        mask = next_mask;
    }
    return overflow;
}

template <int Order, int Prec, bool Grad, int StackCap, bool Count>
__global__ __launch_bounds__(k_taylor_block) void taylor_wave_kernel(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node,
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, taylor_outputs o, std::size_t n, float beta2
) {
    constexpr int k_waves = k_taylor_block / 64;
    __shared__ std::uint32_t s_node[k_waves][StackCap];
    __shared__ std::uint64_t s_mask[k_waves][StackCap];
    int const wave = threadIdx.x >> 6;
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_taylor_block + threadIdx.x;
    bool const active = i < n;
    std::size_t const q = active ? (order ? order[i] : i) : 0;
    float const x = active ? qx[q] : 0.0f;
    float const y = active ? qy[q] : 0.0f;
    float const z = active ? qz[q] : 0.0f;
    if (__ballot(active) == 0ull)
        return;
    taylor_sums<Prec, Grad> acc;
    std::uint32_t n_tests = 0, n_accept = 0, n_leaf = 0;
    bool const overflow = taylor_wave_traverse<Order, Prec, Grad, Count>(
        records, tris, root_node, active, x, y, z, beta2, acc, n_tests, n_accept, n_leaf, s_node[wave], s_mask[wave],
        StackCap);
    if (!active)
        return;
    acc.store(overflow, q, o.out, o.gx, o.gy, o.gz);
    if constexpr (Count) {
        o.counters[3 * q + 0] = n_tests;
        o.counters[3 * q + 1] = n_accept;
        o.counters[3 * q + 2] = n_leaf;
    }
}

template <int Prec, bool Grad>
__global__ __launch_bounds__(256) void leaf_root_kernel(
    tri_record const *__restrict__ tris, std::uint64_t offset, std::uint32_t count,
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    taylor_outputs o, std::size_t n
) {
    std::size_t const q = static_cast<std::size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (q >= n)
        return;
    float const x = qx[q], y = qy[q], z = qz[q];
    taylor_sums<Prec, Grad> acc;
    for (std::uint32_t k = 0; k < count; ++k)
        acc.leaf(tris[offset + k], x, y, z);
    acc.store(false, q, o.out, o.gx, o.gy, o.gz);
    if (o.counters != nullptr) {
        o.counters[3 * q + 0] = 0;
        o.counters[3 * q + 1] = 0;
        o.counters[3 * q + 2] = count;
    }
}

// What one lane of a quad reads of a node: its slot's reference, acceptance fields and coefficients.
template <int Order, bool Grad> struct quad_slot {
    static constexpr int k_fields = moment_field_count(Order);
    static constexpr int k_block = eval_slot_floats(Order);
    std::uint32_t ref;
    float mp, cx, cy, cz;
    float c[Grad ? 4 * k_fields : k_block];  // Grad: field k at [4 k]

    __device__ static quad_slot load(float4 const *__restrict__ records, std::uint32_t node, int j) {
        constexpr int RV = Grad ? moment_record_vec4(Order) : eval_record_vec4(Order);
        float const *const w = reinterpret_cast<float const *>(records + static_cast<std::size_t>(node) * RV) + j;
        quad_slot s;
        s.ref = __float_as_uint(w[0]);
        s.mp = w[4];
        s.cx = w[8];
        s.cy = w[12];
        s.cz = w[16];
        if constexpr (Grad) {
#pragma unroll
            for (int k = 4; k < k_fields; ++k)
                s.c[4 * k] = w[4 + 4 * k];
        } else {
            float4 const *const b = reinterpret_cast<float4 const *>(w - j + 20 + j * k_block);
#pragma unroll
            for (int k = 0; k < k_block / 4; ++k) {
                float4 const v = b[k];
                s.c[4 * k] = v.x;
                s.c[4 * k + 1] = v.y;
                s.c[4 * k + 2] = v.z;
                s.c[4 * k + 3] = v.w;
            }
        }
        return s;
    }
};

// Adds the terms of a row's 16 lanes (or a quad's four) to the sum in lane order.
template <int Lanes> __device__ inline void ordered_add(float &sum, float v) { add_in_lane_order<Lanes>(sum, v); }
template <int Lanes, int J = 0> __device__ inline void ordered_add(double &sum, double v) {
    if constexpr (J < Lanes) {
        constexpr int k_ctrl = Lanes == 4 ? J * 0x55 : 0x150 + J;
        std::uint64_t const b = __builtin_bit_cast(std::uint64_t, v);
        std::uint32_t const lo = static_cast<std::uint32_t>(
            __builtin_amdgcn_update_dpp(0, static_cast<int>(b), k_ctrl, 0xf, 0xf, false));
        std::uint32_t const hi = static_cast<std::uint32_t>(
            __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), k_ctrl, 0xf, 0xf, false));
        sum += __builtin_bit_cast(double, (static_cast<std::uint64_t>(hi) << 32) | lo);
        ordered_add<Lanes, J + 1>(sum, v);
    }
}
template <int Lanes, int Prec, bool Grad>
__device__ inline void add_terms(taylor_sums<Prec, Grad> &acc, taylor_sums<Prec, Grad> const &term) {
    if constexpr (Prec == GWN_PRECISION_PLAIN) {
        ordered_add<Lanes>(acc.omega, term.omega);
        if constexpr (Grad) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
                ordered_add<Lanes>(acc.gf[k], term.gf[k]);
        }
    } else {
        ordered_add<Lanes>(acc.near, term.near);
        if constexpr (Grad) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
                ordered_add<Lanes>(acc.gd[k], term.gd[k]);
        }
    }
}

// One query's decisions at one child slot.
template <int Order, bool Grad> struct slot_test {
    float w;
    float g[3];
    bool valid, accepted, leaf, inner;

    __device__ slot_test(quad_slot<Order, Grad> const &slot, float x, float y, float z, float beta2, bool held) {
        float const qrx = x - slot.cx, qry = y - slot.cy, qrz = z - slot.cz;
        float const ql2 = squared_norm_unfused(qrx, qry, qrz);
        bool const far = !(!(ql2 > 0.0f) || ql2 <= product_unfused(slot.mp, beta2));
        if constexpr (Grad)
            w = taylor_term<Order, true>(slot.c, 0, qrx, qry, qrz, ql2, g);
        else
            w = taylor_value<Order>(slot.c, qrx, qry, qrz, ql2);
        valid = held && slot.ref != k_invalid;
        accepted = valid && far && isfinite(w);
        leaf = valid && !accepted && (slot.ref & k_cref_leaf) != 0u;
        inner = valid && !accepted && (slot.ref & k_cref_leaf) == 0u;
    }
};

// Taylor traversal with four lanes per query, lane j of the quad owning child slot j: the four
// acceptance tests, expansions and leaf triangles of a node are evaluated side by side and their terms
// added in slot order (add_terms; a slot without a term adds zero, which leaves every sum as it is, since
// a sum starts at +0 and never becomes -0); descended children are pushed in slot order and the last one
// entered, as taylor_traverse does.  Decisions, terms and the order of every sum are those of the per-lane
// traversal, so the results are too, bit for bit.  The stack is the quad's column of an LDS array, of StackCap
// entries or, with StackCap 0, of `cap`.
//
// A chain of dependent node reads per query: one lane per query waited for the header, then for each
// accepted slot's coefficients and each leaf's triangle in turn (about eight waits a node); here a node's
// header and all four slots' coefficients arrive together, and the next node's are requested as soon as
// the decisions are known, before the leaf triangles are evaluated.  Measured (sort included), the wave
// traversal against this form: 500,009 queries of 131,072 triangles (order 2, scale 2) 1.80 / 1.05 ms;
// unsorted, one lane per query against this form: 262,144 of 131,072 2.26 / 1.38 ms.
// Tried and slower: holding a quad's leaf triangles back until half of the wave's quads have some, so that
// they are evaluated with more lanes active (5-20 %); handing a finished quad another query of the wave
// (15-70 %: a wave's queries are then no longer neighbours, and their reads no longer shared).
template <int Order, int Prec, bool Grad, int StackCap>
__device__ inline bool taylor_quad_traverse(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node, float x, float y,
    float z, float beta2, taylor_sums<Prec, Grad> &acc, std::uint32_t &n_tests, std::uint32_t &n_accept,
    std::uint32_t &n_leaf, std::uint32_t *stack, int stride, int cap
) {
    using slot_type = quad_slot<Order, Grad>;
    int const limit = StackCap != 0 ? StackCap : cap;
    int const j = static_cast<int>(threadIdx.x & 3);
    int const shift = static_cast<int>(threadIdx.x & 60);
    int sp = 0;
    bool overflow = false;
    bool live = true;
    slot_type slot = slot_type::load(records, root_node, j);
    while (live) {
        slot_test<Order, Grad> const v(slot, x, y, z, beta2, true);
        std::uint32_t const c = slot.ref;
        n_tests += v.valid ? 1u : 0u;
        n_accept += v.accepted ? 1u : 0u;
        n_leaf += v.leaf ? 1u : 0u;
        // The node's triangles, requested before the next node.
        tri_record t{};
        if (__ballot(v.leaf) != 0ull)
            t = tris[v.leaf ? (c & ~k_cref_leaf) : 0u];
        // The last descended internal child is entered, the others are pushed in slot order.
        std::uint32_t const bits = static_cast<std::uint32_t>(__ballot(v.inner) >> shift) & 15u;
        std::uint32_t const c0 = quad_bcast<0>(c), c1 = quad_bcast<1>(c), c2 = quad_bcast<2>(c), c3 = quad_bcast<3>(c);
        int const pushed = __popc(bits) - 1;
        std::uint32_t next = bits & 8u ? c3 : (bits & 4u ? c2 : (bits & 2u ? c1 : c0));
        int const at = sp + __popc(bits & ((1u << j) - 1u));
        if (v.inner && (bits >> j) != 1u && at < limit)
            stack[at * stride] = c;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (pushed >= 0) {
            sp += pushed;
            overflow = sp > limit;
            live = !overflow;
        } else if (sp > 0) {
            next = stack[--sp * stride];
        } else {
            live = false;
        }
        slot = slot_type::load(records, live ? next : root_node, j);
        taylor_sums<Prec, Grad> term;
        if (v.accepted)
            term.far_term(v.w, v.g);
        if (v.leaf)
            term.leaf(t, x, y, z);
        add_terms<4>(acc, term);
    }
    return overflow;
}

template <int Order, int Prec, bool Grad, int StackCap>
__global__ __launch_bounds__(k_taylor_block) void taylor_quad_kernel(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node,
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, taylor_outputs o, std::size_t n, float beta2
) {
    constexpr int k_quads = k_taylor_block / 4;
    __shared__ std::uint32_t s_stack[StackCap * k_quads];  // entry e of quad k at [e * k_quads + k]
    std::size_t const i = (static_cast<std::size_t>(blockIdx.x) * k_taylor_block + threadIdx.x) >> 2;
    if (i >= n)
        return;  // whole quads
    int const j = static_cast<int>(threadIdx.x & 3);
    std::size_t const q = order ? order[i] : i;
    taylor_sums<Prec, Grad> acc;
    std::uint32_t n_tests = 0, n_accept = 0, n_leaf = 0;  // this lane's
    bool const overflow = taylor_quad_traverse<Order, Prec, Grad, StackCap>(
        records, tris, root_node, qx[q], qy[q], qz[q], beta2, acc, n_tests, n_accept, n_leaf,
        s_stack + (threadIdx.x >> 2), k_quads, StackCap);
    if (j == 0)
        acc.store(overflow, q, o.out, o.gx, o.gy, o.gz);
    if (o.counters != nullptr) {
        n_tests = quad_sum(n_tests);
        n_accept = quad_sum(n_accept);
        n_leaf = quad_sum(n_leaf);
        if (j == 0) {
            o.counters[3 * q + 0] = n_tests;
            o.counters[3 * q + 1] = n_accept;
            o.counters[3 * q + 2] = n_leaf;
        }
    }
}

// The quad traversal with a row of 16 lanes per query: quad g tests the g-th entry from the top of the
// stack.  Entries are settled in stack order up to the first whose node has children to descend into, and
// those are pushed (what the quads behind it found is dropped, their entries stay on the stack), so nodes
// take effect and terms are added in the quad traversal's order.  Most nodes of a traversal have no
// children to descend into, so a row settles two to four at a time.
template <int Order, int Prec, bool Grad, int StackCap>
__global__ __launch_bounds__(k_taylor_block) void taylor_row_kernel(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node,
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    std::uint32_t const *__restrict__ order, taylor_outputs o, std::size_t n, float beta2
) {
    using slot_type = quad_slot<Order, Grad>;
    constexpr int k_rows = k_taylor_block / 16;
    // Entry e of row k at [e * k_rows + k]; the entered node is on the stack too.
    __shared__ std::uint32_t s_stack[(StackCap + 1) * k_rows];
    std::size_t const i = (static_cast<std::size_t>(blockIdx.x) * k_taylor_block + threadIdx.x) >> 4;
    if (i >= n)
        return;  // whole rows
    std::uint32_t const lane = threadIdx.x & 15u;
    int const j = static_cast<int>(lane & 3u);
    std::uint32_t const g = lane >> 2;
    std::uint32_t const shift = threadIdx.x & 48u;
    std::uint32_t *const stack = s_stack + (threadIdx.x >> 4);
    std::size_t const q = order ? order[i] : i;
    float const x = qx[q], y = qy[q], z = qz[q];
    taylor_sums<Prec, Grad> acc;
    std::uint32_t n_tests = 0, n_accept = 0, n_leaf = 0;  // this lane's
    bool overflow = false;
    bool live = true;
    int sp = 1;
    bool held = g == 0u;
    if (held)
        stack[0] = root_node;
    slot_type slot = slot_type::load(records, root_node, j);
    while (live) {
        slot_test<Order, Grad> const v(slot, x, y, z, beta2, held);
        std::uint32_t const c = slot.ref;
        std::uint32_t const inners = static_cast<std::uint32_t>(__ballot(v.inner) >> shift) & 0xffffu;
        std::uint32_t const last = inners != 0u ? static_cast<std::uint32_t>(__builtin_ctz(inners)) >> 2 : 3u;
        bool const settled = g <= last;
        bool const leaf = v.leaf && settled;
        n_tests += v.valid && settled ? 1u : 0u;
        n_accept += v.accepted && settled ? 1u : 0u;
        n_leaf += leaf ? 1u : 0u;
        tri_record t{};
        if (__ballot(leaf) != 0ull)
            t = tris[leaf ? (c & ~k_cref_leaf) : 0u];
        sp = sp > static_cast<int>(last) + 1 ? sp - static_cast<int>(last) - 1 : 0;
        std::uint32_t const bits = (inners >> (4u * last)) & 15u;  // zero without one
        int const at = sp + __popc(bits & ((1u << j) - 1u));
        if (v.inner && g == last && at <= StackCap)
            stack[at * k_rows] = c;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        sp += __popc(bits);
        overflow = sp > StackCap + 1;
        live = sp > 0 && !overflow;
        int const e = sp - 1 - static_cast<int>(g);
        held = live && e >= 0;
        slot = slot_type::load(records, held ? stack[e * k_rows] : root_node, j);
        taylor_sums<Prec, Grad> term;
        if (v.accepted && settled)
            term.far_term(v.w, v.g);
        if (leaf)
            term.leaf(t, x, y, z);
        add_terms<16>(acc, term);
    }
    if (lane == 0u)
        acc.store(overflow, q, o.out, o.gx, o.gy, o.gz);
    if (o.counters != nullptr) {
        n_tests = row_sum(n_tests);
        n_accept = row_sum(n_accept);
        n_leaf = row_sum(n_leaf);
        if (lane == 0u) {
            o.counters[3 * q + 0] = n_tests;
            o.counters[3 * q + 1] = n_accept;
            o.counters[3 * q + 2] = n_leaf;
        }
    }
}

// Up to this many queries each has a row: the chip is not full, and the batch lasts as long as its longest
// query.  Measured, a row against a quad per query, sort included, order 2, scale 2: 1,000 of 5,120 triangles
// 109 / 171 us, 20,000 of 500 99 / 114, 65,536 of 500 149 / 130, of 5,120 200 / 198, of 131,072 337 / 506, of
// 1,048,576 0.67 / 1.23 ms; 131,072 of 5,120 287 / 252 us, of 131,072 453 / 552, of 1,048,576 0.77 / 1.30 ms; 262,144
// of 5,120 467 / 355 us, of 131,072 703 / 672, of 1,048,576 0.97 / 1.46 ms; split, scale 6.25: 65,536 of 5,120 0.95 /
// 0.78 ms, of 131,072 1.81 / 1.90, 262,144 of 131,072 4.6 / 3.8, of 1,048,576 6.5 / 6.9.  So the crossing rises with
// the triangles, from some 40,000 queries at 500 to more than 262,144 at 1,048,576; one line in the middle.
constexpr std::size_t k_row_queries = std::size_t(1) << 16;

// Reciprocal square root and reciprocal in FP64 from the hardware approximations and Newton
// steps (relative error at FP64 rounding level, not correctly rounded).  x > 0 / x != 0.
__device__ inline double rsq_f64_fast(double x) {
    double r = __builtin_amdgcn_rsq(x);
    double const h = 0.5 * x;
    r = r * fma(-h * r, r, 1.5);
    r = r * fma(-h * r, r, 1.5);
    return r;
}
__device__ inline double rcp_f64_fast(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    r = fma(r, fma(-x, r, 1.0), r);
    return r;
}
__device__ inline double rsq_fast(double x) { return rsq_f64_fast(x); }
__device__ inline float rsq_fast(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ inline double rcp_fast(double x) { return rcp_f64_fast(x); }
__device__ inline float rcp_fast(float x) { return __builtin_amdgcn_rcpf(x); }

// Derivatives of one triangle's solid angle W(a, b, c) seen from the origin of a, b, c (vertices
// relative to the query), from the unnormalised form W = 2 atan2(a.(b x c), D) with
// D = |a||b||c| + (a.b)|c| + (a.c)|b| + (b.c)|a| (equal to the Van Oosterom-Strackee quotient
// scaled by |a||b||c|):  dW = 2 (D dnum - num dD) / (num^2 + D^2).  Zero where W is defined as 0.
template <class R>
__device__ inline void solid_angle_vertex_grad(
    R const (&a)[3], R const (&b)[3], R const (&c)[3], R (&da)[3], R (&db)[3], R (&dc)[3]
) {
#pragma unroll
    for (int k = 0; k < 3; ++k)
        da[k] = db[k] = dc[k] = R(0);
    R const aa = a[0] * a[0] + a[1] * a[1] + a[2] * a[2];
    R const bb = b[0] * b[0] + b[1] * b[1] + b[2] * b[2];
    R const cc = c[0] * c[0] + c[1] * c[1] + c[2] * c[2];
    if (aa == R(0) || bb == R(0) || cc == R(0))
        return;
    R const ia = rsq_fast(aa), ib = rsq_fast(bb), ic = rsq_fast(cc);
    R const la = aa * ia, lb = bb * ib, lc = cc * ic;
    R const bc[3] = {b[1] * c[2] - b[2] * c[1], b[2] * c[0] - b[0] * c[2], b[0] * c[1] - b[1] * c[0]};
    R const ca[3] = {c[1] * a[2] - c[2] * a[1], c[2] * a[0] - c[0] * a[2], c[0] * a[1] - c[1] * a[0]};
    R const ab[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
    R const num = a[0] * bc[0] + a[1] * bc[1] + a[2] * bc[2];
    if (num == R(0))
        return;
    R const dab = a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
    R const dac = a[0] * c[0] + a[1] * c[1] + a[2] * c[2];
    R const dbc = b[0] * c[0] + b[1] * c[1] + b[2] * c[2];
    R const den = la * lb * lc + dab * lc + dac * lb + dbc * la;
    R const sc = R(2) * rcp_fast(num * num + den * den);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        R const ha = a[k] * ia, hb = b[k] * ib, hc = c[k] * ic;
        R const dDa = ha * lb * lc + b[k] * lc + c[k] * lb + dbc * ha;
        R const dDb = hb * la * lc + a[k] * lc + c[k] * la + dac * hb;
        R const dDc = hc * la * lb + a[k] * lb + b[k] * la + dab * hc;
        da[k] = sc * (den * bc[k] - num * dDa);
        db[k] = sc * (den * ca[k] - num * dDb);
        dc[k] = sc * (den * ab[k] - num * dDc);
    }
}

// u * dW/d(a, b, c) of one descended triangle into t9 (9 floats) and -(da + db + dc) * u into dq.
// Split like the forward's precision split: within about four edge lengths (where the terms are
// ~1/d^2, cancel between neighbouring triangles and lose ~|a|/d of their FP32 digits) in FP64 from
// exact differences of the float vertices and query; beyond it in FP32.
__device__ inline void adjoint_leaf_terms(
    tri_record const &t, float x, float y, float z, double sud, float (&t9)[9], double (&dq)[3]
) {
    float const e1x = t.v1x - t.v0x, e1y = t.v1y - t.v0y, e1z = t.v1z - t.v0z;
    float const e2x = t.v2x - t.v0x, e2y = t.v2y - t.v0y, e2z = t.v2z - t.v0z;
    float const ax = t.v0x - x, ay = t.v0y - y, az = t.v0z - z;
    float const le1 = squared_norm_unfused(e1x, e1y, e1z);
    float const le2 = squared_norm_unfused(e2x, e2y, e2z);
    float const dq2 = squared_norm_unfused(ax, ay, az);
    if (!(dq2 > product_unfused(k_split_near_scale2, fmaxf(le1, le2)))) {
        double const qd[3] = {x, y, z};
        double const a[3] = {double(t.v0x) - qd[0], double(t.v0y) - qd[1], double(t.v0z) - qd[2]};
        double const b[3] = {double(t.v1x) - qd[0], double(t.v1y) - qd[1], double(t.v1z) - qd[2]};
        double const c[3] = {double(t.v2x) - qd[0], double(t.v2y) - qd[1], double(t.v2z) - qd[2]};
        double da[3], db[3], dc[3];
        solid_angle_vertex_grad<double>(a, b, c, da, db, dc);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            t9[k] = static_cast<float>(sud * da[k]);
            t9[3 + k] = static_cast<float>(sud * db[k]);
            t9[6 + k] = static_cast<float>(sud * dc[k]);
            dq[k] -= sud * (da[k] + db[k] + dc[k]);
        }
    } else {
        float const a[3] = {ax, ay, az};
        float const b[3] = {t.v1x - x, t.v1y - y, t.v1z - z};
        float const c[3] = {t.v2x - x, t.v2y - y, t.v2z - z};
        float da[3], db[3], dc[3];
        solid_angle_vertex_grad<float>(a, b, c, da, db, dc);
        float const su = static_cast<float>(sud);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            t9[k] = su * da[k];
            t9[3 + k] = su * db[k];
            t9[6 + k] = su * dc[k];
            dq[k] -= sud * double(da[k] + db[k] + dc[k]);
        }
    }
}

// Adds one descended triangle's adjoint to its record's 9 entries and its query part to dq.
__device__ inline void adjoint_leaf(
    tri_record const &t, std::size_t rec, float x, float y, float z, double sud, float *__restrict__ dtri,
    double (&dq)[3]
) {
    float t9[9];
    adjoint_leaf_terms(t, x, y, z, sud, t9, dq);
    float *d = dtri + rec * 9;
#pragma unroll
    for (int k = 0; k < 9; ++k)
        atomicAdd(d + k, t9[k]);
}

// Adjoint of sum_q u_q w_q (orders 0, 1): the per-lane traversal (taylor_traverse) with the same
// accept/descend decisions.  An accepted child adds u/(4 pi) (dw/dP, dw/dN, dw/dT) to its slot's
// 12 entries (dw/dP = -dw/dq); a near triangle adds u/(4 pi) dW/d(a, b, c) to its record's 9
// entries; the query gradient goes to dq.  root_node = k_invalid evaluates the leaf root instead.
template <int Order, int StackCap>
__global__ __launch_bounds__(k_taylor_block) void taylor_adjoint_kernel(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node,
    std::uint64_t root_leaf, float const *__restrict__ qx, float const *__restrict__ qy,
    float const *__restrict__ qz, float const *__restrict__ u, std::uint32_t const *__restrict__ order,
    std::size_t n, float beta2, float *__restrict__ dslot, float *__restrict__ dtri, float *__restrict__ dqx,
    float *__restrict__ dqy, float *__restrict__ dqz
) {
    static_assert(Order <= 1, "adjoint orders are 0 and 1");
    constexpr int RV = moment_record_vec4(Order);
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_taylor_block + threadIdx.x;
    if (i >= n)
        return;
    std::size_t const q = order ? order[i] : i;
    float const x = qx[q], y = qy[q], z = qz[q];
    float const su = u[q] * k_inv_4pi_f;
    double const sud = double(u[q]) * (1.0 / (4.0 * k_pi_d));
    double dq[3] = {0.0, 0.0, 0.0};  // FP64 per-query sum of the far and near parts
    if (root_node == k_invalid) {
        std::uint64_t const off = ref_offset(root_leaf);
        std::uint32_t const cnt = ref_count(root_leaf);
        for (std::uint32_t k = 0; k < cnt; ++k)
            adjoint_leaf(tris[off + k], off + k, x, y, z, sud, dtri, dq);
    } else {
        std::uint32_t stack[StackCap];
        int sp = 0;
        bool overflow = false;
        std::uint32_t node = root_node;
        while (node != k_invalid && !overflow) {
            float4 const *rec = records + static_cast<std::size_t>(node) * RV;
            float4 const refs = rec[0];
            float4 const mp = rec[1], px = rec[2], py = rec[3], pz = rec[4];
            float const *fields = reinterpret_cast<float const *>(rec + 1);
            std::uint32_t const cref[4] = {__float_as_uint(refs.x), __float_as_uint(refs.y),
                                           __float_as_uint(refs.z), __float_as_uint(refs.w)};
            float const mpd[4] = {mp.x, mp.y, mp.z, mp.w};
            float const cx[4] = {px.x, px.y, px.z, px.w};
            float const cy[4] = {py.x, py.y, py.z, py.w};
            float const cz[4] = {pz.x, pz.y, pz.z, pz.w};
            std::uint32_t next = k_invalid;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                std::uint32_t const c = cref[s];
                if (c == k_invalid || overflow)
                    continue;
                float const qrx = x - cx[s], qry = y - cy[s], qrz = z - cz[s];
                float const ql2 = squared_norm_unfused(qrx, qry, qrz);
                bool const descend = !(ql2 > 0.0f) || ql2 <= product_unfused(mpd[s], beta2);
                if (!descend) {
                    float g[3];
                    float const w = taylor_term<Order, true>(fields, s, qrx, qry, qrz, ql2, g);
                    if (isfinite(w)) {
                        float const m1 = __builtin_amdgcn_rsqf(ql2);
                        float const m2 = m1 * m1;
                        float const qn[3] = {qrx * m1, qry * m1, qrz * m1};
                        float *d = dslot + (static_cast<std::size_t>(node) * 4 + s) * 12;
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            atomicAdd(d + k, -su * g[k]);
                            atomicAdd(d + 3 + k, -su * m2 * qn[k]);
                            dq[k] += double(su * g[k]);
                        }
                        if constexpr (Order >= 1) {
                            float const m3 = m2 * m1;
                            atomicAdd(d + 6, su * m3 * (1.0f - 3.0f * qn[0] * qn[0]));
                            atomicAdd(d + 7, su * m3 * (1.0f - 3.0f * qn[1] * qn[1]));
                            atomicAdd(d + 8, su * m3 * (1.0f - 3.0f * qn[2] * qn[2]));
                            atomicAdd(d + 9, -3.0f * su * m3 * qn[0] * qn[1]);
                            atomicAdd(d + 10, -3.0f * su * m3 * qn[1] * qn[2]);
                            atomicAdd(d + 11, -3.0f * su * m3 * qn[2] * qn[0]);
                        }
                        continue;
                    }
                }
                if (c & k_cref_leaf) {
                    std::uint32_t const r = c & ~k_cref_leaf;
                    adjoint_leaf(tris[r], r, x, y, z, sud, dtri, dq);
                    continue;
                }
                if (next != k_invalid) {
                    if (sp < StackCap)
                        stack[sp++] = next;
                    else
                        overflow = true;
                }
                next = c;
            }
            if (next == k_invalid && sp > 0)
                next = stack[--sp];
            node = next;
        }
        if (overflow)
            dq[0] = dq[1] = dq[2] = __builtin_nan("");
    }
    if (dqx != nullptr) {
        dqx[q] = static_cast<float>(dq[0]);
        dqy[q] = static_cast<float>(dq[1]);
        dqz[q] = static_cast<float>(dq[2]);
    }
}

// Whether Hilbert-ordered queries are dense enough for 64 of them to walk the tree together.  The wave
// traversal does little per query, but its time does not fall below that of its longest wave, whose
// union of paths grows with the square root of the triangles near it and with beta; the quad
// traversal's time is proportional to the queries.  Measured (MI355X, mixed queries, sort included),
// wave against quad, order 2:
//   beta 2:    500 triangles, 131k queries 181 / 167 us, 262k 205 / 240; 5,120, 262k 391 / 355, 1M 559 / 881;
//              131,072, 1M 1.54 / 1.37 ms, 4M 2.41 / 4.15; 1,048,576, 1M 3.99 / 2.12, 4M 4.86 / 4.75
//   beta 6.25 (split): 2,000, 131k 884 / 959 us; 5,120, 131k 1.21 / 1.21 ms, 262k 1.47 / 1.93; 131,072, 262k
//              4.23 / 3.82 ms, 1M 6.39 / 9.66; 1,048,576, 262k 12.0 / 6.9, 1M 12.8 / 14.1
// The crossings lie near 4500 sqrt(triangles) (2 / beta)^1.5, for few triangles above it.
bool dense_queries(std::size_t triangles, std::size_t n, float beta2) {
    double const beta = std::sqrt(std::max(1.0, double(beta2)));
    return double(n) >= 4500.0 * std::sqrt(double(triangles)) * std::pow(2.0 / beta, 1.5);
}

// Whether a single batch takes whole waves.  Dense queries, but below 100,000 of them only where the tree is tiny:
// elsewhere a row or a quad per query is the faster form there (wave against row, beta 6.25: 65,536 queries of 350
// triangles 304 / 447 us, of 2,000 878 / 781, of 5,120 1,300 / 949).  And, in any order of the queries, trees so tiny
// for their beta that a query descends most of them anyway (unsorted, wave against row or quad: beta 2, 65,536 of
// 12 triangles 21 / 32 us, of 50 52 / 53, 1,000,003 of 50 197 / 402, of 200 779 / 671; beta 6.25, 65,536 of 200
// 177 / 277, of 500 454 / 391, 1,000,003 of 500 2.64 / 4.74 ms, of 2,000 9.6 / 8.0; 20,000 of 50 36 / 31 us).
bool whole_waves(std::size_t triangles, std::size_t n, float beta2, bool sorted) {
    double const scale = std::max(1.0, double(beta2));
    bool const tiny = double(triangles) <= 25.0 * scale;
    return (tiny && double(n) >= 32768.0 + 4000.0 * double(triangles) / scale) ||
           (sorted && (tiny || n >= 100000) && dense_queries(triangles, n, beta2));
}

// The outputs of the queries from `at` on.
inline taylor_outputs outputs_from(taylor_outputs o, std::size_t at) {
    for (float **p : {&o.out, &o.gx, &o.gy, &o.gz})
        *p = *p != nullptr ? *p + at : nullptr;
    o.counters = o.counters != nullptr ? o.counters + 3 * at : nullptr;
    return o;
}

template <int Order, int Prec, bool Grad, int Cap>
void launch_taylor_cap(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy,
    float const *qz, std::uint32_t const *order, taylor_outputs const &o, std::size_t n, float beta2,
    hipStream_t stream
) {
    std::uint32_t const root = static_cast<std::uint32_t>(ref_offset(bvh.root.reference));
    // The value alone reads the evaluation records; the gradient the traversal records.
    float4 const *records = Grad ? m.records.ptr : m.eval_records.ptr;
    if (whole_waves(bvh.triangle_count, n, beta2, order != nullptr)) {
        // Neighbouring lanes share most of their paths.  VALU bound:
        // 16,777,216 queries of 1,048,576 triangles (order 2, split, scale 6.25) took 69.0 ms with 189,111
        // instructions a wave, 59.5 ms with the 166,216 of unmasked tests and terms, tallies on demand only
        // and half_angle_far.
        if (o.counters != nullptr)
            taylor_wave_kernel<Order, Prec, Grad, Cap, true><<<grid_for(n, k_taylor_block), k_taylor_block, 0, stream>>>(
                records, bvh.triangles.ptr, root, qx, qy, qz, order, o, n, beta2
            );
        else
            taylor_wave_kernel<Order, Prec, Grad, Cap, false><<<grid_for(n, k_taylor_block), k_taylor_block, 0, stream>>>(
                records, bvh.triangles.ptr, root, qx, qy, qz, order, o, n, beta2
            );
    } else if (n <= k_row_queries) {
        taylor_row_kernel<Order, Prec, Grad, Cap><<<grid_for(16 * n, k_taylor_block), k_taylor_block, 0, stream>>>(
            records, bvh.triangles.ptr, root, qx, qy, qz, order, o, n, beta2
        );
    } else {
        for_each_slice(n, k_quad_slice, [&](std::size_t first, std::size_t count) {
            // With an order its entries say where a query lies, without one it lies at its own place.
            std::size_t const at = order != nullptr ? 0 : first;
            taylor_quad_kernel<Order, Prec, Grad, Cap><<<grid_for(4 * count, k_taylor_block), k_taylor_block, 0, stream>>>(
                records, bvh.triangles.ptr, root, qx + at, qy + at, qz + at, order != nullptr ? order + first : nullptr,
                outputs_from(o, at), count, beta2
            );
        });
    }
    GWN_LAUNCH_CHECK();
}

template <int Order, int Prec, bool Grad>
void launch_taylor(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy,
    float const *qz, std::uint32_t const *order, taylor_outputs const &o, std::size_t n, float beta2,
    hipStream_t stream
) {
    // The stack only ever holds internal_stack_bound entries; the smallest compiled capacity that
    // covers the bound keeps the LDS / register footprint small.
    int const need = static_cast<int>(bvh.internal_stack_bound);
    if (need <= 32)
        launch_taylor_cap<Order, Prec, Grad, 32>(bvh, m, qx, qy, qz, order, o, n, beta2, stream);
    else if (need <= 64)
        launch_taylor_cap<Order, Prec, Grad, 64>(bvh, m, qx, qy, qz, order, o, n, beta2, stream);
    else if (need <= 128)
        launch_taylor_cap<Order, Prec, Grad, 128>(bvh, m, qx, qy, qz, order, o, n, beta2, stream);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
}


template <int Ctrl, int RowMask>
__device__ inline float dpp_f32(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), Ctrl, RowMask, 0xf, false));
}

// The two results of a v_permlane{16,32}_swap, forced into registers before use: summing them
// straight from the builtin's pair, hipcc (ROCm 7.2) emitted `v_add_f32 vA, vA, vA` -- the first
// result twice -- after the swap; the empty asm keeps both operands distinct.
__device__ inline float swap_pair_sum(int x, int y) {
    asm volatile("" : "+v"(x), "+v"(y));
    return __builtin_bit_cast(float, x) + __builtin_bit_cast(float, y);
}

// Wave totals of 12 per-lane values with a transposing butterfly (gfx950): v_permlane32_swap adds
// the upper half-wave of value k + 6 to the lower half of value k (and the reverse), leaving value k
// in lanes 0-31 and k + 6 in lanes 32-63; v_permlane16_swap does the same between the rows of each
// half; DPP then sums within each 16-lane row.  On return every lane of row r (lanes 16r..16r+15)
// holds in out[k] the wave total of value k + 3r.  About 30 VALU operations instead of 12 DPP
// reductions (84).  Every lane must be active.
__device__ inline void wave_sum12(float const (&f)[12], float (&out)[3]) {
    float g[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        auto const p = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(int, f[k]),
                                                        __builtin_bit_cast(int, f[k + 6]), false, false);
        g[k] = swap_pair_sum(p[0], p[1]);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        auto const p = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(int, g[k]),
                                                        __builtin_bit_cast(int, g[k + 3]), false, false);
        float h = swap_pair_sum(p[0], p[1]);
        h += dpp_f32<0xb1, 0xf>(h);   // quad_perm [1, 0, 3, 2]
        h += dpp_f32<0x4e, 0xf>(h);   // quad_perm [2, 3, 0, 1]
        h += dpp_f32<0x141, 0xf>(h);  // row_half_mirror
        h += dpp_f32<0x140, 0xf>(h);  // row_mirror
        out[k] = h;
    }
}

// Adds the wave's per-lane values f[0..F) (F <= 12) into d[0..F): wave totals from wave_sum12, then
// one atomic instruction whose active lanes 16r + k (k < 3) add total k + 3r, so the F adds of a
// call go to F consecutive floats in one request.  A lone contributing lane goes the same way (its
// values plus zeros are its values exactly): one request instead of F.
template <int F>
__device__ inline void wave_atomic_add(float *__restrict__ d, float const (&f)[F]) {
    static_assert(F <= 12, "at most 12 values per wave sum");
    float v[12];
#pragma unroll
    for (int k = 0; k < 12; ++k)
        v[k] = k < F ? f[k] : 0.0f;
    float out[3];
    wave_sum12(v, out);
    int const lane = threadIdx.x & 63;
    int const k = lane & 15;
    int const idx = k + 3 * (lane >> 4);
    if (k < 3 && idx < F)
        atomicAdd(d + idx, k == 0 ? out[0] : (k == 1 ? out[1] : out[2]));
}

// The adjoint of taylor_adjoint_kernel, wave-cooperative: a wave walks the tree once for its 64
// (Hilbert-ordered) queries with the same per-query accept/descend decisions, and the field and
// vertex adjoints of a child slot or near triangle are summed over the wave and added with one
// atomic instruction over consecutive floats, instead of every query adding its own (the top
// slots are shared by every query, so per-query atomics serialise on them).
template <int Order, int StackCap>
__global__ __launch_bounds__(k_taylor_block) void taylor_adjoint_wave_kernel(
    float4 const *__restrict__ records, tri_record const *__restrict__ tris, std::uint32_t root_node,
    float const *__restrict__ qx, float const *__restrict__ qy, float const *__restrict__ qz,
    float const *__restrict__ u, std::uint32_t const *__restrict__ order, std::size_t n, float beta2,
    float *__restrict__ dslot, float *__restrict__ dtri, float *__restrict__ dqx, float *__restrict__ dqy,
    float *__restrict__ dqz
) {
    static_assert(Order <= 1, "adjoint orders are 0 and 1");
    constexpr int RV = moment_record_vec4(Order);
    constexpr int F = Order >= 1 ? 12 : 6;
    constexpr int k_waves = k_taylor_block / 64;
    __shared__ std::uint32_t s_node[k_waves][StackCap];
    __shared__ std::uint64_t s_mask[k_waves][StackCap];
    int const wave = threadIdx.x >> 6;
    int const lane = threadIdx.x & 63;
    std::size_t const i = static_cast<std::size_t>(blockIdx.x) * k_taylor_block + threadIdx.x;
    bool const active = i < n;
    std::size_t const q = active ? (order ? order[i] : i) : 0;
    float const x = active ? qx[q] : 0.0f;
    float const y = active ? qy[q] : 0.0f;
    float const z = active ? qz[q] : 0.0f;
    float const su = active ? u[q] * k_inv_4pi_f : 0.0f;
    double const sud = active ? double(u[q]) * (1.0 / (4.0 * k_pi_d)) : 0.0;
    std::uint64_t mask = __ballot(active);
    if (mask == 0ull)
        return;
    std::uint64_t const my_bit = 1ull << lane;
    double dq[3] = {0.0, 0.0, 0.0};
    std::uint32_t node = root_node;
    int sp = 0;
    bool overflow = false;  // wave-uniform
    while (node != k_invalid && !overflow) {
        node = __builtin_amdgcn_readfirstlane(node);
        float4 const *rec = records + static_cast<std::size_t>(node) * RV;
        float4 const refs = rec[0];
        float4 const mp = rec[1], px = rec[2], py = rec[3], pz = rec[4];
        float const *fields = reinterpret_cast<float const *>(rec + 1);
        std::uint32_t const cref[4] = {__float_as_uint(refs.x), __float_as_uint(refs.y),
                                       __float_as_uint(refs.z), __float_as_uint(refs.w)};
        float const mpd[4] = {mp.x, mp.y, mp.z, mp.w};
        float const cx[4] = {px.x, px.y, px.z, px.w};
        float const cy[4] = {py.x, py.y, py.z, py.w};
        float const cz[4] = {pz.x, pz.y, pz.z, pz.w};
        bool const in = (mask & my_bit) != 0ull;
        std::uint32_t next = k_invalid;
        std::uint64_t next_mask = 0ull;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            std::uint32_t const c = __builtin_amdgcn_readfirstlane(cref[s]);
            if (c == k_invalid || overflow)
                continue;
            bool descend = false, accepted = false;
            float f[F];
#pragma unroll
            for (int k = 0; k < F; ++k)
                f[k] = 0.0f;
            if (in) {
                float const qrx = x - cx[s], qry = y - cy[s], qrz = z - cz[s];
                float const ql2 = squared_norm_unfused(qrx, qry, qrz);
                descend = !(ql2 > 0.0f) || ql2 <= product_unfused(mpd[s], beta2);
                if (!descend) {
                    float g[3];
                    float const w = taylor_term<Order, true>(fields, s, qrx, qry, qrz, ql2, g);
                    if (isfinite(w)) {
                        accepted = true;
                        float const m1 = __builtin_amdgcn_rsqf(ql2);
                        float const m2 = m1 * m1;
                        float const qn[3] = {qrx * m1, qry * m1, qrz * m1};
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            f[k] = -su * g[k];
                            f[3 + k] = -su * m2 * qn[k];
                            dq[k] += double(su * g[k]);
                        }
                        if constexpr (Order >= 1) {
                            float const m3 = m2 * m1;
                            f[6] = su * m3 * (1.0f - 3.0f * qn[0] * qn[0]);
                            f[7] = su * m3 * (1.0f - 3.0f * qn[1] * qn[1]);
                            f[8] = su * m3 * (1.0f - 3.0f * qn[2] * qn[2]);
                            f[9] = -3.0f * su * m3 * qn[0] * qn[1];
                            f[10] = -3.0f * su * m3 * qn[1] * qn[2];
                            f[11] = -3.0f * su * m3 * qn[2] * qn[0];
                        }
                    } else {
                        descend = true;
                    }
                }
            }
            std::uint64_t const amask = __ballot(accepted);
            if (amask != 0ull)
                wave_atomic_add<F>(dslot + (static_cast<std::size_t>(node) * 4 + s) * 12, f);
            std::uint64_t const dmask = __ballot(descend);
            if (dmask == 0ull)
                continue;
            if (c & k_cref_leaf) {
                std::uint32_t const r = c & ~k_cref_leaf;
                float t9[9];
#pragma unroll
                for (int k = 0; k < 9; ++k)
                    t9[k] = 0.0f;
                if (dmask & my_bit)
                    adjoint_leaf_terms(tris[r], x, y, z, sud, t9, dq);
                wave_atomic_add<9>(dtri + static_cast<std::size_t>(r) * 9, t9);
                continue;
            }
            if (next != k_invalid) {
                if (sp < StackCap) {
                    s_node[wave][sp] = next;
                    s_mask[wave][sp] = next_mask;
                    ++sp;
                } else {
                    overflow = true;
                }
            }
            next = c;
            next_mask = dmask;
        }
        if (next == k_invalid && sp > 0) {
            --sp;
            next = s_node[wave][sp];
            next_mask = s_mask[wave][sp];
        }
        node = next;
        mask = next_mask;
    }
    if (!active)
        return;
    if (overflow)
        dq[0] = dq[1] = dq[2] = __builtin_nan("");
    if (dqx != nullptr) {
        dqx[q] = static_cast<float>(dq[0]);
        dqy[q] = static_cast<float>(dq[1]);
        dqz[q] = static_cast<float>(dq[2]);
    }
}

template <int Order>
void launch_taylor_adjoint(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy, float const *qz,
    float const *u, std::uint32_t const *order, std::size_t n, float beta2, float *dslot, float *dtri,
    float *dqx, float *dqy, float *dqz, hipStream_t stream
) {
    bool const leaf_root = ref_leaf(bvh.root.reference);
    std::uint32_t const root = leaf_root ? k_invalid : static_cast<std::uint32_t>(ref_offset(bvh.root.reference));
    int const need = leaf_root ? 0 : static_cast<int>(bvh.internal_stack_bound);
    float4 const *records = leaf_root ? nullptr : m.records.ptr;
    // Hilbert-ordered queries (large batches) take the wave-cooperative form.
#define GWN_ADJ(C)                                                                                           \
    do {                                                                                                     \
        if (order != nullptr && !leaf_root)                                                                  \
            taylor_adjoint_wave_kernel<Order, C><<<grid_for(n, k_taylor_block), k_taylor_block, 0, stream>>>( \
                records, bvh.triangles.ptr, root, qx, qy, qz, u, order, n, beta2, dslot, dtri, dqx, dqy, dqz);  \
        else                                                                                                 \
            taylor_adjoint_kernel<Order, C><<<grid_for(n, k_taylor_block), k_taylor_block, 0, stream>>>(    \
                records, bvh.triangles.ptr, root, bvh.root.reference, qx, qy, qz, u, order, n, beta2, dslot,   \
                dtri, dqx, dqy, dqz);                                                                        \
    } while (0)
    if (need <= 32)
        GWN_ADJ(32);
    else if (need <= 64)
        GWN_ADJ(64);
    else if (need <= 128)
        GWN_ADJ(128);
    else
        throw_invalid("Traversal stack bound exceeds the largest compiled stack (128).");
#undef GWN_ADJ
    GWN_LAUNCH_CHECK();
}

// LDS of the stacks: 12 bytes an entry and wave, 4 bytes an entry and quad.
std::size_t batch_lds_bytes(int cap, int block, bool waves, bool quads) {
    std::size_t const entries = static_cast<std::size_t>(cap) * static_cast<std::size_t>(block);
    return std::max(waves ? entries / 64 * 12 : 0, quads ? entries : 0);
}

} // namespace

// The single-mesh rule or 32 queries per triangle at beta 2, or fewer where the batch is ten times as long as a wave
// of the mesh: its work decides then and not its longest wave.  That wave takes some 4 us sqrt(triangles), the
// batch with four lanes per query 0.5 ns a query at beta 2.  Measured, 6M queries over equal meshes, four lanes /
// whole waves: beta 2, 16 queries per triangle of 300 2.01 / 1.79 ms, of 3,000 2.69 / 2.50, of 20,000 2.70 / 2.86
// (25.6M queries of 64 meshes, 20 per triangle of 20,000: 11.2 / 8.8), 8 per triangle of 300 1.13 / 1.15, of 3,000
// 2.86 / 2.99; beta 4, 4 per triangle of 300 1.85 / 1.90, 8 of 300 3.36 / 2.51, 1 of 3,000 7.7 / 8.2, 2 of 3,000 14.0 /
// 11.7, 2 of 20,000 14.8 / 12.4, 2 of 100,000 14.3 / 13.9, 4 of 100,000 13.8 / 11.1.  128 uneven meshes of up to
// 100,000 triangles with 5.1M queries: 2.24 ms, 2.67 with the waves of three meshes of 6,700 to 12,000 triangles, of
// which the batch is only six to eight times as long.
bool batch_dense_queries(std::size_t triangles, std::size_t queries, std::size_t total_queries, float accuracy_scale) {
    double const beta = std::max(1.0, double(accuracy_scale)) / 2.0, t = double(triangles), n = double(queries);
    bool const lasting = 0.5e-3 * double(total_queries) * std::pow(beta, 2.25) >= 10.0 * 4.0 * std::sqrt(t);
    bool const dense = n >= 1500.0 && n >= 12.0 * t * std::pow(beta, -3.3) * std::pow(std::max(1.0, t / 4000.0), 0.25);
    return (lasting && dense) || dense_queries(triangles, queries, accuracy_scale * accuracy_scale) ||
           n >= 32.0 * t * std::pow(beta, -1.5);
}

void taylor_batch_launch(
    batch_mesh const *meshes, std::uint32_t mesh_count, std::uint64_t total_chunks, float accuracy_scale,
    std::uint64_t *counter, int order, int cap, int block, int blocks_per_cu, int cu_count, bool waves, bool quads,
    hipStream_t stream
) {
    float const beta2 = accuracy_scale * accuracy_scale;
    if (block <= 0 || block > 256 || (block & 63) != 0)
        throw_invalid("Batched query block size must be 64, 128, 192 or 256.");
    int const grid = std::max(1, blocks_per_cu * cu_count);
    std::size_t const lds = batch_lds_bytes(cap, block, waves, quads);
#define GWN_BATCH(O, W, Q) \
    taylor_batch_kernel<O, W, Q><<<grid, block, lds, stream>>>(meshes, mesh_count, total_chunks, beta2, cap, counter)
#define GWN_BATCH_ORDER(O) \
    (waves && quads ? GWN_BATCH(O, true, true) : waves ? GWN_BATCH(O, true, false) : GWN_BATCH(O, false, true))
    switch (order) {
    case 0: GWN_BATCH_ORDER(0); break;
    case 1: GWN_BATCH_ORDER(1); break;
    default: GWN_BATCH_ORDER(2); break;
    }
#undef GWN_BATCH_ORDER
#undef GWN_BATCH
}

void taylor_adjoint_traverse(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy, float const *qz,
    float const *u, std::uint32_t const *order, std::size_t n, float accuracy_scale, float *dslot, float *dtri,
    float *dqx, float *dqy, float *dqz, hipStream_t stream
) {
    float const beta2 = accuracy_scale * accuracy_scale;
    if (m.order == 0)
        launch_taylor_adjoint<0>(bvh, m, qx, qy, qz, u, order, n, beta2, dslot, dtri, dqx, dqy, dqz, stream);
    else if (m.order == 1)
        launch_taylor_adjoint<1>(bvh, m, qx, qy, qz, u, order, n, beta2, dslot, dtri, dqx, dqy, dqz, stream);
    else
        throw_invalid("The winding adjoint supports Taylor orders 0 and 1.");
}

void winding_exact(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz, void *out,
    std::size_t n, int precision, query_launch const &, hipStream_t stream
) {
    switch (precision) {
    case -1: // reference-form float output
        launch_exact_plain(bvh, qx, qy, qz, static_cast<float *>(out), n, stream);
        break;
    case GWN_PRECISION_PLAIN:
        launch_exact_plain(bvh, qx, qy, qz, static_cast<double *>(out), n, stream);
        break;
    case GWN_PRECISION_SPLIT:
        launch_exact<GWN_PRECISION_SPLIT>(bvh, qx, qy, qz, static_cast<double *>(out), n, stream);
        break;
    case GWN_PRECISION_FP64:
        launch_exact<GWN_PRECISION_FP64>(bvh, qx, qy, qz, static_cast<double *>(out), n, stream);
        break;
    default: throw_invalid("Unknown winding precision mode.");
    }
}

namespace {

// Device words the Hilbert presort of n queries needs besides the order itself: keys, their
// alternate buffer, the alternate id buffer and the sort's own workspace.
std::size_t query_order_workspace_words(std::size_t n) {
    return 3 * n + radix_sort_workspace_words(n, 0, 30);
}

// Hilbert presort with caller-given scratch (query_order_workspace_words(n) words): allocates
// nothing.
void query_order_ws(
    aabb const &box, float const *qx, float const *qy, float const *qz,
    std::uint32_t *order, std::size_t n, std::uint32_t *ws, hipStream_t stream
) {
    std::uint32_t *const keys = ws;
    std::uint32_t *const keys_alt = ws + n;
    std::uint32_t *const ids_alt = ws + 2 * n;
    query_key_kernel<<<grid_for(n, 256), 256, 0, stream>>>(qx, qy, qz, n, box, keys, order);
    GWN_LAUNCH_CHECK();
    std::uint32_t *sk = nullptr;
    std::uint32_t *sorted = nullptr;
    radix_sort_pairs_u32_ws(keys, keys_alt, order, ids_alt, n, 0, 30, ws + 3 * n, &sk, &sorted, stream);
    if (sorted != order)
        GWN_HIP(hipMemcpyAsync(order, sorted, n * sizeof(std::uint32_t), hipMemcpyDeviceToDevice, stream));
}

} // namespace

void query_order(
    gwn_bvh_handle const &bvh, float const *qx, float const *qy, float const *qz,
    std::uint32_t *order, std::size_t n, hipStream_t stream
) {
    query_order_box(bvh.root.bounds, qx, qy, qz, order, n, stream);
}

void query_order_box(
    aabb const &box, float const *qx, float const *qy, float const *qz, std::uint32_t *order, std::size_t n,
    hipStream_t stream
) {
    if (n == 0)
        return;
    device_buffer<std::uint32_t> ws(query_order_workspace_words(n), stream);
    query_order_ws(box, qx, qy, qz, order, n, ws.ptr, stream);
}

void winding_taylor(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy,
    float const *qz, float *out, float *gx, float *gy, float *gz, std::size_t n, float accuracy_scale,
    int precision, query_launch const &cfg, std::uint32_t const *given_order, std::uint32_t *counters,
    hipStream_t stream
) {
    if (n == 0)
        return;
    if (precision != GWN_PRECISION_PLAIN && precision != GWN_PRECISION_SPLIT)
        throw_invalid("Taylor winding supports the plain and split precision modes.");
    bool const grad = gx != nullptr;
    taylor_outputs const o{out, gx, gy, gz, counters};
    if (ref_leaf(bvh.root.reference)) {
        unsigned const grid = grid_for(n, 256);
        std::uint64_t const off = ref_offset(bvh.root.reference);
        std::uint32_t const cnt = ref_count(bvh.root.reference);
#define GWN_LEAF_ROOT(P, G) leaf_root_kernel<P, G><<<grid, 256, 0, stream>>>(bvh.triangles.ptr, off, cnt, qx, qy, qz, o, n)
        if (precision == GWN_PRECISION_PLAIN)
            grad ? GWN_LEAF_ROOT(GWN_PRECISION_PLAIN, true) : GWN_LEAF_ROOT(GWN_PRECISION_PLAIN, false);
        else
            grad ? GWN_LEAF_ROOT(GWN_PRECISION_SPLIT, true) : GWN_LEAF_ROOT(GWN_PRECISION_SPLIT, false);
#undef GWN_LEAF_ROOT
        GWN_LAUNCH_CHECK();
        return;
    }
    bool const sort = given_order == nullptr &&
                      (cfg.sort_queries > 0 || (cfg.sort_queries < 0 && n >= (1u << 16)));
    device_buffer<std::uint32_t> own_order;
    std::uint32_t const *order = given_order;
    if (sort) {
        own_order.allocate(n, stream);
        query_order(bvh, qx, qy, qz, own_order.ptr, n, stream);
        order = own_order.ptr;
    }
    float const beta2 = accuracy_scale * accuracy_scale;
#define GWN_TAYLOR_CASE(O, P, G) launch_taylor<O, P, G>(bvh, m, qx, qy, qz, order, o, n, beta2, stream)
#define GWN_TAYLOR_ORDERS(P, G)                                                                     \
    switch (m.order) {                                                                              \
    case 0: GWN_TAYLOR_CASE(0, P, G); break;                                                        \
    case 1: GWN_TAYLOR_CASE(1, P, G); break;                                                        \
    default: GWN_TAYLOR_CASE(2, P, G); break;                                                       \
    }
    if (precision == GWN_PRECISION_PLAIN) {
        if (grad) {
            GWN_TAYLOR_ORDERS(GWN_PRECISION_PLAIN, true)
        } else {
            GWN_TAYLOR_ORDERS(GWN_PRECISION_PLAIN, false)
        }
    } else {
        if (grad) {
            GWN_TAYLOR_ORDERS(GWN_PRECISION_SPLIT, true)
        } else {
            GWN_TAYLOR_ORDERS(GWN_PRECISION_SPLIT, false)
        }
    }
#undef GWN_TAYLOR_ORDERS
#undef GWN_TAYLOR_CASE
}

// ---------------------------------------------------------------------------------------------
// Allocation-free Taylor batch.  Its only scratch is the Hilbert presort's (the visiting order,
// keys, alternate buffers and the sort's digit table), which lives in one static device array per
// GPU, sized for k_noalloc_max_queries queries.  Host code never passes the array's name to a
// kernel: that name is a host-side stand-in.  The array's device address is looked up once per
// device with hipGetSymbolAddress (with that device current) and that pointer is used instead.
// Every call on one GPU shares the array and leaves the last call's contents in it; the sort
// clears its digit bases itself, and everything else is fully overwritten before it is read.
// Calls that overlap on one GPU (different streams, or host threads) race on the array.
// ---------------------------------------------------------------------------------------------

namespace {

constexpr std::size_t k_noalloc_order_words = k_noalloc_max_queries;
constexpr std::size_t k_noalloc_sort_words =
    3 * k_noalloc_max_queries + 4 * 256 + (k_noalloc_max_queries + 4095) / 4096 * 256;
constexpr std::size_t k_noalloc_scratch_words = k_noalloc_order_words + k_noalloc_sort_words;

__device__ __align__(256) std::uint32_t scratch[k_noalloc_scratch_words];

constexpr int k_max_devices = 64;
std::mutex g_scratch_mutex;
std::uint32_t *g_scratch_ptr[k_max_devices] = {};

// The calling thread's current device's copy of `scratch` (resolved once per device).
std::uint32_t *device_scratch() {
    int dev = 0;
    GWN_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= k_max_devices)
        throw_internal("noalloc Taylor batch: device ordinal out of range.");
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void *ptr = nullptr;
        GWN_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        if (ptr == nullptr)
            throw_internal("noalloc Taylor batch: scratch symbol has no device address.");
        g_scratch_ptr[dev] = static_cast<std::uint32_t *>(ptr);
    }
    return g_scratch_ptr[dev];
}

} // namespace

void winding_taylor_noalloc(
    gwn_bvh_handle const &bvh, gwn_moment_handle const &m, float const *qx, float const *qy,
    float const *qz, float *out, std::size_t n, float accuracy_scale, int precision, query_launch const &cfg,
    hipStream_t stream
) {
    if (n > k_noalloc_max_queries)
        throw_invalid("noalloc Taylor batch: query count exceeds the static scratch capacity (1048576 queries).");
    static_assert(k_noalloc_sort_words >= 3 * k_noalloc_max_queries + 4 * 256 + (k_noalloc_max_queries + 4095) / 4096 * 256,
                  "presort scratch must cover query_order_workspace_words(k_noalloc_max_queries)");
    if (n == 0)
        return;
    bool const sort = !ref_leaf(bvh.root.reference) &&
                      (cfg.sort_queries > 0 || (cfg.sort_queries < 0 && n >= (1u << 16)));
    if (!sort) {
        winding_taylor(bvh, m, qx, qy, qz, out, nullptr, nullptr, nullptr, n, accuracy_scale, precision, cfg,
                       nullptr, nullptr, stream);
        return;
    }
    if (query_order_workspace_words(n) > k_noalloc_sort_words)
        throw_internal("noalloc Taylor batch: presort scratch too small.");
    std::uint32_t *const base = device_scratch();
    std::uint32_t *const order = base;
    query_order_ws(bvh.root.bounds, qx, qy, qz, order, n, base + k_noalloc_order_words, stream);
    winding_taylor(bvh, m, qx, qy, qz, out, nullptr, nullptr, nullptr, n, accuracy_scale, precision, cfg, order,
                   nullptr, stream);
}

} // namespace gwn
