// Gradients of y = (x @ W^T) * scale + bias for a frozen prepacked fp8 weight W:
//   grad_x[m, k]  = sum_n grad[m, n] * scale[n] * W[n, k]        grad_bias[n] = sum_m grad[m, n]
// grad_x is the forward's own matmul on the transposed weight: the prepacked [K/16][N][16] becomes [N/16][K][16]
// (one pass over the weight, here), and the ring, wide and streaming kernels contract over N.
//
// The products are those of fp32 arithmetic, on the 16-bit MFMAs: an fp8 code is exact in fp16 and bf16, so a
// 16-bit gradient times a code is exact in the fp32 accumulator. A per-tensor scale goes into the decode (its
// power of two) and the epilogue. A per-column scale sits inside the sum: grad * scale is formed in fp32 and split
// into three bf16 terms that sum to it (column_slab), and the matmul runs over the three side by side, a contraction
// three times as long over three copies of the weight. bf16 gradients reach sizes whose products with a scale (2^-19
// of the weight's size in e5m2) have no three terms left above bf16's least value, so there the scales are taken times
// the power of two that brings the largest near 1 (scale_up), and the weight's decode divides by it.
//
// Measured, forward and backward of 4096 rows through 3072 -> 12288 in bf16, one scale: 2744 us with torch's fp32
// operations (2.0 ms its fp32 matmul, 0.27 ms the column sums, 0.17 ms dequantizing the weight), 436 us here: the
// matmul's 309 GFLOP take 215-238 us (1.3-1.4 PFLOP/s, the rate of the forward's). 1000 rows through 2560 -> 5120 in
// fp16 with per-column scales: 334 us of kernels, 128 here (the three-term matmul 74 us, 1.06 PFLOP/s).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "feather_internal.h"
#include "scaled_mm_kernels.h"
#include "scaled_mm_launch.h"

namespace feather {
namespace {

constexpr int kThreads = 256;

// ---- weight transpose ----------------------------------------------------------------------------------------
//
// b [K/16][N][16] -> out [copies][N16][K][16], N16 = ceil(N / 16): out[c][n / 16][k][n % 16] = b[k / 16][n][k % 16],
// zero for n >= N. Copies after the first (e5m2) hold zero for an infinite code: they meet the small terms of the split
// gradient, and a zero term times inf would add NaN to the first copy's inf. A workgroup takes 8 chunks of k by 128 columns n (16 KiB): 2 KiB runs in, 2 KiB runs out, through
// LDS, the byte transpose in registers (16 dwords of 4 k each -> 4 x 16 bytes, by 4 x 4 byte transposes). HBM-bound:
// 13.4 us for a 37.7 MB weight, 5.6 TB/s read and written.
constexpr int kTileChunks = 8;                 // 128 k
constexpr int kTileCols = 128;                 // 8 groups of 16 n
constexpr int kGroupPitch = 16 * 16 + 128;     // LDS bytes of 16 columns of one chunk: neighbours 32 banks apart
constexpr int kChunkPitch = 8 * kGroupPitch + 16;   // neighbouring chunks 4 banks apart

// The dword's four e5m2 codes without the infinite ones (0x7c, 0xfc), which become zero.
__device__ __forceinline__ uint32_t drop_e5m2_inf(uint32_t w) {
    const uint32_t other = (((w & 0x7f7f7f7fu) ^ 0x7c7c7c7cu) + 0x7f7f7f7fu) & 0x80808080u;   // set where not inf
    return w & ((other >> 7) * 0xffu);
}

// The place of 16-byte unit k of a group's 128: the writes below take every fourth unit, the reads consecutive ones,
// and both spread over all banks.
__device__ __forceinline__ uint32_t swizzled_unit(uint32_t k) {
    return (k & ~3u) | ((k ^ (k >> 4)) & 3u);
}

__device__ __forceinline__ void transpose_tile(const uint8_t* b, uint8_t* out, uint32_t K, uint32_t N, uint32_t n16,
                                               uint32_t copies, bool e5m2, uint32_t k_tiles, uint32_t tile,
                                               uint8_t* lds) {
    const uint32_t t = threadIdx.x;
    const uint32_t chunk0 = tile % k_tiles * kTileChunks;
    const uint32_t n0 = tile / k_tiles * kTileCols;
    const uint32_t chunks = K / 16u;
    const rsrc_t src = make_rsrc(b, chunks * N * 16u);
    const rsrc_t dst = make_rsrc(out, copies * n16 * K * 16u);
    u32x4 in[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t chunk = chunk0 + t / kTileCols + 2u * i;
        const uint32_t n = n0 + t % kTileCols;
        in[i] = buf_load16(src, chunk < chunks && n < N ? (chunk * N + n) * 16u : kOob);
    }
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t n = t % kTileCols;
        *reinterpret_cast<u32x4*>(lds + (t / kTileCols + 2u * i) * kChunkPitch + n / 16u * kGroupPitch + n % 16u * 16u) =
            in[i];
    }
    __syncthreads();
    // Work-item t: columns 16 (t / 32) .. + 15, k values 4 (t % 32) .. + 3 of the tile.
    const uint32_t group = t / 32u;
    const uint32_t k4 = t % 32u;
    uint32_t o[4][4];   // [k][4 columns]
    const uint8_t* base = lds + k4 / 4u * kChunkPitch + group * kGroupPitch + k4 % 4u * 4u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t d[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = *reinterpret_cast<const uint32_t*>(base + (4 * r + i) * 16);
        const uint32_t a0 = __builtin_amdgcn_perm(d[1], d[0], perm_sel(0, 4, 1, 5));
        const uint32_t a1 = __builtin_amdgcn_perm(d[1], d[0], perm_sel(2, 6, 3, 7));
        const uint32_t c0 = __builtin_amdgcn_perm(d[3], d[2], perm_sel(0, 4, 1, 5));
        const uint32_t c1 = __builtin_amdgcn_perm(d[3], d[2], perm_sel(2, 6, 3, 7));
        o[0][r] = __builtin_amdgcn_perm(c0, a0, perm_sel(0, 1, 4, 5));
        o[1][r] = __builtin_amdgcn_perm(c0, a0, perm_sel(2, 3, 6, 7));
        o[2][r] = __builtin_amdgcn_perm(c1, a1, perm_sel(0, 1, 4, 5));
        o[3][r] = __builtin_amdgcn_perm(c1, a1, perm_sel(2, 3, 6, 7));
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        *reinterpret_cast<u32x4*>(lds + group * 2048u + swizzled_unit(4u * k4 + j) * 16u) =
            u32x4{o[j][0], o[j][1], o[j][2], o[j][3]};
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t g = t / 128u + 2u * i;
        const uint32_t k = t % 128u;
        u32x4 v = *reinterpret_cast<const u32x4*>(lds + g * 2048u + swizzled_unit(k) * 16u);
        const uint32_t ng = n0 / 16u + g;
        const uint32_t kk = chunk0 * 16u + k;
        for (uint32_t c = 0; c < copies; ++c) {
            const uint32_t off = ng < n16 && kk < K ? ((c * n16 + ng) * K + kk) * 16u : kOob;
            __builtin_amdgcn_raw_buffer_store_b128(v, dst, static_cast<int>(off), 0, 0);
            if (e5m2 && c == 0) {
#pragma unroll
                for (int w = 0; w < 4; ++w) v[w] = drop_e5m2_inf(v[w]);
            }
        }
    }
}

// ---- per-column scales -----------------------------------------------------------------------------------------

// h (24 significant bits) = t[0] + t[1] + t[2], bf16 bits each, by truncation: exact from |h| = 2^-110 on (below, what
// falls under bf16's least value, 2^-133, is lost), and t[0] never overflows. Of inf and NaN the first term carries
// everything.
__device__ __forceinline__ void split3(float h, uint32_t (&t)[3]) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, h);
    const bool finite = (bits & 0x7f800000u) != 0x7f800000u;
    // a NaN whose payload lies in the low half keeps being one
    t[0] = (bits >> 16) | ((bits & 0x7fffffffu) > 0x7f800000u ? 0x40u : 0u);
    const float r1 = h - __builtin_bit_cast(float, bits & 0xffff0000u);
    const uint32_t bits1 = __builtin_bit_cast(uint32_t, r1);
    const float r2 = r1 - __builtin_bit_cast(float, bits1 & 0xffff0000u);
    t[1] = finite ? bits1 >> 16 : 0u;
    t[2] = finite ? __builtin_bit_cast(uint32_t, r2) >> 16 : 0u;
}

// The power of two, 1 to 2^100, that takes the largest finite |scale| of N into [0.5, 1), or as near below as it goes; 1
// where that is 0.5 or more. |gradient * scale| then stays under |gradient|, so nothing overflows that did not, and what
// split3 loses of a product is under 2^-132 times the largest weight, about the least step of a bf16 result. Every
// workgroup reads all the scales (64 KiB at N = 16384, from L2).
__device__ __forceinline__ float scale_up(const float* scale, uint32_t N, uint32_t (&top)[kThreads / kWave]) {
    const rsrc_t src = make_rsrc(scale, N * 4u);
    uint32_t most = 0;
    for (uint32_t n = threadIdx.x * 4u; n < N; n += kThreads * 4u) {
        const u32x4 v = buf_load16(src, n * 4u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t magnitude = v[i] & 0x7fffffffu;
            most = max(most, magnitude < 0x7f800000u ? magnitude : 0u);
        }
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, d)));
    if (threadIdx.x % kWave == 0) top[threadIdx.x / kWave] = most;
    __syncthreads();
    const uint32_t exponent = max(max(top[0], top[1]), max(top[2], top[3])) >> 23;
    const uint32_t up = exponent >= 126u ? 0u : min(126u - exponent, 100u);
    return __builtin_bit_cast(float, (127u + up) << 23);
}

// g [M, N] with N % 16 = 8 -> out [M, N + 8], zero in the new columns (pads_columns).
__global__ __launch_bounds__(kThreads) void pad_columns_kernel(const uint16_t* g, uint16_t* out, uint32_t M, uint32_t N) {
    const uint32_t pieces = N / 8u + 1u;
    const uint32_t piece = blockIdx.x * kThreads + threadIdx.x;
    const uint32_t row = piece / pieces;
    const uint32_t col = piece % pieces * 8u;
    if (row >= M) return;
    const u32x4 v = buf_load16(make_rsrc(g, M * N * 2u), col < N ? (row * N + col) * 2u : kOob);
    __builtin_amdgcn_raw_buffer_store_b128(v, make_rsrc(out, M * (N + 8u) * 2u),
                                           static_cast<int>((row * (N + 8u) + col) * 2u), 0, 0);
}

// ---- column sums -----------------------------------------------------------------------------------------------

constexpr uint32_t kSumCols = 256;    // columns of a workgroup: 32 work-items x 8
constexpr uint32_t kSumLanes = 8;     // rows summed side by side
constexpr uint32_t kSumMinRows = 32;  // rows of a workgroup, at least

template <bool kBf16>
__device__ __forceinline__ uint16_t round16(float x) {
    return static_cast<uint16_t>(pack_out<kBf16>(x, x) & 0xffffu);
}

struct Columns {
    const uint16_t* g;      // [M, N]
    float* partial;         // [slabs][N] sums of a slab's rows, or nullptr (no sums)
    uint16_t* sums;         // [N], written here where there is a single slab
    const float* scale;     // kSplit: [N]
    float* unscale;         // kSplit of bf16 gradients: 1 / scale_up goes here, for the matmul
    uint16_t* terms;        // kSplit: [M, 3 nc] bf16, the terms of column n at n, nc + n and 2 nc + n, zero past N
    uint32_t M, N, nc;      // nc = 16 * ceil(N / 16)
    uint32_t rows, slabs;   // rows of a slab
};

// A slab's rows of 256 columns: their sums in fp32, in a fixed order (each work-item 8 columns of every eighth row, four
// 16-byte loads in flight), and, kSplit, each element times its column's scale as three bf16 terms. HBM-bound (sums of
// 4096 x 12288 alone: 17.4 us, 5.8 TB/s, against 272 for torch's sum).
template <bool kBf16, bool kSplit>
__device__ __forceinline__ void column_slab(const Columns& p, uint32_t tile, uint32_t slab, float (*red)[kSumCols],
                                            uint32_t (&top)[kThreads / kWave]) {
    const rsrc_t src = make_rsrc(p.g, p.M * p.N * 2u);
    const uint32_t lane = threadIdx.x / 32u;
    const uint32_t col_in = threadIdx.x % 32u * 8u;
    const uint32_t col = tile * kSumCols + col_in;
    const uint32_t end = min(p.M, (slab + 1) * p.rows);
    float scale[8];
    if constexpr (kSplit) {
        const rsrc_t scale_rsrc = make_rsrc(p.scale, p.N * 4u);
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const f32x4 s = __builtin_bit_cast(f32x4, buf_load16(scale_rsrc, col < p.N ? col * 4u + 16u * h : kOob));
#pragma unroll
            for (int i = 0; i < 4; ++i) scale[4 * h + i] = s[i];
        }
        if constexpr (kBf16) {
            const float up = scale_up(p.scale, p.N, top);
            if (blockIdx.x == 0 && threadIdx.x == 0) *p.unscale = 1.0f / up;
#pragma unroll
            for (int i = 0; i < 8; ++i) scale[i] *= up;
        }
    }
    float sum[8] = {};
    constexpr uint32_t kUnroll = kSplit ? 4 : 8;
    for (uint32_t row = slab * p.rows + lane; row < end; row += kUnroll * kSumLanes) {
        u32x4 v[kUnroll];
#pragma unroll
        for (uint32_t i = 0; i < kUnroll; ++i) {
            const uint32_t r = row + i * kSumLanes;
            v[i] = buf_load16(src, r < end && col < p.N ? (r * p.N + col) * 2u : kOob);
        }
#pragma unroll
        for (uint32_t i = 0; i < kUnroll; ++i) {
            u32x4 t[3];
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint32_t pair = v[i][w];
                float lo, hi;
                if constexpr (kBf16) {
                    lo = __builtin_bit_cast(float, pair << 16);
                    hi = __builtin_bit_cast(float, pair & 0xffff0000u);
                } else {
                    const half2v h = __builtin_bit_cast(half2v, pair);
                    lo = static_cast<float>(h[0]);
                    hi = static_cast<float>(h[1]);
                }
                sum[2 * w] += lo;
                sum[2 * w + 1] += hi;
                if constexpr (kSplit) {
                    uint32_t tl[3], th[3];
                    split3(lo * scale[2 * w], tl);
                    split3(hi * scale[2 * w + 1], th);
#pragma unroll
                    for (int j = 0; j < 3; ++j) t[j][w] = tl[j] | (th[j] << 16);
                }
            }
            if constexpr (kSplit) {
                const rsrc_t dst = make_rsrc(p.terms, p.M * p.nc * 6u);
                const uint32_t r = row + i * kSumLanes;
#pragma unroll
                for (uint32_t j = 0; j < 3; ++j) {
                    const uint32_t off = r < end && col < p.nc ? (r * 3u * p.nc + j * p.nc + col) * 2u : kOob;
                    __builtin_amdgcn_raw_buffer_store_b128(t[j], dst, static_cast<int>(off), 0, 0);
                }
            }
        }
    }
    if (!p.partial) return;
#pragma unroll
    for (int i = 0; i < 8; ++i) red[lane][col_in + i] = sum[i];
    __syncthreads();
    const uint32_t c = tile * kSumCols + threadIdx.x;
    if (c >= p.N) return;
    float total = 0.f;
#pragma unroll
    for (uint32_t i = 0; i < kSumLanes; ++i) total += red[i][threadIdx.x];
    if (p.slabs == 1) {
        p.sums[c] = round16<kBf16>(total);
    } else {
        p.partial[slab * p.N + c] = total;
    }
}

// What the matmul needs and the bias's gradient, in one launch: the first workgroups take a slab of the gradient's columns,
// the last `transposes` a tile of the weight, side by side (1000 x 2560 -> 5120 with per-column scales: 15.8 us against
// 10.2 + 8.0 + 5.1 in launches of their own).
template <bool kBf16, bool kSplit>
__global__ __launch_bounds__(kThreads) void prepare_kernel(const uint8_t* b, uint8_t* weight, uint32_t K, uint32_t n16,
                                                            bool e5m2, uint32_t k_tiles, uint32_t transposes,
                                                            Columns columns, uint32_t col_tiles) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kTileChunks * kChunkPitch];
    static_assert(sizeof(lds) >= sizeof(float) * kSumLanes * kSumCols, "the sums' join fits");
    __shared__ uint32_t top[kThreads / kWave];
    const uint32_t slab_blocks = gridDim.x - transposes;
    if (blockIdx.x >= slab_blocks) {
        transpose_tile(b, weight, K, columns.N, n16, kSplit ? 3u : 1u, e5m2, k_tiles, blockIdx.x - slab_blocks, lds);
    } else {
        const uint32_t i = blockIdx.x;
        column_slab<kBf16, kSplit>(columns, i % col_tiles, i / col_tiles, reinterpret_cast<float(*)[kSumCols]>(lds),
                                   top);
    }
}

template <bool kBf16>
__global__ __launch_bounds__(kThreads) void column_sums_join_kernel(const float* partial, uint16_t* out, uint32_t N,
                                                                     uint32_t slabs) {
    const uint32_t c = blockIdx.x * kThreads + threadIdx.x;
    if (c >= N) return;
    float total = 0.f;
#pragma unroll 8
    for (uint32_t s = 0; s < slabs; ++s) total += partial[s * N + c];
    out[c] = round16<kBf16>(total);
}

// Slabs of rows of the column sums: about four workgroups per CU, at least kSumMinRows rows each.
int64_t sum_slabs(int64_t M, int64_t N) {
    const int64_t col_tiles = (N + kSumCols - 1) / kSumCols;
    return std::max<int64_t>(1, std::min<int64_t>((1024 + col_tiles - 1) / col_tiles, M / kSumMinRows));
}

// ---- workspace -------------------------------------------------------------------------------------------------

constexpr int64_t align256(int64_t n) {
    return (n + 255) / 256 * 256;
}

struct Layout {
    int64_t depth;         // the matmul's contraction: N (16 for 8), or 3 * 16 * ceil(N / 16) with per-column scales
    int64_t weight;        // bytes of the transposed weight, at 0
    int64_t terms;         // of the split gradient, or of a padded one (N % 16 = 8), after it
    int64_t sums;          // of the column sums' partials, after that
    int64_t unscale;       // of one float, last
    int64_t total() const { return weight + terms + sums + unscale; }
};

Layout layout(int64_t M, int64_t N, int64_t K, bool per_column) {
    const int64_t n16 = (N + 15) / 16;
    Layout l{};
    l.depth = per_column ? 3 * 16 * n16 : std::max<int64_t>(N, 16);
    l.weight = align256((l.depth + 127) / 128 * 8 * K * 16);
    l.terms = per_column ? align256(M * l.depth * 2) : N % 16 ? align256(M * 16 * n16 * 2) : 0;
    l.sums = align256(sum_slabs(M, N) * N * 4);
    l.unscale = per_column ? align256(4) : 0;
    return l;
}

// The matmul takes the gradient padded to whole chunks: on streaming tiles, whose rows are whole chunks, and on every
// tile where one chunk is all there is.
bool pads_columns(int64_t N, bool per_column, bool prefetch) {
    return !per_column && N % 16 != 0 && (!prefetch || N < 16);
}

// The contraction of the launch itself: the padded columns included.
int64_t launch_depth(int64_t N, bool per_column, bool prefetch) {
    return pads_columns(N, per_column, prefetch) ? N + 8 : layout(1, N, 16, per_column).depth;
}

bool aligned16(const void* p) {
    return (reinterpret_cast<uintptr_t>(p) & 15u) == 0;
}

}  // namespace
}  // namespace feather

extern "C" int64_t feather_linear_backward_depth(const int64_t N, const bool per_column) {
    return feather::layout(1, N, 16, per_column).depth;
}

extern "C" int64_t feather_linear_backward_split_bytes(const int64_t M, const int64_t N, const int64_t K,
                                                       const bool per_column, const int block_warps_m,
                                                       const int block_warps_n, const int unroll_k, const int repeat_m,
                                                       const int repeat_n, const bool prefetch, const int splits) {
    if (feather_linear_backward_workspace_bytes(M, N, K, per_column) < 0) return -1;
    const feather::TileQuery tile{block_warps_m, block_warps_n, unroll_k, repeat_m, repeat_n, prefetch};
    return feather::grad_matmul_split_bytes(tile, M, K, feather::launch_depth(N, per_column, prefetch), true, splits);
}

extern "C" int64_t feather_linear_backward_workspace_bytes(const int64_t M, const int64_t N, const int64_t K,
                                                           const bool per_column) {
    if (M < 1 || N < 8 || N % 8 != 0 || K < 16 || K % 16 != 0) return -1;
    constexpr int64_t most = (int64_t{1} << 31) - 1;   // buffer offsets
    const feather::Layout l = feather::layout(M, N, K, per_column);
    if (M * N * 2 > most || M * K * 2 > most || l.weight > most || l.terms > most || l.sums > most) return -1;
    return l.total();
}

extern "C" bool feather_linear_backward(const uint16_t* const grad, const uint8_t* const b_prepacked,
                                        const float* const scale, uint16_t* const grad_x, uint16_t* const grad_bias,
                                        const int64_t M, const int64_t N, const int64_t K, const bool per_column,
                                        const bool use_fp8_e5m2, const bool bf16, const int block_warps_m,
                                        const int block_warps_n, const int unroll_k, const int repeat_m,
                                        const int repeat_n, const bool prefetch, const int splits,
                                        void* const split_workspace, const int64_t split_workspace_bytes,
                                        void* const workspace, const int64_t workspace_bytes, hipStream_t stream) {
    using namespace feather;
    const int64_t need = feather_linear_backward_workspace_bytes(M, N, K, per_column);
    if (need < 0 || !workspace || workspace_bytes < need || !aligned16(workspace)) return false;
    if (!grad || !aligned16(grad) || (!grad_x && !grad_bias)) return false;
    const Layout l = layout(M, N, K, per_column);
    uint8_t* const weight = static_cast<uint8_t*>(workspace);
    const uint32_t m = static_cast<uint32_t>(M), n = static_cast<uint32_t>(N), k = static_cast<uint32_t>(K);
    const bool pad = pads_columns(N, per_column, prefetch);
    const int64_t depth = launch_depth(N, per_column, prefetch);
    const TileQuery tile{block_warps_m, block_warps_n, unroll_k, repeat_m, repeat_n, prefetch};
    uint16_t* const made = reinterpret_cast<uint16_t*>(weight + l.weight);
    if (grad_x) {
        if (!b_prepacked || !scale || !aligned16(b_prepacked) || !aligned16(grad_x)) return false;
        if (per_column && !aligned16(scale)) return false;
        const int64_t split_bytes = grad_matmul_split_bytes(tile, M, K, depth, bf16 || per_column, splits);
        if (split_bytes < 0 || split_bytes > split_workspace_bytes) return false;
        if (splits > 1 && (!split_workspace || (reinterpret_cast<uintptr_t>(split_workspace) & 255u))) return false;
    }
    const bool split = grad_x && per_column;
    const uint32_t n16 = (n + 15) / 16;
    const uint32_t k_tiles = (k + 16 * kTileChunks - 1) / (16 * kTileChunks);
    const uint32_t transposes = grad_x ? k_tiles * ((n + kTileCols - 1) / kTileCols) : 0;
    const int64_t slabs = sum_slabs(M, N);
    Columns columns{};
    columns.g = grad;
    columns.partial = grad_bias ? reinterpret_cast<float*>(weight + l.weight + l.terms) : nullptr;
    columns.sums = grad_bias;
    columns.scale = scale;
    columns.unscale = reinterpret_cast<float*>(weight + l.weight + l.terms + l.sums);
    columns.terms = made;
    columns.M = m;
    columns.N = n;
    columns.nc = 16 * n16;
    columns.rows = static_cast<uint32_t>((M + slabs - 1) / slabs);
    columns.slabs = (m + columns.rows - 1) / columns.rows;
    const uint32_t col_tiles = (columns.nc + kSumCols - 1) / kSumCols;
    const uint32_t slab_blocks = grad_bias || split ? col_tiles * columns.slabs : 0;
    const auto prepare = split ? (bf16 ? prepare_kernel<true, true> : prepare_kernel<false, true>)
                               : (bf16 ? prepare_kernel<true, false> : prepare_kernel<false, false>);
    hipLaunchKernelGGL(prepare, dim3(transposes + slab_blocks), dim3(kThreads), 0, stream, b_prepacked, weight, k, n16,
                       use_fp8_e5m2, k_tiles, transposes, columns, col_tiles);
    if (grad_x) {
        if (pad) {
            const uint32_t blocks = static_cast<uint32_t>((M * (N / 8 + 1) + kThreads - 1) / kThreads);
            hipLaunchKernelGGL(pad_columns_kernel, dim3(blocks), dim3(kThreads), 0, stream, grad, made, m, n);
        }
        const float* const rest = !per_column ? scale : bf16 ? columns.unscale : nullptr;
        if (!launch_grad_matmul(tile, split || pad ? made : grad, weight, rest, grad_x, M, K, depth, use_fp8_e5m2,
                                bf16 || per_column, bf16, splits, split_workspace, stream)) {
            return false;
        }
    }
    if (grad_bias && columns.slabs > 1) {
        hipLaunchKernelGGL(bf16 ? column_sums_join_kernel<true> : column_sums_join_kernel<false>,
                           dim3((n + kThreads - 1) / kThreads), dim3(kThreads), 0, stream, columns.partial, grad_bias, n,
                           columns.slabs);
    }
    return true;
}
