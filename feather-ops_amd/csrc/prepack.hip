// Weight prepack on the GPU: b [K, N] fp8 codes (row-major; the GEMM's B, i.e. W^T) ->
// b_prepacked [K_pad / 16, N, 16] with K_pad = ceil(K / 128) * 128 and zero pad rows, so that
// b_prepacked[k / 16, n, k % 16] = b[k, n] (the layout of the reference's prepack_b_for_scaled_mm,
// feather_ops/scaled_mm.py:137-150). A pure byte permutation: bit-exact, dtype-agnostic.
//
// One block per (16-deep chunk, 128 columns): 256 work-items read the chunk's 16 rows x 128 columns
// with coalesced 8-byte loads (each row segment is 128 contiguous bytes) into LDS, then each work-item
// writes half of one column's 16 contiguous bytes. HBM-bound: 1 byte read and 1 written per element.
//
// Further down, the same layout from W as a Linear stores it, [N, K] (pack_rows_kernel): fp8 codes as they are, or
// a bf16, fp16 or fp32 weight quantized on the way.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "feather_internal.h"
#include "scaled_mm_kernels.h"

namespace feather {
namespace {

constexpr int kPrepackThreads = 256;
constexpr int kPrepackCols = 128;

__global__ __launch_bounds__(kPrepackThreads) void prepack_kernel(const uint8_t* b, uint8_t* out, uint32_t K,
                                                                   uint32_t N, uint32_t col_tiles,
                                                                   uint32_t chunks) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[16][kPrepackCols];
    const uint32_t chunk = blockIdx.x / col_tiles;
    const uint32_t n0 = (blockIdx.x % col_tiles) * kPrepackCols;
    const rsrc_t src = make_rsrc(b, K * N);
    const rsrc_t dst = make_rsrc(out, chunks * N * 16u);
    const uint32_t t = threadIdx.x;

    // Load: work-item t takes row t / 16 of the chunk, columns 8 * (t % 16) .. + 7 (N % 8 == 0, so such a
    // group is all inside N or all past it). Rows past K are the zero padding.
    {
        const uint32_t k = chunk * 16u + t / 16u;
        const uint32_t col = n0 + 8u * (t % 16u);
        const uint32_t off = (k < K && col < N) ? k * N + col : kOob;
        *reinterpret_cast<u32x2*>(&tile[t / 16u][8u * (t % 16u)]) = buf_load8(src, off);
    }
    __syncthreads();

    // Store: work-item t writes bytes 8h .. 8h + 7 (h = t % 2) of column t / 2's 16-byte group.
    const uint32_t col = t / 2u;
    const uint32_t h = t % 2u;
    uint32_t w[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        const uint32_t r = 8u * h + 4u * d;
        w[d] = static_cast<uint32_t>(tile[r][col]) | (static_cast<uint32_t>(tile[r + 1][col]) << 8) |
               (static_cast<uint32_t>(tile[r + 2][col]) << 16) | (static_cast<uint32_t>(tile[r + 3][col]) << 24);
    }
    const uint32_t n = n0 + col;
    buf_store8(u32x2{w[0], w[1]}, dst, n < N ? (chunk * N + n) * 16u + 8u * h : kOob);
}

// ---- [N, K] weights --------------------------------------------------------------------------------------------
//
// w [N, K] row-major, K a multiple of 16 -> out [K_pad/16][N][16]. The 16 codes of a unit (n, k / 16) stay together, so
// this is a transpose of 16-byte units: a workgroup takes 32 rows by 32 units, reads 512-byte runs of codes (1-2 KiB
// of a weight to quantize), passes the units through LDS and writes 512-byte runs. HBM-bound: 14336 x 4096 codes
// 18.2 us (6.4 TB/s read and written; 74 us by torch's strided byte copy), a bf16 12288 x 3072 weight per row 13.6 us
// for the rows' maxima and 18.4 us here (its second read comes from the last-level cache), 245 us by torch's operations.
constexpr uint32_t kTileRows = 32;
constexpr uint32_t kTileUnits = 32;
constexpr uint32_t kUnitPitch = kTileUnits * 16 + 16;   // a row of units in LDS: its column reads touch all banks

enum class Source { kCodes, kBf16, kFp16, kFp32 };

constexpr uint32_t source_bytes(Source s) {
    return s == Source::kCodes ? 1 : s == Source::kFp32 ? 4 : 2;
}

// 16 weights of a unit as fp32, from a buffer offset in bytes.
template <Source S>
__device__ __forceinline__ void load_unit(rsrc_t src, uint32_t off, float (&x)[16]) {
    constexpr int kLoads = static_cast<int>(source_bytes(S));
    u32x4 v[kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) v[i] = buf_load16(src, off == kOob ? kOob : off + 16u * i);
#pragma unroll
    for (int i = 0; i < kLoads; ++i)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const uint32_t bits = v[i][w];
            if constexpr (S == Source::kFp32) {
                x[4 * i + w] = __builtin_bit_cast(float, bits);
            } else if constexpr (S == Source::kBf16) {
                x[8 * i + 2 * w] = __builtin_bit_cast(float, bits << 16);
                x[8 * i + 2 * w + 1] = __builtin_bit_cast(float, bits & 0xffff0000u);
            } else {
                const half2v h = __builtin_bit_cast(half2v, bits);
                x[8 * i + 2 * w] = static_cast<float>(h[0]);
                x[8 * i + 2 * w + 1] = static_cast<float>(h[1]);
            }
        }
}

// A scale and what dividing by it takes. `amax` holds the bits of the largest magnitude; as unsigned integers the
// magnitudes order as they do as floats, with NaN above all. amax > 0: the scale is amax times the fp32 reciprocal of
// the format's largest value (what torch's division by a number does on the GPU); otherwise, NaN included, 1.
struct Scale {
    float value;
    float reciprocal;
    bool fast;   // amax finite and the scale far from the ends of fp32's range: Markstein's division below is exact
};

template <bool kE5M2>
__device__ __forceinline__ Scale make_scale(uint32_t amax) {
    constexpr float kInverseMax = 1.0f / (kE5M2 ? 57344.0f : 448.0f);
    const float a = __builtin_bit_cast(float, amax);
    Scale s;
    s.value = a > 0.0f ? a * kInverseMax : 1.0f;
    s.reciprocal = 1.0f / s.value;
    s.fast = amax < 0x7f800000u && s.value >= 0x1p-60f && s.value <= 0x1p60f;
    return s;
}

// x / s rounded to nearest even. Markstein's division (IBM J. Res. Dev. 34(1), 1990): with y = RN(1 / s), one step on
// q = RN(x y) gives a quotient within an ulp, and a second one the correctly rounded quotient; 5 instructions against
// about 14 of a full division. Residuals are exact while x is above 2^-100; below, the quotient is under every code
// and only its sign counts, hence the copysign.
__device__ __forceinline__ float divide(float x, const Scale& s) {
    float q = x * s.reciprocal;
    q = __builtin_fmaf(__builtin_fmaf(-q, s.value, x), s.reciprocal, q);
    q = __builtin_fmaf(__builtin_fmaf(-q, s.value, x), s.reciprocal, q);
    return __builtin_copysignf(q, x);
}

// Four quotients -> four codes, rounded to nearest even. NaN and e4m3 overflow give 0x7f with the sign, e5m2 overflow
// infinity, as a tensor cast does; only the slow path meets them.
template <bool kE5M2>
__device__ __forceinline__ uint32_t to_codes(const float (&q)[4]) {
    int d = 0;
    if constexpr (kE5M2) {
        d = __builtin_amdgcn_cvt_pk_bf8_f32(q[0], q[1], d, false);
        d = __builtin_amdgcn_cvt_pk_bf8_f32(q[2], q[3], d, true);
    } else {
        d = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], d, false);
        d = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], d, true);
    }
    return static_cast<uint32_t>(d);
}

template <bool kE5M2>
__device__ __forceinline__ uint32_t special_code(float q, uint32_t code) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, q);
    const uint32_t magnitude = bits & 0x7fffffffu;
    const uint32_t sign = (bits >> 24) & 0x80u;
    if (magnitude > 0x7f800000u) return sign | 0x7fu;
    // the least magnitude that rounds past the largest value: 61440 (the tie goes to infinity), above 464
    if constexpr (kE5M2) {
        return magnitude >= 0x47700000u ? sign | 0x7cu : code;
    } else {
        return magnitude > 0x43e80000u ? sign | 0x7fu : code;
    }
}

template <bool kE5M2>
__device__ __forceinline__ u32x4 quantize_unit(const float (&x)[16], const Scale& s) {
    u32x4 out;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        float q[4];
        if (s.fast) {
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] = divide(x[4 * w + i], s);
            out[w] = to_codes<kE5M2>(q);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) q[i] = x[4 * w + i] / s.value;
            const uint32_t codes = to_codes<kE5M2>(q);
            uint32_t d = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) d |= special_code<kE5M2>(q[i], (codes >> (8 * i)) & 0xffu) << (8 * i);
            out[w] = d;
        }
    }
    return out;
}

// amax (quantizing sources): the bits of each row's largest magnitude, or (per tensor) kAmaxParts partial ones of the
// whole weight. scale: where to write the scale, N or one.
constexpr uint32_t kAmaxParts = 1024;

template <Source S, bool kE5M2, bool kPerRow>
__global__ __launch_bounds__(kPrepackThreads) void pack_rows_kernel(const uint8_t* w, const uint32_t* amax,
                                                                     float* scale, uint8_t* out, uint32_t N,
                                                                     uint32_t units, uint32_t units_pad,
                                                                     uint32_t unit_tiles) {
    __shared__ __attribute__((aligned(16))) uint8_t tile[kTileRows * kUnitPitch];
    const uint32_t t = threadIdx.x;
    const uint32_t u0 = blockIdx.x % unit_tiles * kTileUnits;
    const uint32_t n0 = blockIdx.x / unit_tiles * kTileRows;
    constexpr uint32_t kUnitBytes = 16u * source_bytes(S);
    constexpr uint32_t kPasses = kTileRows * kTileUnits / kPrepackThreads;   // 4: work-item t, rows t / 32 + 8 i
    const uint32_t u = u0 + t % kTileUnits;
    const auto offset = [&](uint32_t n) { return n < N && u < units ? (n * units + u) * kUnitBytes : kOob; };
    const rsrc_t src = make_rsrc(w, N * units * kUnitBytes);
    u32x4 code[kPasses];
    if constexpr (S == Source::kCodes) {
#pragma unroll
        for (uint32_t i = 0; i < kPasses; ++i) code[i] = buf_load16(src, offset(n0 + t / kTileUnits + 8u * i));
    } else {
        Scale whole;
        if constexpr (!kPerRow) {
            // every workgroup joins the partial maxima: 4 KiB from L2
            __shared__ uint32_t top[kPrepackThreads / kWave];
            uint32_t most = 0;
#pragma unroll
            for (uint32_t i = 0; i < kAmaxParts / kPrepackThreads; ++i) most = max(most, amax[t + i * kPrepackThreads]);
#pragma unroll
            for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, d)));
            if (t % kWave == 0) top[t / kWave] = most;
            __syncthreads();
            whole = make_scale<kE5M2>(max(max(top[0], top[1]), max(top[2], top[3])));
            if (blockIdx.x == 0 && t == 0) scale[0] = whole.value;
        }
#pragma unroll
        for (uint32_t i = 0; i < kPasses; ++i) {
            const uint32_t n = n0 + t / kTileUnits + 8u * i;
            float x[16];
            load_unit<S>(src, offset(n), x);
            Scale s = whole;
            if constexpr (kPerRow) {
                s = make_scale<kE5M2>(n < N ? amax[n] : 0u);
                if (u0 == 0 && t % kTileUnits == 0 && n < N) scale[n] = s.value;
            }
            code[i] = quantize_unit<kE5M2>(x, s);
        }
    }
#pragma unroll
    for (uint32_t i = 0; i < kPasses; ++i) {
        *reinterpret_cast<u32x4*>(tile + (t / kTileUnits + 8u * i) * kUnitPitch + t % kTileUnits * 16u) = code[i];
    }
    __syncthreads();
    const rsrc_t dst = make_rsrc(out, units_pad * N * 16u);
    const uint32_t n = n0 + t % kTileRows;
#pragma unroll
    for (uint32_t i = 0; i < kPasses; ++i) {
        const uint32_t v = t / kTileRows + 8u * i;
        const u32x4 unit = *reinterpret_cast<const u32x4*>(tile + t % kTileRows * kUnitPitch + v * 16u);
        const uint32_t off = n < N && u0 + v < units_pad ? ((u0 + v) * N + n) * 16u : kOob;
        __builtin_amdgcn_raw_buffer_store_b128(unit, dst, static_cast<int>(off), 0, 0);
    }
}

// The largest magnitude of 16 weights' worth of bits, as an unsigned integer.
template <Source S>
__device__ __forceinline__ uint32_t unit_amax(rsrc_t src, uint32_t off) {
    float x[16];
    load_unit<S>(src, off, x);
    uint32_t most = 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) most = max(most, __builtin_bit_cast(uint32_t, x[i]) & 0x7fffffffu);
    return most;
}

// One wave per row: amax[n]. HBM-bound.
template <Source S>
__global__ __launch_bounds__(kPrepackThreads) void row_amax_kernel(const uint8_t* w, uint32_t* amax, uint32_t N,
                                                                    uint32_t units) {
    constexpr uint32_t kUnitBytes = 16u * source_bytes(S);
    const uint32_t lane = threadIdx.x % kWave;
    const uint32_t n = blockIdx.x * (kPrepackThreads / kWave) + threadIdx.x / kWave;
    if (n >= N) return;
    const rsrc_t src = make_rsrc(w, N * units * kUnitBytes);
    uint32_t most = 0;
#pragma unroll 4
    for (uint32_t u = lane; u < units; u += kWave) most = max(most, unit_amax<S>(src, (n * units + u) * kUnitBytes));
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, d)));
    if (lane == 0) amax[n] = most;
}

// kAmaxParts workgroups over the whole weight: amax[part].
template <Source S>
__global__ __launch_bounds__(kPrepackThreads) void part_amax_kernel(const uint8_t* w, uint32_t* amax, uint32_t total) {
    constexpr uint32_t kUnitBytes = 16u * source_bytes(S);
    __shared__ uint32_t top[kPrepackThreads / kWave];
    const uint32_t t = threadIdx.x;
    const rsrc_t src = make_rsrc(w, total * kUnitBytes);
    uint32_t most = 0;
#pragma unroll 4
    for (uint32_t u = blockIdx.x * kPrepackThreads + t; u < total; u += kAmaxParts * kPrepackThreads) {
        most = max(most, unit_amax<S>(src, u * kUnitBytes));
    }
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(most, d)));
    if (t % kWave == 0) top[t / kWave] = most;
    __syncthreads();
    if (t == 0) amax[blockIdx.x] = max(max(top[0], top[1]), max(top[2], top[3]));
}

// The sizes pack_rows_kernel takes: whole units, 32-bit buffer offsets on both sides.
bool rows_ok(const void* w, const void* out, int64_t N, int64_t K, int64_t bytes) {
    if (N < 1 || K < 16 || K % 16 != 0 || !w || !out) return false;
    if ((reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) & 15u) return false;
    return N * K * bytes < (int64_t{1} << 31) && (K + 127) / 128 * 128 * N < (int64_t{1} << 31);
}

template <Source S, bool kE5M2, bool kPerRow>
void launch_pack_rows(const void* w, const uint32_t* amax, float* scale, uint8_t* out, int64_t N, int64_t K,
                      hipStream_t stream) {
    const uint32_t units_pad = static_cast<uint32_t>((K + 127) / 128 * 8);
    const uint32_t unit_tiles = (units_pad + kTileUnits - 1) / kTileUnits;
    const uint32_t row_tiles = static_cast<uint32_t>((N + kTileRows - 1) / kTileRows);
    hipLaunchKernelGGL((pack_rows_kernel<S, kE5M2, kPerRow>), dim3(unit_tiles * row_tiles), dim3(kPrepackThreads), 0,
                       stream, static_cast<const uint8_t*>(w), amax, scale, out, static_cast<uint32_t>(N),
                       static_cast<uint32_t>(K / 16), units_pad, unit_tiles);
}

template <Source S>
void launch_quantize(const void* w, uint32_t* amax, float* scale, uint8_t* out, int64_t N, int64_t K, bool e5m2,
                     bool per_row, hipStream_t stream) {
    const uint8_t* const src = static_cast<const uint8_t*>(w);
    const uint32_t units = static_cast<uint32_t>(K / 16);
    if (per_row) {
        constexpr uint32_t kRows = kPrepackThreads / kWave;
        hipLaunchKernelGGL((row_amax_kernel<S>), dim3((static_cast<uint32_t>(N) + kRows - 1) / kRows),
                           dim3(kPrepackThreads), 0, stream, src, amax, static_cast<uint32_t>(N), units);
        if (e5m2) {
            launch_pack_rows<S, true, true>(w, amax, scale, out, N, K, stream);
        } else {
            launch_pack_rows<S, false, true>(w, amax, scale, out, N, K, stream);
        }
    } else {
        hipLaunchKernelGGL((part_amax_kernel<S>), dim3(kAmaxParts), dim3(kPrepackThreads), 0, stream, src, amax,
                           static_cast<uint32_t>(N) * units);
        if (e5m2) {
            launch_pack_rows<S, true, false>(w, amax, scale, out, N, K, stream);
        } else {
            launch_pack_rows<S, false, false>(w, amax, scale, out, N, K, stream);
        }
    }
}

}  // namespace
}  // namespace feather

extern "C" bool feather_prepack_b(const uint8_t* b, uint8_t* b_prepacked, int64_t K, int64_t N, hipStream_t stream) {
    if (K < 1 || N < 8 || N % 8 != 0 || !b || !b_prepacked) return false;
    if ((reinterpret_cast<uintptr_t>(b) & 7u) || (reinterpret_cast<uintptr_t>(b_prepacked) & 15u)) return false;
    const int64_t k_pad = (K + 127) / 128 * 128;
    if (k_pad * N >= (int64_t{1} << 31)) return false;  // 32-bit buffer offsets
    const uint32_t chunks = static_cast<uint32_t>(k_pad / 16);
    const uint32_t col_tiles = static_cast<uint32_t>((N + feather::kPrepackCols - 1) / feather::kPrepackCols);
    hipLaunchKernelGGL(feather::prepack_kernel, dim3(chunks * col_tiles), dim3(feather::kPrepackThreads), 0, stream, b,
                       b_prepacked, static_cast<uint32_t>(K), static_cast<uint32_t>(N), col_tiles, chunks);
    return true;
}

extern "C" bool feather_prepack_rows(const uint8_t* w, uint8_t* out, int64_t N, int64_t K, hipStream_t stream) {
    using namespace feather;
    if (!rows_ok(w, out, N, K, 1)) return false;
    launch_pack_rows<Source::kCodes, false, false>(w, nullptr, nullptr, out, N, K, stream);
    return true;
}

extern "C" bool feather_quantize_rows(const void* w, int source, uint8_t* out, float* scale, uint32_t* amax, int64_t N,
                                      int64_t K, bool use_fp8_e5m2, bool per_row, hipStream_t stream) {
    using namespace feather;
    if (source < 0 || source > 2 || !scale || !amax || !rows_ok(w, out, N, K, source == 2 ? 4 : 2)) return false;
    switch (source) {
        case 0: launch_quantize<Source::kBf16>(w, amax, scale, out, N, K, use_fp8_e5m2, per_row, stream); break;
        case 1: launch_quantize<Source::kFp16>(w, amax, scale, out, N, K, use_fp8_e5m2, per_row, stream); break;
        default: launch_quantize<Source::kFp32>(w, amax, scale, out, N, K, use_fp8_e5m2, per_row, stream);
    }
    return true;
}
