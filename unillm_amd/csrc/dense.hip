// dense.hip -- dense (GGML F32 / F16 / BF16) projection weights.
//
// candle's QMatMul::from_arc dequantizes an F32 / F16 / BF16 tensor to an f32
// tensor, and its forward multiplies in f32 (the Tensor variant: x.matmul(w.t())).
// The reference's loader wraps every *_proj.weight / lm_head.weight tensor in a
// QMatMul whatever its GGML type (crates/runtime/src/weight_loader_core.rs:554-571),
// so a GGUF with F16 projections takes this variant.  A weight is held in its own type
// (a widening to f32 would double the bytes a decode step streams) as rows of
// row_bytes, k padded with zeros to a multiple of 64, and the product is f32:
//
//  - dense_gemv_kernel (m <= 8 where x fits in LDS): the weights widen in registers
//    and every product is an f32 FMA.  Bound by the weight stream.
//  - dense_gemm_kernel: bf16 matrix cores at f32's precision.  x is split exactly into
//    three bf16 parts (xsplit_kernel); a BF16 weight is one part as it stands, an F16 weight
//    is split in registers into two, an F32 weight into three.  The products of parts are
//    summed in f32, the leading one and the small ones each in a sum of their own: 3 a
//    weight for BF16 (all of them), 5 for F16 and 6 for F32 (the ones left out come to
//    0.5 and 0.9 times 2^-24 of the product at most, either sign).  gfx950's 16-bit matrix
//    cores run 16 times its f32 ones, so up to 6 of them are still 2.7 times faster, and the
//    error against f64 is below an f32 GEMM's, which rounds once a k
//    (profiles/dense_weights.md has both).  bf16 has f32's range: a row of x keeps all its
//    bits however far apart its values are.  (f16 parts, three products for F16, hold no
//    element below 2^-40 of its row's largest: behind an outlier of 1e9 in a column of zero
//    weights the product was off by 5.6e-4.)
//  - dense_short_kernel (k <= 4, m > 8): f32 FMAs.  So short a sum has few roundings in f32
//    too, and the matrix cores' sums, which do not round to nearest, are the less exact ones
//    (BF16, k 1 / 2 / 3, against f64: 3.3e-8 / 3.3e-8 / 3.2e-8, f32 2.6e-8 / 3.1e-8 / 3.6e-8).
//
// All give the same bits on every call (no atomics; split-k slabs add in order), and
// an F16 or BF16 weight on the GEMV the same bits as its widened F32 copy.  A
// non-finite x or weight makes 0 * inf terms in the split products: an output that comes out
// non-finite is recomputed as a plain f32 dot (dense_dot), so infinities propagate as f32
// products would.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "internal.hpp"
#include "lds.hpp"
#include "split.hpp"

namespace unillm {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kKPad = 64;  // rows are padded with zeros to a multiple of this many weights

int64_t padded_k(int64_t k) { return (k + kKPad - 1) / kKPad * kKPad; }

// ---- upload, dequant, layer norm ---------------------------------------------------------

// dst row r (row_bytes) <- src row r (k elements), a workgroup a row at a time; the padding
// was zeroed when the weight was allocated
template <class T>
__global__ __launch_bounds__(256) void dense_upload_kernel(const T* __restrict__ src,
                                                           uint8_t* __restrict__ dst, int64_t n,
                                                           int64_t k, int64_t row_bytes) {
    for (int64_t r = blockIdx.x; r < n; r += gridDim.x) {
        const T* sr = src + r * k;
        T* dr = reinterpret_cast<T*>(dst + r * row_bytes);
        for (int64_t i = threadIdx.x; i < k; i += 256) dr[i] = sr[i];
    }
}

// weight i of a row
template <int QT>
__device__ __forceinline__ float widen1(const uint8_t* row, int64_t i) {
    if constexpr (QT == UNILLM_QTYPE_F32) return reinterpret_cast<const float*>(row)[i];
    const uint16_t v = reinterpret_cast<const uint16_t*>(row)[i];
    if constexpr (QT == UNILLM_QTYPE_F16) return __half2float(__ushort_as_half(v));
    return __uint_as_float((uint32_t)v << 16);
}

// out[n, k] f32 <- the weight's values, widened exactly
template <int QT>
__global__ __launch_bounds__(256) void dense_widen_kernel(const uint8_t* __restrict__ base,
                                                          int64_t row_bytes,
                                                          float* __restrict__ out, int64_t n,
                                                          int64_t k) {
    const int64_t count = n * k;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (int64_t)gridDim.x * blockDim.x)
        out[i] = widen1<QT>(base + i / k * row_bytes, i % k);
}

// out[r] = (x[r] - mean) / sqrt(var + eps) * gamma (+ beta), one workgroup a row: the
// mean, then the mean of the squared deviations (ops_fn::layer_norm's two passes,
// tensor_core.rs:973-1008), in f32
__global__ __launch_bounds__(256) void norm_rows_kernel(const float* __restrict__ x, int64_t k,
                                                        NormArgs norm, float* __restrict__ out) {
    __shared__ float red[4];
    const float* xr = x + (int64_t)blockIdx.x * k;
    float* orow = out + (int64_t)blockIdx.x * k;
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    auto block_sum = [&](float v) {
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (lane == 0) red[wv] = v;
        __syncthreads();
        const float s = (red[0] + red[1]) + (red[2] + red[3]);
        __syncthreads();
        return s;
    };
    float acc = 0.0f;
    for (int64_t i = t; i < k; i += 256) acc += xr[i];
    const float mean = block_sum(acc) / (float)k;
    acc = 0.0f;
    for (int64_t i = t; i < k; i += 256) {
        const float d = xr[i] - mean;
        acc += d * d;
    }
    const float sd = sqrtf(block_sum(acc) / (float)k + norm.eps);
    for (int64_t i = t; i < k; i += 256)
        orow[i] = (xr[i] - mean) / sd * norm.gamma[i] + (norm.beta ? norm.beta[i] : 0.0f);
}

__device__ __forceinline__ bool non_finite(float v) {
    return (__float_as_uint(v) & 0x7F800000u) == 0x7F800000u;
}

// ---- GEMV, m <= 8 ------------------------------------------------------------------------
// One workgroup of 16 waves a CU; a wave takes rows wave, wave + W, ...; lane l holds
// the 8 consecutive weights of groups l, l + 64, ... of the row (one 16-byte load; two
// for F32), U groups requested ahead of the ones being multiplied, so 128 bytes a lane
// stay in flight across row ends.  x sits in LDS as two planes of 4 floats a group:
// every read is 16 consecutive bytes a lane, free of bank conflicts.  Bound by the
// weight stream at one token: F16 k4096 n11008 (90 MB) 16.3 us in the kernel (5.5 TB/s; 17.9 a
// call in an eager loop), against 228 us as an f32 library GEMM of rows widened to f32.  From three tokens on, by x's reads from
// LDS (32 bytes a token for 8 weights): two of the wave's rows are multiplied by each read,
// with half the groups in flight for each.  F16 m4 29.4 -> 24.1 us, m8 45.4 -> 33.0; F32 m8
// 53.6 -> 41.1 (a single last row runs alone: no products are made for rows past the end).
// x is staged 16 bytes a lane where its rows allow it (m1 18.8 -> 18.1, called eagerly).
constexpr int kGemvThreads = 1024;
constexpr int64_t kGemvLds = 128 << 10;

template <int QT>
struct Row8 {  // 8 weights as loaded
    static constexpr int L = QT == UNILLM_QTYPE_F32 ? 2 : 1;
    u32x4 v[L];
};

template <int QT>
__device__ __forceinline__ Row8<QT> load8(const uint8_t* row, int g) {
    Row8<QT> r;
#pragma unroll
    for (int i = 0; i < Row8<QT>::L; ++i)
        r.v[i] = *reinterpret_cast<const u32x4*>(row + ((int64_t)g * Row8<QT>::L + i) * 16);
    return r;
}

template <int QT>
__device__ __forceinline__ float elem8(const Row8<QT>& r, int e) {
    if constexpr (QT == UNILLM_QTYPE_F32) return __uint_as_float(r.v[e / 4][e % 4]);
    const uint32_t u = r.v[0][e / 2];
    if constexpr (QT == UNILLM_QTYPE_F16)
        return (float)__builtin_bit_cast(_Float16, (uint16_t)(e % 2 ? u >> 16 : u & 0xFFFFu));
    return __uint_as_float(e % 2 ? u & 0xFFFF0000u : u << 16);
}

// The plain f32 dot of one output, in k order: what an output that came out non-finite is
// recomputed with.  16 products' operands at a time in flight (more take registers from
// dense_sum_kernel's waves), and done once the sum is NaN.
template <int QT>
__device__ __noinline__ float dense_dot(const float* x, const uint8_t* row, int64_t k) {
    float s = 0.0f;
    int64_t i = 0;
    for (; i + 16 <= k && s == s; i += 16) {
        Row8<QT> w[2];
        float v[16];
#pragma unroll
        for (int u = 0; u < 2; ++u) w[u] = load8<QT>(row, (int)(i / 8) + u);
        __builtin_memcpy(v, x + i, sizeof(v));
#pragma unroll
        for (int e = 0; e < 16; ++e) s = fmaf(v[e], elem8<QT>(w[e / 8], e % 8), s);
    }
    for (; i < k && s == s; ++i) s = fmaf(x[i], widen1<QT>(row, i), s);
    return s;
}

// A non-finite output again (nan: its row of x holds a NaN).  BF16 m512 k4096 n11008, us a
// call (169 all finite): every row with a NaN 177, one row with an infinity 509, every row
// 10700.
template <int QT>
__device__ __forceinline__ float dense_redo(uint32_t nan, const float* x, const uint8_t* row,
                                            int64_t k) {
    return nan ? __builtin_nanf("") : dense_dot<QT>(x, row, k);
}

// M: the token count the code is built for (m <= M; x past m is zero and not stored)
template <int QT, int M>
__global__ __launch_bounds__(kGemvThreads, 1) void dense_gemv_kernel(
    const uint8_t* __restrict__ base, int64_t row_bytes, const float* __restrict__ x, int m,
    int64_t n, int k, float* __restrict__ y, int add) {
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    f32x4* xs = reinterpret_cast<f32x4*>(smem);  // [M][2][G]
    const int G = (k + 7) / 8;
    const int lane = threadIdx.x & 63;
    const int64_t wave =
        (int64_t)__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * gridDim.x + blockIdx.x;
    const int64_t waves = (int64_t)(kGemvThreads / 64) * gridDim.x;
    constexpr int R = M >= 4 ? 2 : 1;  // rows at a time
    constexpr int U = (QT == UNILLM_QTYPE_F32 ? 4 : M <= 4 ? 8 : 4) / R;
    const int T = (G + 64 * U - 1) / (64 * U);  // batches of U groups a lane in a row

    auto request = [&](int64_t row, int t, Row8<QT>(&r)[R][U]) {
#pragma unroll
        for (int i = 0; i < R; ++i) {
            if (row + i * waves >= n) break;
            const uint8_t* p = base + (row + i * waves) * row_bytes;
#pragma unroll
            for (int u = 0; u < U; ++u) r[i][u] = load8<QT>(p, min((t * U + u) * 64 + lane, G - 1));
        }
    };
    // the first batch is in flight while x is staged
    Row8<QT> cur[R][U] = {}, nxt[R][U] = {};
    request(wave, 0, cur);
    const bool vec = k % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
#pragma unroll
    for (int t = 0; t < M; ++t) {
        const float* xt = x + (int64_t)t * k;
        for (int q = threadIdx.x; q < 2 * G; q += kGemvThreads) {
            f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (t < m) {
                if (vec) {
                    if (4 * q < k) v = reinterpret_cast<const f32x4*>(xt)[q];
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (4 * q + e < k) v[e] = xt[4 * q + e];
                }
            }
            xs[(t * 2 + q % 2) * G + q / 2] = v;
        }
    }
    __syncthreads();

    float acc[R][M];
    // batch b of the first `rows` rows
    auto batch = [&](int b, auto rows) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int g = (b * U + u) * 64 + lane;
            if (g < G) {
#pragma unroll
                for (int t = 0; t < M; ++t) {
                    const f32x4 lo = xs[(t * 2) * G + g], hi = xs[(t * 2 + 1) * G + g];
#pragma unroll
                    for (int i = 0; i < rows.value; ++i) {
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i][t] = fmaf(elem8<QT>(cur[i][u], e), lo[e], acc[i][t]);
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            acc[i][t] = fmaf(elem8<QT>(cur[i][u], 4 + e), hi[e], acc[i][t]);
                    }
                }
            }
        }
    };
    for (int64_t row0 = wave; row0 < n; row0 += R * waves) {
        const bool whole = row0 + (R - 1) * waves < n;
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int t = 0; t < M; ++t) acc[i][t] = 0.0f;
        for (int b = 0; b < T; ++b) {
            const bool last = b + 1 == T;
            request(last ? row0 + R * waves : row0, last ? 0 : b + 1, nxt);
            if (whole) batch(b, std::integral_constant<int, R>{});
            else batch(b, std::integral_constant<int, 1>{});
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int u = 0; u < U; ++u) cur[i][u] = nxt[i][u];
        }
#pragma unroll
        for (int i = 0; i < R; ++i) {
            const int64_t row = row0 + i * waves;
            if (row >= n) break;
#pragma unroll
            for (int t = 0; t < M; ++t) {
                float s = acc[i][t];
                for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
                if (lane == 0 && t < m) {
                    float* dst = y + (int64_t)t * n + row;
                    *dst = add ? *dst + s : s;
                }
            }
        }
    }
}

int64_t gemv_m(int64_t m) { return m <= 2 ? m : m <= 4 ? 4 : 8; }
int64_t gemv_lds(int64_t m, int64_t k) { return gemv_m(m) * ((k + 7) / 8) * 32; }

// x in LDS: 8 tokens take k <= 4096, 4 take 8192, one 32768
bool dense_gemv_supports(const QWeight& w, int64_t m) {
    return m <= 8 && gemv_lds(m, w.k) <= kGemvLds;
}

template <int QT, int M>
hipError_t launch_gemv_m(const QWeight& w, const float* x, int64_t m, float* y, hipStream_t s,
                         int add) {
    static const bool attr = hipFuncSetAttribute((const void*)dense_gemv_kernel<QT, M>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 (int)kGemvLds) == hipSuccess;
    if (!attr) return hipErrorInvalidValue;
    // wave numbers run across workgroups, so few rows still spread over the CUs
    const int blocks = (int)std::min<int64_t>(device_info().cu_count, w.n);
    dense_gemv_kernel<QT, M><<<blocks, kGemvThreads, gemv_lds(m, w.k), s>>>(
        w.base, w.row_bytes, x, (int)m, w.n, (int)w.k, y, add);
    return hipGetLastError();
}

template <int QT>
hipError_t launch_gemv_qt(const QWeight& w, const float* x, int64_t m, float* y, hipStream_t s,
                          int add) {
    switch (gemv_m(m)) {
        case 1: return launch_gemv_m<QT, 1>(w, x, m, y, s, add);
        case 2: return launch_gemv_m<QT, 2>(w, x, m, y, s, add);
        case 4: return launch_gemv_m<QT, 4>(w, x, m, y, s, add);
        default: return launch_gemv_m<QT, 8>(w, x, m, y, s, add);
    }
}

// ---- k <= 4, m > 8 -----------------------------------------------------------------------
// A thread a column: its weights in registers, f32 FMAs over 64 rows of x.  Bound by the
// store of y.
constexpr int kShortK = 4;

template <int QT>
__global__ __launch_bounds__(256) void dense_short_kernel(const uint8_t* __restrict__ base,
                                                          int64_t row_bytes,
                                                          const float* __restrict__ x, int64_t m,
                                                          int64_t n, int k, float* __restrict__ y,
                                                          int add) {
    const int64_t col = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (col >= n) return;
    float w[kShortK];  // (zeros past k: the row's padding)
#pragma unroll
    for (int i = 0; i < kShortK; ++i)
        w[i] = widen1<QT>(base + col * row_bytes, i);
    for (int64_t row0 = (int64_t)blockIdx.y * 64; row0 < m; row0 += (int64_t)gridDim.y * 64)
        for (int64_t row = row0; row < min(row0 + 64, m); ++row) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < kShortK; ++i)
                if (i < k) s = fmaf(x[row * k + i], w[i], s);
            float* dst = y + row * n + col;
            *dst = add ? *dst + s : s;
        }
}

// ---- x in three bf16 parts ---------------------------------------------------------------
// xp[p][m][kp]: x = part 0 + part 1 + part 2 exactly (rows padded with zeros to kp), each
// part what is left rounded to bf16 (split.hpp; a finite value keeps a finite part 0).  A
// non-finite value keeps its kind in part 0, the others zero.  nan_row[r]: whether row r holds
// a NaN (its outputs then are NaN, without a look at the weights).  One workgroup a row; bound
// by its bytes (4 in, 6 out an element).
__global__ __launch_bounds__(256) void xsplit_kernel(const float* __restrict__ x, int64_t k,
                                                     int64_t kp, uint16_t* __restrict__ xp,
                                                     int64_t plane,
                                                     uint32_t* __restrict__ nan_row) {
    const float* xr = x + (int64_t)blockIdx.x * k;
    uint16_t* o = xp + (int64_t)blockIdx.x * kp;
    int nan = 0;
    for (int64_t i = threadIdx.x; i < kp; i += 256) {
        const float v = i < k ? xr[i] : 0.0f;
        nan |= v != v;
        const uint32_t u = __float_as_uint(v);
        uint16_t p0 = (uint16_t)pack_bf16(v, 0.0f), p1 = 0, p2 = 0;
        if (!non_finite(v)) {
            if ((p0 & 0x7F80u) == 0x7F80u) p0 = (uint16_t)(u >> 16);  // (rounded to infinity)
            const float r1 = v - bf16_lo(p0);
            p1 = (uint16_t)pack_bf16(r1, 0.0f);
            p2 = (uint16_t)pack_bf16(r1 - bf16_lo(p1), 0.0f);
        }
        o[i] = p0;
        o[plane + i] = p1;
        o[2 * plane + i] = p2;
    }
    nan = __syncthreads_or(nan);
    if (threadIdx.x == 0) nan_row[blockIdx.x] = nan;
}

// ---- GEMM --------------------------------------------------------------------------------
// Tile BM x BN, k in steps of 32, eight waves in a 2 x 4 grid of (BM / 2) x (BN / 4)
// blocks of 16 x 16 x 32 MFMAs.  Operands reach LDS by direct global -> LDS loads
// through a ring of 4 stages; a step's first fragments are read during the
// last MFMAs of the step before, so a step starts straight into its MFMAs:
//   A  [3 parts][BM rows][64 B], the 16-byte chunk c of row r in slot c ^ f(r / 4 % 4),
//      f = 0 3 2 1: the 16 lanes that an LDS read serves together touch all banks once;
//   B  [BN rows][64 B], the same (F32: [BN][128 B], chunk c in slot c ^ r % 8).
// Bound by the matrix cores (BF16 at three products a weight, m512 k4096 n11008: 159 us a
// call, 290 TFLOP/s of f32 product, against 451 us as an f32 library GEMM; 172 tiles on 256
// CUs.  F16 at five and the split of its weights: 251) and by the weight stream and the
// split's fixed cost at few rows (m16: 37 us, F16 47).
template <int QT, int BM>
struct DTile {
    static constexpr bool F32W = QT == UNILLM_QTYPE_F32;
    static constexpr int BN = F32W ? 128 : 256;
    static constexpr int NP = 3;
    static constexpr int A = NP * BM * 64;
    static constexpr int B = BN * (F32W ? 128 : 64);
    static constexpr int STAGE = A + B;
    static constexpr int STAGES = 4;
    static constexpr int BYTES = STAGES * STAGE;
    static constexpr int AI = A / 1024, BI = B / 1024;     // direct loads a stage
    static constexpr int AW = (AI + 7) / 8, BW = BI / 8;   // a wave
    static constexpr int DMA = AW + BW;
    static constexpr int TI = BM / 32, TJ = BN / 64;       // 16 x 16 tiles a wave
};

__device__ __forceinline__ uint32_t swz64(uint32_t row) { return (4u - ((row >> 2) & 3u)) & 3u; }

__device__ __forceinline__ f32x4 mfma_parts(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// A fragment's 8 weights -> their bf16 parts: three of an F32, two of an F16 (8 of its 11
// bits, the rest), itself of a BF16 (an infinity's or a NaN's lower parts come out NaN: the
// output is recomputed)
template <int QT>
__device__ __forceinline__ void split_weights(const u32x4 (&w)[QT == UNILLM_QTYPE_F32 ? 2 : 1],
                                              u32x4 (&p)[3]) {
    if constexpr (QT == UNILLM_QTYPE_BF16) p[0] = w[0];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
        if constexpr (QT == UNILLM_QTYPE_F32) {
            uint32_t p0, p1, p2;
            split2(w[h / 2][2 * (h % 2)], w[h / 2][2 * (h % 2) + 1], p0, p1, p2);
            p[0][h] = p0;
            p[1][h] = p1;
            p[2][h] = p2;
        } else if constexpr (QT == UNILLM_QTYPE_F16) {
            const uint32_t u = w[0][h];  // (a bit cast of the element itself takes element 0)
            const f16x2 v = __builtin_bit_cast(f16x2, u);
            const float a = (float)v[0], b = (float)v[1];
            const uint32_t p0 = pack_bf16(a, b);
            p[0][h] = p0;
            p[1][h] = pack_bf16(a - bf16_lo(p0), b - bf16_hi(p0));
        }
    }
}

template <int QT, int BM>
__global__ __launch_bounds__(512, 1) void dense_gemm_kernel(
    const uint8_t* __restrict__ base, int64_t row_bytes, const uint16_t* __restrict__ xp,
    int64_t plane, int64_t kp, const uint32_t* __restrict__ nan_row,
    const float* __restrict__ x, int64_t k, float* __restrict__ y, int64_t M,
    int64_t N, int tiles_n, int tiles, int units_pad, int S, int add, float* __restrict__ part) {
    using D = DTile<QT, BM>;
    constexpr int TI = D::TI, TJ = D::TJ, NP = D::NP;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

    // unit u = (k slice sp, m-tile, n-tile), a contiguous run of units per XCD
    const int u = (blockIdx.x % 8) * (units_pad / 8) + blockIdx.x / 8;
    if (u >= tiles * S) return;
    const int sp = u / tiles, t = u % tiles;
    const int64_t m0 = (int64_t)(t / tiles_n) * BM, n0 = (int64_t)(t % tiles_n) * D::BN;
    const int lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rw = wv / 4, cw = wv % 4;
    // this slice's steps, always whole pairs
    const int kpairs = (int)(kp / kKPad);
    const int ks0 = 2 * (int)((int64_t)sp * kpairs / S);
    const int nks = 2 * (int)((int64_t)(sp + 1) * kpairs / S) - ks0;

    // direct-load sources at step 0 (rows past the end re-read the last row)
    const uint8_t* asrc[D::AW];
    const uint8_t* bsrc[D::BW];
    uint32_t adst[D::AW], bdst[D::BW];
#pragma unroll
    for (int q = 0; q < D::AW; ++q) {
        const int i = (wv * D::AW + q) % D::AI;  // an uneven split loads a part twice
        const int r = i % (BM / 16) * 16 + lane / 4;
        const int c = (lane % 4) ^ swz64(r);
        asrc[q] = reinterpret_cast<const uint8_t*>(
            xp + (i / (BM / 16)) * plane + min(m0 + r, M - 1) * kp + c * 8);
        adst[q] = i * 1024;
    }
#pragma unroll
    for (int q = 0; q < D::BW; ++q) {
        const int i = wv * D::BW + q;
        const int r = D::F32W ? i * 8 + lane / 8 : i * 16 + lane / 4;
        const int c = D::F32W ? (lane % 8) ^ (r % 8) : (lane % 4) ^ swz64(r);
        bsrc[q] = base + min(n0 + r, N - 1) * row_bytes + c * 16;
        bdst[q] = D::A + i * 1024;
    }
    auto issue = [&](int j) {  // the direct loads of step ks0 + j
        uint8_t* st = smem + (j % D::STAGES) * D::STAGE;
        const int64_t ko = (int64_t)(ks0 + j) * 64;
#pragma unroll
        for (int q = 0; q < D::AW; ++q) dma16(asrc[q] + ko, st + adst[q]);
#pragma unroll
        for (int q = 0; q < D::BW; ++q) dma16(bsrc[q] + (D::F32W ? 2 * ko : ko), st + bdst[q]);
    };

    // fragment offsets in a stage: A row (BM / 2) rw + 16 i + fr, B row (BN / 4) cw + 16 j + fr
    const uint32_t g = lane / 16, fr = lane % 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;
    const uint32_t aoff = lds0 + ((BM / 2) * rw + fr) * 64 + (g ^ swz64(fr)) * 16;
    const uint32_t brow = (D::BN / 4) * cw + fr;
    const uint32_t boff0 = lds0 + D::A + (D::F32W ? brow * 128 + ((2 * g) ^ (fr % 8)) * 16
                                                  : brow * 64 + (g ^ swz64(fr)) * 16);
    const uint32_t boff1 = lds0 + D::A + brow * 128 + ((2 * g + 1) ^ (fr % 8)) * 16;

    constexpr int BL = D::F32W ? 2 : 1;
    struct Frags {
        u32x4 a[NP];       // row tile 0
        u32x4 b[TJ][BL];
    };
    auto read_first = [&](int j, Frags& f) {
        const uint32_t st = (uint32_t)((j % D::STAGES) * D::STAGE);
        constexpr_for<TJ>([&](auto J) {
            f.b[J.value][0] = lds_read128<J.value * 16 * (D::F32W ? 128 : 64)>(st + boff0);
            if constexpr (D::F32W) f.b[J.value][1] = lds_read128<J.value * 16 * 128>(st + boff1);
        });
        constexpr_for<NP>([&](auto P) { f.a[P.value] = lds_read128<P.value * BM * 64>(st + aoff); });
    };
    auto wait_first = [&](Frags& f) {
        static_assert(TJ == 4 || (TJ == 2 && BL == 2), "fragments named below");
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(f.a[0]), "+v"(f.a[1]), "+v"(f.a[2]), "+v"(f.b[0][0]),
                       "+v"(f.b[TJ == 4 ? 1 : 0][BL - 1]), "+v"(f.b[TJ == 4 ? 2 : 1][0]),
                       "+v"(f.b[TJ - 1][BL - 1]));
    };

    f32x4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 low[TI][TJ] = {};  // the small products' sums

    // prologue: three stages in flight; step 0's first fragments read
    constexpr int AHEAD = D::STAGES - 1;
#pragma unroll
    for (int d = 0; d < AHEAD; ++d)
        if (d < nks) issue(d);
    if (nks > 2) wait_vmcnt<2 * D::DMA>();
    else wait_vmcnt<D::DMA>();
    __builtin_amdgcn_s_barrier();
    Frags f0, f1;
    read_first(0, f0);
    wait_first(f0);
    // step j: wait for this wave's loads of step j + 1 and meet the others (so stage
    // j + 1 is whole, and stage j - 1, whose slot step j + 3 takes, is no longer read)
    auto step = [&](int j, Frags& f, Frags& nf) {
        if (j + 2 < nks) wait_vmcnt<D::DMA>();
        else wait_vmcnt<0>();
        __builtin_amdgcn_s_barrier();
        if (j + AHEAD < nks) issue(j + AHEAD);
        const uint32_t st = (uint32_t)((j % D::STAGES) * D::STAGE);
        u32x4 wb[TJ][NP];
#pragma unroll
        for (int q = 0; q < TJ; ++q) split_weights<QT>(f.b[q], wb[q]);
        u32x4 a[2][NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) a[0][p] = f.a[p];
        constexpr_for<TI>([&](auto I) {
            constexpr int i = I.value;
            // the reads may land in registers of products just consumed: keep the wait
            // states after an MFMA that the compiler keeps before its own LDS reads
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_nop 7");
            if constexpr (i + 1 < TI)
                constexpr_for<NP>([&](auto P) {
                    a[(i + 1) % 2][P.value] =
                        lds_read128<P.value * BM * 64 + (i + 1) * 1024>(st + aoff);
                });
            else if (j + 1 < nks)
                read_first(j + 1, nf);
            __builtin_amdgcn_sched_barrier(0);  // (left free, the reads sink behind the MFMAs)
            // the small products in sums of their own: one rounding of the large sum a 32 k (F32
            // in one sum, k 64: 1.3e-7 against 0.8e-7)
            auto small = [&](int pa, int pb) {
#pragma unroll
                for (int q = 0; q < TJ; ++q)
                    low[i][q] = mfma_parts(a[i % 2][pa], wb[q][pb], low[i][q]);
            };
#pragma unroll
            for (int q = 0; q < TJ; ++q) {
                low[i][q] = mfma_parts(a[i % 2][2], wb[q][0], low[i][q]);
                acc[i][q] = mfma_parts(a[i % 2][0], wb[q][0], acc[i][q]);
            }
            if constexpr (D::F32W) small(0, 2);
            if constexpr (QT != UNILLM_QTYPE_BF16) small(1, 1);
            small(1, 0);
            if constexpr (QT != UNILLM_QTYPE_BF16) small(0, 1);
            if constexpr (i + 1 < TI)
                asm volatile("s_waitcnt lgkmcnt(0)"
                             : "+v"(a[(i + 1) % 2][0]), "+v"(a[(i + 1) % 2][1]),
                               "+v"(a[(i + 1) % 2][2]));
            else if (j + 1 < nks)
                wait_first(nf);
        });
    };
    for (int j = 0; j < nks; j += 2) {
        step(j, f0, f1);
        step(j + 1, f1, f0);
    }

#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int q = 0; q < TJ; ++q) acc[i][q] += low[i][q];
    // epilogue: lane holds rows 4 g + e, column fr of each 16 x 16 tile
#pragma unroll
    for (int q = 0; q < TJ; ++q) {
        const int64_t col = n0 + (D::BN / 4) * cw + 16 * q + fr;
        if (col >= N) continue;
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t row = m0 + (BM / 2) * rw + 16 * i + 4 * g + e;
                if (row >= M) continue;
                if (S > 1) {
                    part[((int64_t)sp * M + row) * N + col] = acc[i][q][e];
                    continue;
                }
                float v = acc[i][q][e];
                if (non_finite(v)) v = dense_redo<QT>(nan_row[row], x + row * k, base + col * row_bytes, k);
                float* dst = y + row * N + col;
                *dst = add ? *dst + v : v;
            }
    }
}

// y (+)= the S slabs of a split k in slice order
template <int QT>
__global__ __launch_bounds__(256) void dense_sum_kernel(const float* __restrict__ part, int S,
                                                        int64_t M, int64_t N,
                                                        const uint8_t* __restrict__ base,
                                                        int64_t row_bytes,
                                                        const uint32_t* __restrict__ nan_row,
                                                        const float* __restrict__ x, int64_t k,
                                                        int add, float* __restrict__ y) {
    const int64_t MN = M * N;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < MN;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t row = i / N, col = i % N;
        float v = part[i];
        for (int sl = 1; sl < S; ++sl) v += part[sl * MN + i];
        if (non_finite(v)) v = dense_redo<QT>(nan_row[row], x + row * k, base + col * row_bytes, k);
        y[i] = add ? y[i] + v : v;
    }
}

// Tile height and k split: the cheapest of 64- and 128-row tiles with k in up to 16
// slices (at least 4 pairs of steps each, at most two workgroups a CU), by what a
// workgroup's pair of steps was measured to take (64 / 128 rows: BF16 1.5 / 2.35 us, F16
// 2.4 / 3.75, F32 1.75 / 2.65) times the rounds over the CUs, plus a split's slabs written
// and read once (3.5 TB/s) and the summing launch.  Measured against every choice, BF16 us a
// call: k4096 n11008 m300 157.9 (128 rows, 129 tiles on 256 CUs) -> 107.0 (64 rows, 215),
// m512 158.7 (128, one slice; 64: 199.8); k4096 n2048 m128 36.2 -> 29.1 (64 rows in 12).
struct DensePlan {
    int bm, S;
};
constexpr int64_t kDenseMaxSlices = 16;
constexpr int64_t kDenseMaxRounds = 2;  // workgroups a CU when k is split

int64_t dense_bn(const QWeight& w) { return w.qtype == UNILLM_QTYPE_F32 ? 128 : 256; }

DensePlan dense_plan(const QWeight& w, int64_t m) {
    const int64_t cus = device_info().cu_count, kpairs = padded_k(w.k) / kKPad;
    const int64_t tiles_n = (w.n + dense_bn(w) - 1) / dense_bn(w);
    DensePlan best{128, 1};
    int64_t least = INT64_MAX;
    for (int bm : {64, 128}) {
        const int64_t pair_ns = w.qtype == UNILLM_QTYPE_F32   ? (bm == 64 ? 1750 : 2650)
                                : w.qtype == UNILLM_QTYPE_F16 ? (bm == 64 ? 2400 : 3750)
                                                              : (bm == 64 ? 1500 : 2350);
        const int64_t tiles = (m + bm - 1) / bm * tiles_n;
        for (int64_t S = 1; S <= kDenseMaxSlices; ++S) {
            if (S > 1 && (S > kpairs / 4 || tiles * S > kDenseMaxRounds * cus)) break;
            const int64_t rounds = (tiles * S + cus - 1) / cus;
            int64_t ns = rounds * ((kpairs + S - 1) / S) * pair_ns;
            if (S > 1) ns += 3000 + S * m * w.n * 8 / 3500;
            if (ns < least) {
                least = ns;
                best = {bm, (int)S};
            }
        }
    }
    return best;
}

size_t up256(size_t b) { return (b + 255) / 256 * 256; }

// Rows of x a launch takes: their parts within 256 MiB (k 4096: 10880 rows, 85 tiles of 128),
// so that a stream's workspace, which is kept, and the launch's 2^32 threads hold any m.
int64_t dense_chunk_rows(const QWeight& w) {
    const int64_t rows = ((int64_t)256 << 20) / (6 * padded_k(w.k));
    return rows >= 128 ? rows / 128 * 128 : std::max<int64_t>(rows, 1);
}

// x parts | its rows' NaN flags | slabs
size_t dense_bytes(const QWeight& w, int64_t m, int64_t slab_rows) {
    return up256((size_t)3 * m * padded_k(w.k) * 2) + up256((size_t)m * 4) +
           (size_t)slab_rows * w.n * 4;
}

template <int QT, int BM>
hipError_t launch_gemm_bm(const QWeight& w, const float* x, int64_t m, float* y, int S, void* ws,
                          hipStream_t s, int add) {
    using D = DTile<QT, BM>;
    static const bool attr = hipFuncSetAttribute((const void*)dense_gemm_kernel<QT, BM>,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 D::BYTES) == hipSuccess;
    if (!attr) return hipErrorInvalidValue;
    const int64_t kp = padded_k(w.k), plane = m * kp;
    uint16_t* xp = static_cast<uint16_t*>(ws);
    uint32_t* nan_row =
        reinterpret_cast<uint32_t*>(static_cast<uint8_t*>(ws) + up256((size_t)3 * plane * 2));
    float* part = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(nan_row) + up256((size_t)m * 4));
    xsplit_kernel<<<(unsigned)m, 256, 0, s>>>(x, w.k, kp, xp, plane, nan_row);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int64_t tiles_n = (w.n + D::BN - 1) / D::BN;
    const int64_t tiles = (m + BM - 1) / BM * tiles_n;
    if (tiles * S > (int64_t)INT32_MAX - 8) return hipErrorInvalidValue;
    const int units_pad = (int)((tiles * S + 7) / 8 * 8);
    dense_gemm_kernel<QT, BM><<<units_pad, 512, D::BYTES, s>>>(
        w.base, w.row_bytes, xp, plane, kp, nan_row, x, w.k, y, m, w.n, (int)tiles_n, (int)tiles,
        units_pad, S, add, part);
    if ((e = hipGetLastError()) != hipSuccess || S == 1) return e;
    const int blocks =
        (int)std::min<int64_t>((m * w.n + 255) / 256, 8 * (int64_t)device_info().cu_count);
    dense_sum_kernel<QT><<<blocks, 256, 0, s>>>(part, S, m, w.n, w.base, w.row_bytes, nan_row, x,
                                                w.k, add, y);
    return hipGetLastError();
}

template <int QT>
hipError_t launch_dense_qt(const QWeight& w, const float* x, int64_t m, float* y, hipStream_t s,
                           int add) {
    if (dense_gemv_supports(w, m)) return launch_gemv_qt<QT>(w, x, m, y, s, add);
    if (w.k <= kShortK) {
        const dim3 grid((unsigned)((w.n + 255) / 256),
                        (unsigned)std::min<int64_t>((m + 63) / 64, 65535));
        dense_short_kernel<QT><<<grid, 256, 0, s>>>(w.base, w.row_bytes, x, m, w.n, (int)w.k, y,
                                                    add);
        return hipGetLastError();
    }
    const int64_t chunk = dense_chunk_rows(w);
    for (int64_t r = 0; r < m; r += chunk) {
        const int64_t rows = std::min(chunk, m - r);
        const DensePlan p = dense_plan(w, rows);
        void* ws = nullptr;
        hipError_t e =
            stream_workspace(s, dense_bytes(w, rows, p.S > 1 ? p.S * rows : 0), &ws, kDenseSlot);
        if (e != hipSuccess) return e;
        e = p.bm == 64
                ? launch_gemm_bm<QT, 64>(w, x + r * w.k, rows, y + r * w.n, p.S, ws, s, add)
                : launch_gemm_bm<QT, 128>(w, x + r * w.k, rows, y + r * w.n, p.S, ws, s, add);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

bool is_dense(int qtype) {
    return qtype == UNILLM_QTYPE_F32 || qtype == UNILLM_QTYPE_F16 || qtype == UNILLM_QTYPE_BF16;
}

int dense_elem_bytes(int qtype) { return qtype == UNILLM_QTYPE_F32 ? 4 : 2; }

int64_t dense_row_bytes(int qtype, int64_t k) { return padded_k(k) * dense_elem_bytes(qtype); }

hipError_t launch_dense_upload(const QWeight& w, const void* src, hipStream_t s) {
    if (w.k % kKPad == 0)
        return hipMemcpyAsync(w.base, src, (size_t)w.n * (size_t)w.row_bytes,
                              hipMemcpyDeviceToDevice, s);
    // (a launch holds at most 2^32 threads: 2^24 rows of 256)
    const unsigned blocks = (unsigned)std::min<int64_t>(w.n, (int64_t)1 << 20);
    if (w.qtype == UNILLM_QTYPE_F32)
        dense_upload_kernel<<<blocks, 256, 0, s>>>(static_cast<const uint32_t*>(src), w.base, w.n,
                                                   w.k, w.row_bytes);
    else
        dense_upload_kernel<<<blocks, 256, 0, s>>>(static_cast<const uint16_t*>(src), w.base, w.n,
                                                   w.k, w.row_bytes);
    return hipGetLastError();
}

hipError_t launch_dense_widen(const QWeight& w, float* out, hipStream_t s) {
    const int64_t count = w.n * w.k;
    const int blocks = (int)std::min<int64_t>((count + 255) / 256, 8 * device_info().cu_count);
    switch (w.qtype) {
        case UNILLM_QTYPE_F32:
            dense_widen_kernel<UNILLM_QTYPE_F32><<<blocks, 256, 0, s>>>(w.base, w.row_bytes, out,
                                                               w.n, w.k);
            break;
        case UNILLM_QTYPE_F16:
            dense_widen_kernel<UNILLM_QTYPE_F16><<<blocks, 256, 0, s>>>(w.base, w.row_bytes, out,
                                                               w.n, w.k);
            break;
        default:
            dense_widen_kernel<UNILLM_QTYPE_BF16><<<blocks, 256, 0, s>>>(w.base, w.row_bytes, out,
                                                               w.n, w.k);
    }
    return hipGetLastError();
}

hipError_t launch_norm_rows(const float* x, int64_t m, int64_t k, const NormArgs& norm,
                            float* out, hipStream_t s) {
    norm_rows_kernel<<<(unsigned)m, 256, 0, s>>>(x, k, norm, out);
    return hipGetLastError();
}

// A bound for every call of up to m rows: the GEMV takes none; slices x rows of a split
// are at most kDenseMaxSlices m, and at most 128 kDenseMaxRounds CUs / (column tiles).
size_t dense_workspace_bytes(const QWeight& w, int64_t m) {
    m = std::min(m, dense_chunk_rows(w));
    const int64_t tiles_n = (w.n + dense_bn(w) - 1) / dense_bn(w);
    const int64_t rows =
        padded_k(w.k) / kKPad < 8
            ? 0  // never split
            : std::min<int64_t>(kDenseMaxSlices * m,
                                128 * kDenseMaxRounds * (int64_t)device_info().cu_count / tiles_n);
    return dense_bytes(w, m, rows);
}

hipError_t launch_dense(const QWeight& w, const float* x, int64_t m, float* y, hipStream_t s,
                        int add) {
    switch (w.qtype) {
        case UNILLM_QTYPE_F32: return launch_dense_qt<UNILLM_QTYPE_F32>(w, x, m, y, s, add);
        case UNILLM_QTYPE_F16: return launch_dense_qt<UNILLM_QTYPE_F16>(w, x, m, y, s, add);
        case UNILLM_QTYPE_BF16: return launch_dense_qt<UNILLM_QTYPE_BF16>(w, x, m, y, s, add);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace unillm
