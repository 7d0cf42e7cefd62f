// layer_ops.hip -- the Llama layer's ops around attention (model.rs:269-356):
// embedding lookup, RMSNorm (alone or over the step's last rows), row gather,
// residual add, SwiGLU's silu(gate) * up, and greedy argmax.
//
// Numerics: the residual stream is f32 (as the reference's workspace);
// projections' inputs and outputs that feed a GEMM are bf16.  Every op
// computes in f32.  Reductions (RMSNorm's sum of squares, argmax) run as a
// tree over the 256 threads of a workgroup rather than the reference's
// 16-lane dot: the sum differs from the reference's in the last bits, the
// argmax result does not (ties resolve to the lowest index).
//
// Roofline: all HBM-bound.  Algorithmic bytes per row:
//   embed     2*hidden (table row) + 4*hidden (f32 out)
//   rmsnorm   4*hidden (x) + 2*hidden (out) (+ the weight, cache-resident)
//   gather    2 * row bytes (read, written)
//   add       4*cols (sum read) + 4*cols (written) + 2 or 4*cols (x)
//   silu_mul  2*2*cols (gate, up) + 2*cols (out)
//   argmax    4*cols (f32 logits) or 2*cols (bf16)
#include "vo_device.hpp"
#include "vo_kernels.hpp"

namespace vo {
namespace kernels {

namespace {

constexpr int kThreads = 256;
constexpr int kNormRegIt = 4;  // rmsnorm rows up to kThreads * 8 * 4 columns stay in registers

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Sum over the 256 threads of the workgroup; every thread gets the total.
__device__ __forceinline__ float block_sum(float v, float *lds4) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) lds4[wave] = v;
    __syncthreads();
    const float t = (lds4[0] + lds4[1]) + (lds4[2] + lds4[3]);
    return t;
}

// 8 bf16 (one 16-byte word) -> 8 f32.
__device__ __forceinline__ void unpack8(const u32x4 w, float *f) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[2 * k] = __uint_as_float(w[k] << 16);
        f[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
    }
}

__device__ __forceinline__ u32x4 pack8(const float *f) {
    u32x4 w;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        w[k] = static_cast<uint32_t>(f32_to_bf16_bits(f[2 * k])) |
               (static_cast<uint32_t>(f32_to_bf16_bits(f[2 * k + 1])) << 16);
    return w;
}

// Backend::embed (cpu/mod.rs:172-180): out[r] = table[tokens[r]], widened to
// f32 (exact).  One workgroup per row.  V8: 16-byte loads (hidden % 8 == 0).
template <bool V8>
__global__ __launch_bounds__(kThreads) void embed_kernel(const uint16_t *__restrict__ table,
                                                         uint32_t hidden,
                                                         const uint32_t *__restrict__ tokens,
                                                         float *__restrict__ out) {
    const uint32_t r = blockIdx.x;
    const uint16_t *src = table + static_cast<uint64_t>(tokens[r]) * hidden;
    float *dst = out + static_cast<uint64_t>(r) * hidden;
    if constexpr (V8) {
        for (uint32_t c = threadIdx.x * 8; c < hidden; c += kThreads * 8) {
            float f[8];
            unpack8(*reinterpret_cast<const u32x4 *>(src + c), f);
            *reinterpret_cast<floatx4 *>(dst + c) = floatx4{f[0], f[1], f[2], f[3]};
            *reinterpret_cast<floatx4 *>(dst + c + 4) = floatx4{f[4], f[5], f[6], f[7]};
        }
    } else {
        for (uint32_t c = threadIdx.x; c < hidden; c += kThreads) dst[c] = bf16_bits_to_f32(src[c]);
    }
}

// Backend::gather_rows (cpu/mod.rs:360-368): out row i = x row rows[i], a
// byte copy of row_words 4-byte words per row.  One workgroup per output
// row.  V4: 16-byte accesses (row_words % 4 == 0, both bases 16-byte aligned).
template <bool V4>
__global__ __launch_bounds__(kThreads) void gather_rows_kernel(const uint32_t *__restrict__ x,
                                                               uint32_t row_words,
                                                               const uint32_t *__restrict__ rows,
                                                               uint32_t *__restrict__ out) {
    const uint32_t i = blockIdx.x;
    const uint32_t *src = x + static_cast<uint64_t>(rows[i]) * row_words;
    uint32_t *dst = out + static_cast<uint64_t>(i) * row_words;
    if constexpr (V4) {
        for (uint32_t c = threadIdx.x * 4; c < row_words; c += kThreads * 4)
            *reinterpret_cast<u32x4 *>(dst + c) = *reinterpret_cast<const u32x4 *>(src + c);
    } else {
        for (uint32_t c = threadIdx.x; c < row_words; c += kThreads) dst[c] = src[c];
    }
}

// Backend::rmsnorm (cpu/mod.rs:182-197): out = w * (x * (1 / sqrt(mean(x^2)
// + eps))), the reference's (and HF's) order.  Row i of out normalises row
// rows_idx[i] of x (the LM head's gather_rows, model.rs:334-340), or row i
// when rows_idx is null.  One workgroup per output row; x is read once and
// held in registers for rows up to kThreads * 8 * kNormRegIt columns, longer
// rows are read twice, the second time from cache.
template <bool V8>
__global__ __launch_bounds__(kThreads) void rmsnorm_kernel(const float *__restrict__ x,
                                                           uint32_t hidden,
                                                           const uint16_t *__restrict__ w,
                                                           float eps,
                                                           const uint32_t *__restrict__ rows_idx,
                                                           uint16_t *__restrict__ out) {
    __shared__ float lds4[4];
    const uint32_t i = blockIdx.x;
    const uint32_t r = rows_idx ? rows_idx[i] : i;
    const float *src = x + static_cast<uint64_t>(r) * hidden;
    uint16_t *dst = out + static_cast<uint64_t>(i) * hidden;
    float ss = 0.0f;
    if constexpr (V8) {
        if (hidden <= kThreads * 8 * kNormRegIt) {
            // The row stays in registers between the two passes, and the
            // weights load before the reduction; a thread's sum adds the same
            // terms in the same order as the loop below.  Columns past the
            // row load its last 8 (not used), so the loads need no branch.
            floatx4 a[kNormRegIt], b[kNormRegIt];
            u32x4 wv[kNormRegIt];
#pragma unroll
            for (int it = 0; it < kNormRegIt; ++it) {
                const uint32_t c = min(threadIdx.x * 8 + it * kThreads * 8, hidden - 8);
                a[it] = *reinterpret_cast<const floatx4 *>(src + c);
                b[it] = *reinterpret_cast<const floatx4 *>(src + c + 4);
                wv[it] = *reinterpret_cast<const u32x4 *>(w + c);
            }
#pragma unroll
            for (int it = 0; it < kNormRegIt; ++it) {
                if (threadIdx.x * 8 + it * kThreads * 8 < hidden) {
                    ss += a[it][0] * a[it][0] + a[it][1] * a[it][1] + a[it][2] * a[it][2] + a[it][3] * a[it][3];
                    ss += b[it][0] * b[it][0] + b[it][1] * b[it][1] + b[it][2] * b[it][2] + b[it][3] * b[it][3];
                }
            }
            const float mean_square = block_sum(ss, lds4) / static_cast<float>(hidden);
            const float inv_rms = 1.0f / sqrtf(mean_square + eps);
#pragma unroll
            for (int it = 0; it < kNormRegIt; ++it) {
                const uint32_t c = threadIdx.x * 8 + it * kThreads * 8;
                if (c < hidden) {
                    float wf[8], o[8];
                    unpack8(wv[it], wf);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        o[k] = wf[k] * (a[it][k] * inv_rms);
                        o[4 + k] = wf[4 + k] * (b[it][k] * inv_rms);
                    }
                    *reinterpret_cast<u32x4 *>(dst + c) = pack8(o);
                }
            }
            return;
        }
        for (uint32_t c = threadIdx.x * 8; c < hidden; c += kThreads * 8) {
            const floatx4 a = *reinterpret_cast<const floatx4 *>(src + c);
            const floatx4 b = *reinterpret_cast<const floatx4 *>(src + c + 4);
            ss += a[0] * a[0] + a[1] * a[1] + a[2] * a[2] + a[3] * a[3];
            ss += b[0] * b[0] + b[1] * b[1] + b[2] * b[2] + b[3] * b[3];
        }
    } else {
        for (uint32_t c = threadIdx.x; c < hidden; c += kThreads) ss += src[c] * src[c];
    }
    const float mean_square = block_sum(ss, lds4) / static_cast<float>(hidden);
    const float inv_rms = 1.0f / sqrtf(mean_square + eps);
    if constexpr (V8) {
        for (uint32_t c = threadIdx.x * 8; c < hidden; c += kThreads * 8) {
            const floatx4 a = *reinterpret_cast<const floatx4 *>(src + c);
            const floatx4 b = *reinterpret_cast<const floatx4 *>(src + c + 4);
            float wf[8], o[8];
            unpack8(*reinterpret_cast<const u32x4 *>(w + c), wf);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                o[k] = wf[k] * (a[k] * inv_rms);
                o[4 + k] = wf[4 + k] * (b[k] * inv_rms);
            }
            *reinterpret_cast<u32x4 *>(dst + c) = pack8(o);
        }
    } else {
        for (uint32_t c = threadIdx.x; c < hidden; c += kThreads)
            dst[c] = f32_to_bf16_bits(bf16_bits_to_f32(w[c]) * (src[c] * inv_rms));
    }
}

// Backend::add (cpu/mod.rs:351-358): sum += x, x bf16 (widened) or f32.
template <bool XBF16>
__global__ __launch_bounds__(kThreads) void add_kernel(float *__restrict__ sum,
                                                       const void *__restrict__ x, uint64_t n) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kThreads;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride) {
        const float v = XBF16 ? bf16_bits_to_f32(static_cast<const uint16_t *>(x)[i])
                              : static_cast<const float *>(x)[i];
        sum[i] += v;
    }
}

__device__ __forceinline__ float silu_mul1(float g, float u) {
    // silu(g) = g * sigmoid(g) = g / (1 + e^-g); times up (cpu/mod.rs:341-349).
    // e^-g = 2^(-g log2 e) on the hardware exp2 and the quotient through the
    // hardware reciprocal (about an ulp each): the f32 value is within ~2^-20
    // of the correctly rounded one, far inside the bf16 rounding of the
    // output, and the kernel stays bound by HBM rather than by an exact
    // exp and divide per element.  Infinities and NaN come out as the exact
    // form's: g = -inf gives -inf * 0 = NaN, as -inf / inf does.
    constexpr float kLog2e = 1.44269504088896341f;
    const float e = __builtin_amdgcn_exp2f(-g * kLog2e);
    return g * __builtin_amdgcn_rcpf(1.0f + e) * u;
}

// Backend::silu_mul: out = silu(gate) * up, rows with their own strides;
// out may be gate itself (the reference's in-place form).  V8: 8 columns per
// thread with 16-byte accesses (cols and strides % 8 == 0).
template <bool V8>
__global__ __launch_bounds__(kThreads) void silu_mul_kernel(const uint16_t *gate, uint32_t gate_ld,
                                                            const uint16_t *up, uint32_t up_ld,
                                                            uint32_t rows, uint32_t cols,
                                                            uint16_t *out, uint32_t out_ld) {
    constexpr uint32_t V = V8 ? 8 : 1;
    const uint32_t per_row = cols / V;
    const uint64_t n = static_cast<uint64_t>(rows) * per_row;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * kThreads;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x; i < n; i += stride) {
        const uint32_t r = static_cast<uint32_t>(i / per_row);
        const uint32_t c = static_cast<uint32_t>(i % per_row) * V;
        const uint16_t *gp = gate + static_cast<uint64_t>(r) * gate_ld + c;
        const uint16_t *upp = up + static_cast<uint64_t>(r) * up_ld + c;
        uint16_t *op = out + static_cast<uint64_t>(r) * out_ld + c;
        if constexpr (V8) {
            float g[8], u[8], o[8];
            unpack8(*reinterpret_cast<const u32x4 *>(gp), g);
            unpack8(*reinterpret_cast<const u32x4 *>(upp), u);
#pragma unroll
            for (int k = 0; k < 8; ++k) o[k] = silu_mul1(g[k], u[k]);
            *reinterpret_cast<u32x4 *>(op) = pack8(o);
        } else {
            *op = f32_to_bf16_bits(silu_mul1(bf16_bits_to_f32(*gp), bf16_bits_to_f32(*upp)));
        }
    }
}

// (value, index) of a running maximum; index 0xffffffff = no element yet.
struct ArgBest {
    float v;
    uint32_t i;
};

// `o` beats `b`: larger, or equal at a lower index -- the first maximum
// wins (cpu/mod.rs:370-388; torch's rule).
__device__ __forceinline__ bool beats(const ArgBest &o, const ArgBest &b) {
    return o.v > b.v || (o.v == b.v && o.i < b.i);
}

__device__ __forceinline__ float load_logit(const void *p, uint64_t k, bool f32) {
    return f32 ? static_cast<const float *>(p)[k]
               : bf16_bits_to_f32(static_cast<const uint16_t *>(p)[k]);
}

// Backend::argmax: ids[r] = first index of row r's maximum, or 0xffffffff
// when the row holds a NaN (EngineError::NaN, reported by the host).  One
// workgroup of T threads per row; a thread reads VPL values at a time (16
// bytes: f32 with V = 4, bf16 with V = 8; V = 1 where the row is no whole
// number of such words), U of them before it looks at the first, and keeps
// the first maximum of its own columns, which it sees in increasing order
// (strict '>'); the (value, index) pairs then merge by `beats`.
//
// Bound: how much one CU keeps in flight, since a greedy step has few rows
// and each is one workgroup's (a second level over several workgroups would
// need a workspace, which the op's callers do not give).  With 256 threads
// and one load in flight a 128256-column f32 row took 42 us (12 GB/s) and 40
// rows 60 us; with 1024 threads and eight loads each (128 KiB in flight) 9 us
// for 1 to 40 rows, 23 us for 256 (131 MB, 5.8 TB/s).
template <bool F32, int V, int T>
__global__ __launch_bounds__(T) void argmax_kernel(const void *__restrict__ logits, uint32_t cols,
                                                   uint32_t *__restrict__ ids) {
    constexpr int U = V == 1 ? 4 : 8;
    constexpr int W = T / 64;
    __shared__ float lds_v[W];
    __shared__ uint32_t lds_i[W];
    __shared__ int lds_nan[W];
    const uint32_t r = blockIdx.x;
    const uint64_t base = static_cast<uint64_t>(r) * cols;
    ArgBest b{-__builtin_inff(), 0xffffffffu};
    bool nan = false;
    auto take = [&](float v, uint32_t c) {
        nan |= v != v;
        if (b.i == 0xffffffffu || v > b.v) b = ArgBest{v, c};
    };
    // The values at word q of the row (V columns from V q on).
    auto words = [&](const u32x4 &w, uint32_t q) {
        if constexpr (F32) {
#pragma unroll
            for (int k = 0; k < 4; ++k) take(__uint_as_float(w[k]), 4 * q + k);
        } else {
            float f[8];
            unpack8(w, f);
#pragma unroll
            for (int k = 0; k < 8; ++k) take(f[k], 8 * q + k);
        }
    };
    const uint32_t n = cols / V;  // words of the row
    const uint32_t passes = n / (U * T) + (n % (U * T) != 0);
    for (uint32_t p = 0; p < passes; ++p) {
        // Words past the row load its last one and are not looked at.
        const uint32_t q0 = p * (U * T) + threadIdx.x;
        if constexpr (V > 1) {
            const u32x4 *row = reinterpret_cast<const u32x4 *>(
                static_cast<const uint8_t *>(logits) + base * (F32 ? 4 : 2));
            u32x4 w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) w[u] = row[min(q0 + u * T, n - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (q0 + u * T < n) words(w[u], q0 + u * T);
        } else {
            float w[U];
#pragma unroll
            for (int u = 0; u < U; ++u) w[u] = load_logit(logits, base + min(q0 + u * T, n - 1), F32);
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (q0 + u * T < n) take(w[u], q0 + u * T);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const ArgBest x{__shfl_xor(b.v, o, 64), static_cast<uint32_t>(__shfl_xor(static_cast<int>(b.i), o, 64))};
        if (beats(x, b)) b = x;
    }
    const int any_nan = __any(nan) ? 1 : 0;
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        lds_v[wave] = b.v;
        lds_i[wave] = b.i;
        lds_nan[wave] = any_nan;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        ArgBest t{lds_v[0], lds_i[0]};
        int any = lds_nan[0];
#pragma unroll
        for (int k = 1; k < W; ++k) {
            const ArgBest x{lds_v[k], lds_i[k]};
            if (beats(x, t)) t = x;
            any |= lds_nan[k];
        }
        ids[r] = any ? 0xffffffffu : t.i;
    }
}

// Backend::matmul for shapes the library GEMM does not take (rows of x or
// of the weight not a whole number of 16-byte words): out[r][o] = sum_k
// x[r][k] * w[o][k] in f32, k ascending, then out = acc (+ out when
// accumulating), stored as f32 or bf16.  One thread per output element;
// meant for the reference's tiny test shapes, not for throughput.
template <bool OUT_F32>
__global__ __launch_bounds__(kThreads) void matmul_generic_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, uint32_t rows, uint32_t n,
    uint32_t k, void *__restrict__ out, bool accumulate) {
    const uint64_t idx = static_cast<uint64_t>(blockIdx.x) * kThreads + threadIdx.x;
    if (idx >= static_cast<uint64_t>(rows) * n) return;
    const uint32_t r = static_cast<uint32_t>(idx / n), o = static_cast<uint32_t>(idx % n);
    const uint16_t *xr = x + static_cast<uint64_t>(r) * k;
    const uint16_t *wr = w + static_cast<uint64_t>(o) * k;
    float acc = 0.0f;
    for (uint32_t j = 0; j < k; ++j) acc += bf16_bits_to_f32(xr[j]) * bf16_bits_to_f32(wr[j]);
    if constexpr (OUT_F32) {
        float *d = static_cast<float *>(out) + idx;
        *d = accumulate ? *d + acc : acc;
    } else {
        uint16_t *d = static_cast<uint16_t *>(out) + idx;
        *d = f32_to_bf16_bits(accumulate ? bf16_bits_to_f32(*d) + acc : acc);
    }
}

// Four consecutive outputs of one row.  MODE 0: bf16, 1: f32, 2: f32 +=.
template <int MODE>
__device__ __forceinline__ void store_out4(void *out, uint64_t o, floatx4 t) {
    if constexpr (MODE == 0) {
        u32x2 p;
        p[0] = static_cast<uint32_t>(f32_to_bf16_bits(t[0])) |
               (static_cast<uint32_t>(f32_to_bf16_bits(t[1])) << 16);
        p[1] = static_cast<uint32_t>(f32_to_bf16_bits(t[2])) |
               (static_cast<uint32_t>(f32_to_bf16_bits(t[3])) << 16);
        *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(out) + o) = p;
    } else {
        floatx4 *d = reinterpret_cast<floatx4 *>(static_cast<float *>(out) + o);
        if constexpr (MODE == 2) t += *d;
        *d = t;
    }
}

// SwiGLU of four gate and up sums, rounded to bf16 first as their own outputs
// would be.
__device__ __forceinline__ floatx4 swiglu4(floatx4 g, floatx4 u) {
    floatx4 t;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        t[e] = silu_mul1(bf16_bits_to_f32(f32_to_bf16_bits(g[e])),
                         bf16_bits_to_f32(f32_to_bf16_bits(u[e])));
    return t;
}

// Backend::matmul for few rows (skinny_kernel has which): streaming the weight
// is the whole cost.  A workgroup owns 16 / P weight rows
// (outputs) and splits K over its 8 wavefronts and, within one, over P parts;
// each wavefront runs v_mfma_f32_16x16x32_bf16 with A = P blocks of 16 / P
// weight rows, block p from part p of its columns, and B = x^T laid out alike
// (the batch rows in columns 0..rows-1 of each block; columns past the batch
// repeat its last row and are not stored, so no lane branches), so that the P
// diagonal blocks of D hold the parts' sums and the rest is not looked at.
// U steps of loads are issued before their MFMAs.  The partial sums are added
// through LDS in order of wavefront and part, so an output depends only on its
// own row of x, whatever the batch size.  Ordinary loads: a step reads 64
// bytes of each weight row, half a cache line, and the next step the other
// half; non-temporal loads measured 10-15% slower (the line is fetched twice).
//
// P = 1 (up to 4 rows), 8 steps of loads in flight: here, in the order of one
// launch and one round of loads, it beats stream_gemm_kernel below (a weight
// of 3072 x 2048, 4 rows: 5.1 against 5.8 us; 4096 x 4096: 8.7 against 9.4);
// on larger weights of up to 4096 columns, or with more rows, every workgroup's
// reads of x from L2 make it the slower one.
// P = 2 (up to 8 rows): weights of at most 2048 rows, whose 128 tiles of 16
// leave half the 256 CUs idle: a weight of 2048 x 8192, 4 rows, took 13.4 us
// with P = 1 and takes 9.1 (3.7 TB/s); 2048 x 2048 4.9 and 4.0.  P = 4 adds
// nothing (10.2, 4.6), and 2 steps in flight do as well as 4 to 16 (9.2-9.5).
// From 3072 rows on P = 1 is the better one (5.0 against 5.3).
constexpr int kSkinnyWaves = 8;
constexpr uint64_t kSkinnyWeight = 1ull << 24;  // largest small weight
constexpr uint32_t kSkinnyHalfN = 2048;         // largest weight rows of P = 2

template <int MODE, int P, int U>
__global__ __launch_bounds__(64 * kSkinnyWaves) void skinny_gemm_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, uint32_t rows, uint32_t n,
    uint32_t k, void *__restrict__ out) {
    static_assert(P == 1 || P == 2, "blocks of the diagonal");
    constexpr uint32_t R = 16 / P;  // weight rows of the workgroup, largest batch
    __shared__ floatx4 part[kSkinnyWaves][64];
    const uint32_t n0 = blockIdx.x * R;
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t kw = k / (kSkinnyWaves * P);  // of one part; a multiple of 32 * U
    const uint32_t r = lane % R, kg = lane >> 4;
    const uint32_t k0 = (wave * P + (lane & 15) / R) * kw + 8 * kg;
    const uint16_t *wp = w + static_cast<uint64_t>(n0 + r) * k + k0;
    const uint16_t *xp = x + static_cast<uint64_t>(min(r, rows - 1)) * k + k0;
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t kk = 0; kk < kw; kk += 32 * U) {
        u32x4 a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            a[u] = *reinterpret_cast<const u32x4 *>(wp + kk + 32 * u);
            b[u] = *reinterpret_cast<const u32x4 *>(xp + kk + 32 * u);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u]),
                                                          __builtin_bit_cast(bf16x8, b[u]), acc,
                                                          0, 0, 0);
    }
    part[wave][lane] = acc;
    __syncthreads();
    // Lane l of D holds rows 4 (l / 16) + e, e = 0..3, of column l % 16: block
    // p's output 4 kg + e of batch row r is in lane 16 kg + r + 40 p (P = 2).
    if (wave != 0 || (lane & 15) >= R || kg >= 4 / P) return;
    floatx4 t = part[0][lane];
#pragma unroll
    for (int v = 1; v < kSkinnyWaves * P; ++v) t += part[v / P][lane + 40 * (v % P)];
    if (r < rows) store_out4<MODE>(out, static_cast<uint64_t>(r) * n + n0 + 4 * kg, t);
}

// Backend::matmul for up to 64 rows: HBM, the weight read once.  MT = tiles
// of 16 batch rows.  A workgroup owns NW tiles of 16 weight rows, one to a
// wavefront, and splits K over KG groups of NW wavefronts.  A wavefront
// loads its 16 x KC piece of the weight straight into registers, one chunk
// ahead of the MFMAs (KC / 32 loads of 16 bytes per lane in flight while it
// computes), and each group stages the KC columns of x that its wavefronts
// all need in LDS by LDS DMA, through a ring of three stages, two chunks
// ahead: read from L2 once per NW weight tiles and not once per tile, since
// with x loaded by every wavefront the kernel slows in proportion to the
// batch (a 28672 x 4096 weight: 40 us for 1 row, 63 for 16).  The KG partial
// tiles of an output are summed through LDS in group order.
//
// LDS: row r's 16-byte unit c sits at unit c ^ (r % 16) (mod the row's
// units), so the 16 lanes that read one unit of 16 rows hit 16 different
// 4-bank groups; the DMA, whose lanes write in order, applies the same map to
// its sources.
//
// Workgroup b starts its walk over K at chunk b mod (chunks), so that the
// workgroups do not all read the same lines of x, or the same columns of
// their weight rows, at once.  The order in which an output's products are
// added depends on the weight's shape, the output's column and which instance
// runs (launch_stream_rows), so on the number of rows, not on what the
// other rows hold.  Weight loads
// are ordinary ones (see skinny_gemm_kernel).
//
// MODE 3 is the gate and up projections with SwiGLU: the weight is [gate; up],
// the even wavefronts of a workgroup own tiles of the gate half and the odd
// ones the same tiles of the up half, whose sums (each rounded to bf16, as the
// two steps' intermediate is) meet through LDS: one launch and 4 bytes per
// value of traffic less.  16384 x 2048, 4 rows: 13.8 + 4.0 us as two launches,
// 15.1 as one.
//
// Measured, rows 16 / 40 / 64, against the library product it stands in for:
// 28672 x 4096: 42.6 / 49.1 / 47.7 us, library 59.6 / 51.1 / 52.2 (5.5 TB/s
// at 16 rows); 128256 x 2048: 94.8 / 99.9 / 110 us, library 117 / 124 / 130;
// 6144 x 4096: 13.3 / 16.4 us, library 14.1 / 16.8 (64 rows 18.7 and 17.3: the
// library's, see skinny_kernel).
template <int MODE, int MT, int NW, int KG, int KC>
__global__ __launch_bounds__(64 * NW * KG) void stream_gemm_kernel(
    const uint16_t *__restrict__ x, const uint16_t *__restrict__ w, uint32_t rows, uint32_t n,
    uint32_t k, void *__restrict__ out) {
    constexpr int W = NW * KG;
    constexpr int U = KC / 32;              // weight loads per chunk
    constexpr uint32_t UPR = KC / 8;        // 16-byte units of a staged row
    constexpr uint32_t SWZ = UPR < 16 ? UPR - 1 : 15;
    constexpr int XI = 16 * MT * UPR / 64;  // DMA instructions per chunk and group
    constexpr int ND = XI / NW;
    constexpr uint32_t XB = 16 * MT * KC * 2;  // bytes of a group's stage
    static_assert(XI % NW == 0 && ND + U <= 63, "chunk DMA split");
    constexpr bool GLU = MODE == 3;
    static_assert(KG == 1 || W * MT * 64 * 16 <= XB * KG, "the partial tiles fit a stage");
    static_assert(!GLU || (NW % 2 == 0 && W * MT * 64 * 8 <= XB * KG), "gate and up tiles");
    __shared__ __align__(1024) uint8_t st0[XB * KG];
    __shared__ __align__(1024) uint8_t st1[XB * KG];
    __shared__ __align__(1024) uint8_t st2[XB * KG];

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nw = wave % NW, grp = wave / NW;
    const uint32_t r = lane & 15, kg = lane >> 4;
    // A tile past the last one (n is a multiple of 16, not of 16 NW) reads
    // the last one and stores nothing.
    const uint32_t half = GLU ? n / 2 : n;  // outputs
    const uint32_t n0 = (GLU ? blockIdx.x * (NW / 2) + nw / 2 : blockIdx.x * NW + nw) * 16;
    const uint32_t nr = min(n0, half - 16) + (GLU ? nw % 2 * half : 0);
    const uint32_t kslice = k / KG, k0 = grp * kslice, nch = kslice / KC;
    const uint32_t rot = blockIdx.x % nch;
    auto chunk_at = [&](uint32_t c) {  // c < nch
        c += rot;
        return c >= nch ? c - nch : c;
    };
    const uint16_t *wp = w + static_cast<uint64_t>(nr + r) * k + k0 + 8 * kg;
    const auto x_rsrc = buffer_rsrc(x, rows * k * 2);
    uint32_t x_off[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const uint32_t u = (i * NW + nw) * 64 + lane;
        const uint32_t row = u / UPR, c = (u % UPR) ^ (row & SWZ);
        x_off[i] = (min(row, rows - 1) * k + k0 + 8 * c) * 2;
    }
    auto dma = [&](uint8_t *st, uint32_t c) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ND; ++i)
            dma16_at(x_rsrc, st + grp * XB + (i * NW + nw) * 1024, x_off[i], chunk_at(c) * (KC * 2));
    };
    auto load_w = [&](u32x4 (&a)[U], uint32_t c) __attribute__((always_inline)) {
        const uint16_t *p = wp + static_cast<uint64_t>(chunk_at(c)) * KC;
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = *reinterpret_cast<const u32x4 *>(p + 32 * u);
        __builtin_amdgcn_sched_barrier(0);
    };
    floatx4 acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
    // Chunk c: issue the weight loads of chunk c + 1, wait for chunk c's
    // (older, as is this wavefront's share of its x), meet the other
    // wavefronts, refill the stage they read last with x of chunk c + 2.
    // Every step issues its loads (past the last chunk the last one's), so
    // that the wait count stays uniform.
    auto step = [&](u32x4 (&a)[U], u32x4 (&an)[U], const uint8_t *__restrict__ cur,
                    uint8_t *__restrict__ nxt, uint32_t c) __attribute__((always_inline)) {
        load_w(an, min(c + 1, nch - 1));
        wait_barrier<ND + U>();
        dma(nxt, min(c + 2, nch - 1));
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const uint32_t row = 16 * m + r;
                const bf16x8 b = *reinterpret_cast<const bf16x8 *>(
                    cur + grp * XB + (row * UPR + ((4 * u + kg) ^ (row & SWZ))) * 16);
                acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u]),
                                                                 b, acc[m], 0, 0, 0);
            }
    };
    u32x4 a0[U], a1[U];
    dma(st0, 0);
    load_w(a0, 0);
    dma(st1, min(1u, nch - 1));
    for (uint32_t c = 0;;) {
        step(a0, a1, st0, st2, c);
        if (++c >= nch) break;
        step(a1, a0, st1, st0, c);
        if (++c >= nch) break;
        step(a0, a1, st2, st1, c);
        if (++c >= nch) break;
        step(a1, a0, st0, st2, c);
        if (++c >= nch) break;
        step(a0, a1, st1, st0, c);
        if (++c >= nch) break;
        step(a1, a0, st2, st1, c);
        if (++c >= nch) break;
    }
    // The DMA past the last chunk must land before the stages are reused or
    // the workgroup's LDS is released.
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));

    // Lane l holds outputs n0 + 4 (l / 16) + e, e = 0..3, of batch row 16 m +
    // l % 16.
    if constexpr (KG == 1 && !GLU) {
        if (n0 >= n) return;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint32_t row = 16 * m + r;
            if (row < rows)
                store_out4<MODE>(out, static_cast<uint64_t>(row) * n + n0 + 4 * kg, acc[m]);
        }
    } else if constexpr (KG == 1) {
        __syncthreads();
        floatx4 *up = reinterpret_cast<floatx4 *>(st0);  // [NW / 2][MT][64]
        if (nw % 2) {
#pragma unroll
            for (int m = 0; m < MT; ++m) up[(nw / 2 * MT + m) * 64 + lane] = acc[m];
        }
        __syncthreads();
        if (nw % 2 || n0 >= half) return;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const uint32_t row = 16 * m + r;
            if (row < rows)
                store_out4<0>(out, static_cast<uint64_t>(row) * half + n0 + 4 * kg,
                              swiglu4(acc[m], up[(nw / 2 * MT + m) * 64 + lane]));
        }
    } else {
        __syncthreads();
        floatx4 *part = reinterpret_cast<floatx4 *>(st0);  // [W][MT][64]
#pragma unroll
        for (int m = 0; m < MT; ++m) part[(wave * MT + m) * 64 + lane] = acc[m];
        __syncthreads();
        constexpr uint32_t NT = GLU ? NW / 2 : NW;
        auto total = [&](uint32_t tn, uint32_t m) __attribute__((always_inline)) {
            floatx4 sum = part[(tn * MT + m) * 64 + lane];
#pragma unroll
            for (int g = 1; g < KG; ++g) sum += part[((g * NW + tn) * MT + m) * 64 + lane];
            return sum;
        };
        for (uint32_t t = wave; t < NT * MT; t += W) {
            const uint32_t tn = t % NT, m = t / NT;
            const uint32_t row = 16 * m + r, nt = (blockIdx.x * NT + tn) * 16;
            const uint64_t o = static_cast<uint64_t>(row) * half + nt + 4 * kg;
            if (row >= rows || nt >= half) continue;
            if constexpr (GLU) store_out4<0>(out, o, swiglu4(total(2 * tn, m), total(2 * tn + 1, m)));
            else store_out4<MODE>(out, o, total(tn, m));
        }
    }
}

// RMSNorm, then stream_gemm_kernel's product (MODE 0, or 3 with SwiGLU) for the
// few rows of a decode step, whose RMSNorm alone is a launch of 3 us and a gap.
// Every workgroup normalises the rows again, one to a wavefront, while its
// first weight chunk is on its way: 8 loads of 16 bytes per lane and row, out
// of L2 since all workgroups read the same, a reduction within the wavefront,
// and the row in bf16 to LDS, where it stays: no DMA and no barrier in the
// loop over K.  The 16-byte units of a row are swizzled as above.
//
// Rows 1 / 4 / 8 / 16, launched back to back, against RMSNorm and the product:
// 3072 x 2048: 5.7 / 5.9 / 7.1 / 8.7 us, two launches 7.2 / 7.8 / 8.5 / 8.7;
// 4096 x 2048 with SwiGLU: 9.6 / 9.4 / 10.7 / 10.9, 10.9 / 10.8 / 10.8 / 10.9;
// 16384 x 2048 with SwiGLU: 16.6 / 16.8 / 17.2 / 17.0, 17.3 / 17.3 / 16.8 / 17.1
// (a second group of wavefronts per workgroup there: no faster).
//
// MODE 4 is the QKV projection with RoPE and the cache write (QkvRope): a
// tile's 16 weight rows are 8 of a head's first half and the 8 that they are
// rotated with, so that lane l's four sums and their partners in lane l ^ 32
// meet without LDS; each is rounded to bf16 first, as the product's own output
// would be.  No other reader of the product is left, so it is not written.  A
// 16-layer decode step of 4 sequences: 1043 us with RoPE as a launch of its
// own, 953 so.
constexpr uint32_t kNormGemmK = 2048;  // largest k
constexpr uint32_t kNormGemmRows = 8;  // largest batch

template <int MODE, int NW, int KG>
__global__ __launch_bounds__(64 * NW * KG) void norm_gemm_kernel(
    const float *__restrict__ x, const uint16_t *__restrict__ norm, float eps,
    const uint16_t *__restrict__ w, uint32_t rows, uint32_t n, uint32_t k,
    uint16_t *__restrict__ out, QkvRope to) {
    constexpr int W = NW * KG;
    constexpr int U = 8;
    constexpr uint32_t KC = 32 * U;
    constexpr int KJ = kNormGemmK / 512;
    constexpr bool GLU = MODE == 3;
    constexpr bool ROPE = MODE == 4;
    static_assert(!GLU || NW % 2 == 0, "gate and up tiles");
    __shared__ __align__(1024) uint8_t xs[2 * kNormGemmRows * kNormGemmK];
    __shared__ floatx4 part[W][64];

    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nw = wave % NW, grp = wave / NW;
    const uint32_t r = lane & 15, kg = lane >> 4;
    const uint32_t half = GLU ? n / 2 : n;  // outputs
    const uint32_t n0 = (GLU ? blockIdx.x * (NW / 2) + nw / 2 : blockIdx.x * NW + nw) * 16;
    const uint32_t nr = min(n0, half - 16) + (GLU ? nw % 2 * half : 0);
    const uint32_t kslice = k / KG, k0 = grp * kslice, nch = kslice / KC;
    const uint32_t upr = k / 8;  // 16-byte units of a row
    const uint32_t rot = blockIdx.x % nch;
    auto chunk_at = [&](uint32_t c) {  // c < nch
        c += rot;
        return c >= nch ? c - nch : c;
    };
    // The tile's place in its head (MODE 4): pairs 8 j .. 8 j + 7 of `head`.
    const uint32_t hd = ROPE ? to.head_dim : 16;
    const uint32_t wr = ROPE ? nr / hd * hd + nr % hd / 2 + (r & 7) + (r >> 3) * (hd / 2) : nr + r;
    const uint16_t *wp = w + static_cast<uint64_t>(wr) * k + k0 + 8 * kg;
    auto load_w = [&](u32x4 (&a)[U], uint32_t c) __attribute__((always_inline)) {
        const uint16_t *p = wp + chunk_at(c) * KC;
#pragma unroll
        for (int u = 0; u < U; ++u) a[u] = *reinterpret_cast<const u32x4 *>(p + 32 * u);
        __builtin_amdgcn_sched_barrier(0);
    };
    // A lane's columns of a row: 8 from 512 j + 8 lane on (k % 512 == 0; past k
    // the row's last 8, not used).
    floatx4 v[2 * KJ];
    u32x4 g[KJ];
    uint32_t pos = 0, slot = 0;
    if constexpr (ROPE) {
        pos = to.positions[min(r, rows - 1)];
        slot = to.slots[min(r, rows - 1)];
    }
    const float *xr = x + static_cast<uint64_t>(min(wave, rows - 1)) * k;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
        const uint32_t c = min(512 * j + 8 * lane, k - 8);
        v[2 * j] = *reinterpret_cast<const floatx4 *>(xr + c);
        v[2 * j + 1] = *reinterpret_cast<const floatx4 *>(xr + c + 4);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < KJ; ++j)
        g[j] = *reinterpret_cast<const u32x4 *>(norm + min(512 * j + 8 * lane, k - 8));
    __builtin_amdgcn_sched_barrier(0);
    u32x4 a0[U], a1[U];
    load_w(a0, 0);
    if (wave < rows) {  // a wavefront for each row (norm_gemm_supported)
        float ss = 0.0f;
#pragma unroll
        for (int j = 0; j < KJ; ++j)
            if (512 * j < k) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    ss += v[2 * j][e] * v[2 * j][e] + v[2 * j + 1][e] * v[2 * j + 1][e];
            }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, 64);
        const float inv_rms = 1.0f / sqrtf(ss / static_cast<float>(k) + eps);
#pragma unroll
        for (int j = 0; j < KJ; ++j)
            if (512 * j < k) {
                float wf[8], o[8];
                unpack8(g[j], wf);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = wf[e] * (v[2 * j][e] * inv_rms);
                    o[4 + e] = wf[4 + e] * (v[2 * j + 1][e] * inv_rms);
                }
                *reinterpret_cast<u32x4 *>(xs + (wave * upr + ((64 * j + lane) ^ (wave & 15))) * 16) =
                    pack8(o);
            }
    }
    __syncthreads();

    // Lane l's four pairs (MODE 4), under way while K is walked.
    floatx4 rc = {0.f, 0.f, 0.f, 0.f}, rs = rc;
    if constexpr (ROPE) {
        const uint64_t at = static_cast<uint64_t>(pos) * (hd / 2) + nr % hd / 2 + 4 * (kg & 1);
        rc = *reinterpret_cast<const floatx4 *>(to.cos_tab + at);
        rs = *reinterpret_cast<const floatx4 *>(to.sin_tab + at);
    }

    // Columns past the batch repeat its last row and are not stored.
    const uint32_t xrow = min(r, rows - 1);
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
    auto step = [&](u32x4 (&a)[U], u32x4 (&an)[U], uint32_t c) __attribute__((always_inline)) {
        load_w(an, min(c + 1, nch - 1));
        const uint32_t u0 = (k0 + chunk_at(c) * KC) / 8 + kg;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const bf16x8 b = *reinterpret_cast<const bf16x8 *>(
                xs + (xrow * upr + ((u0 + 4 * u) ^ (xrow & 15))) * 16);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[u]), b, acc,
                                                          0, 0, 0);
        }
    };
    for (uint32_t c = 0;;) {
        step(a0, a1, c);
        if (++c >= nch) break;
        step(a1, a0, c);
        if (++c >= nch) break;
    }

    // Lane l holds outputs n0 + 4 (l / 16) + e, e = 0..3, of batch row l % 16.
    part[wave][lane] = acc;
    __syncthreads();
    constexpr uint32_t NT = GLU ? NW / 2 : NW;
    if (wave >= NT) return;
    auto total = [&](uint32_t t) __attribute__((always_inline)) {
        floatx4 sum = part[t][lane];
#pragma unroll
        for (int q = 1; q < KG; ++q) sum += part[q * NW + t][lane];
        return sum;
    };
    const uint32_t nt = (blockIdx.x * NT + wave) * 16;
    if constexpr (ROPE) {
        if (nt >= half) return;
        floatx4 y = total(wave);
        const uint32_t kvd = to.kv_heads * hd;
        if (nt < to.q_cols + kvd) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float own = bf16_bits_to_f32(f32_to_bf16_bits(y[e]));
                const float other = __shfl_xor(own, 32, 64);
                y[e] = kg < 2 ? rot_first(own, other, rc[e], rs[e])
                              : rot_second(other, own, rc[e], rs[e]);
            }
        }
        if (r >= rows) return;
        const uint32_t d = nt % hd / 2 + 4 * (kg & 1) + (kg >> 1) * (hd / 2);
        if (nt < to.q_cols) {
            store_out4<0>(to.q_out, static_cast<uint64_t>(r) * to.q_cols + nt / hd * hd + d, y);
            return;
        }
        if (slot == kSkipSlot) return;
        const uint32_t kvh = (nt - to.q_cols) / hd % to.kv_heads;
        const uint64_t tile = (static_cast<uint64_t>(slot / 16) * to.kv_heads + kvh) * (16 * hd);
        if (nt < to.q_cols + kvd) {
            store_out4<0>(to.k_pool, tile + d / 32 * 512 + slot % 16 * 32 + d % 32, y);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                to.v_pool[tile + (d + e) * 16 + slot % 16] = f32_to_bf16_bits(y[e]);
        }
        return;
    }
    if (r >= rows || nt >= half) return;
    const uint64_t o = static_cast<uint64_t>(r) * half + nt + 4 * kg;
    if constexpr (GLU) store_out4<0>(out, o, swiglu4(total(2 * wave), total(2 * wave + 1)));
    else store_out4<0>(out, o, total(wave));
}

template <int MT, int NW, int KG, int KC>
void launch_stream(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t n, uint32_t k,
                   void *out, int mode, hipStream_t stream) {
    const dim3 grid((n + 16 * NW - 1) / (16 * NW)), block(64 * NW * KG);
#define VO_STREAM(MODE)                                                                        \
    hipLaunchKernelGGL((stream_gemm_kernel<MODE, MT, NW, KG, KC>), grid, block, 0, stream, x, \
                       w, rows, n, k, out)
    if (mode == 0) VO_STREAM(0);
    else if (mode == 1) VO_STREAM(1);
    else if (mode == 2) VO_STREAM(2);
    else if constexpr (NW % 2 == 0) VO_STREAM(3);
#undef VO_STREAM
}

// The workgroup's shape, by how many 16-row weight tiles there are.  While
// they last, a workgroup to each of the 256 CUs and no second round: 1 tile and
// 8 groups up to 4096 weight rows, 2 tiles and 4 groups up to 8192 (16 rows of
// x, 4608 x 4096: 13.0 us, with 1 tile 15.2; 8192 x 8192: 31.4, with 4 tiles
// 38.6; 10240 x 8192: 47.2, with 4 tiles 41.0).  Past that 4 tiles with
// 256-column chunks (each shares x once more); 8 for a vocabulary's worth of
// rows and more than one batch tile (99.9 against 114 us at 128256 x 2048, 40
// rows; 348 against 392 at 128256 x 8192, 32 rows; but weight rows of 8 KiB
// want 4: 128256 x 4096, 17 rows 227 with 8 and 183 with 4, 3584 and 4608
// columns not) and for 4 batch tiles from 24576 on (47.7 against 55.2 us at
// 28672 x 4096).  3 and 4 batch tiles, whose stages would not fit 8 groups,
// and tiles in pairs run 2 and 4 below 4096 too.
template <int MT>
void launch_stream_rows(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t n,
                        uint32_t k, void *out, int mode, hipStream_t stream) {
    if (n > 8192) {
        if constexpr (MT > 1)
            if (n >= 65536 && k != 4096) return launch_stream<MT, 8, 1, 256>(x, w, rows, n, k, out, mode, stream);
        if constexpr (MT == 4)
            if (n >= 24576) return launch_stream<MT, 8, 1, 128>(x, w, rows, n, k, out, mode, stream);
        return launch_stream<MT, 4, 1, 256>(x, w, rows, n, k, out, mode, stream);
    }
    if constexpr (MT <= 2) {
        if (n > 4096) return launch_stream<MT, 2, 4, 128>(x, w, rows, n, k, out, mode, stream);
        if (mode != 3) return launch_stream<MT, 1, 8, 64>(x, w, rows, n, k, out, mode, stream);
    }
    return launch_stream<MT, 2, 4, 64>(x, w, rows, n, k, out, mode, stream);
}

hipError_t launch_stream_any(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t n,
                             uint32_t k, void *out, int mode, hipStream_t stream) {
    switch ((rows + 15) / 16) {
        case 1: launch_stream_rows<1>(x, w, rows, n, k, out, mode, stream); break;
        case 2: launch_stream_rows<2>(x, w, rows, n, k, out, mode, stream); break;
        case 3: launch_stream_rows<3>(x, w, rows, n, k, out, mode, stream); break;
        default: launch_stream_rows<4>(x, w, rows, n, k, out, mode, stream); break;
    }
    return hipGetLastError();
}

uint32_t grid_for(uint64_t items) {
    const uint64_t g = (items + kThreads - 1) / kThreads;
    return static_cast<uint32_t>(g < 65536 ? (g ? g : 1) : 65536);
}

}  // namespace

hipError_t launch_embed(const uint16_t *table, uint32_t hidden, const uint32_t *tokens,
                        uint32_t rows, float *out, hipStream_t stream) {
    if (rows == 0 || hidden == 0) return hipSuccess;
    KernelTimer timer("embed", stream);
    if (hidden % 8 == 0)
        hipLaunchKernelGGL((embed_kernel<true>), dim3(rows), dim3(kThreads), 0, stream, table, hidden,
                           tokens, out);
    else
        hipLaunchKernelGGL((embed_kernel<false>), dim3(rows), dim3(kThreads), 0, stream, table, hidden,
                           tokens, out);
    return hipGetLastError();
}

hipError_t launch_rmsnorm(const float *x, uint32_t hidden, const uint16_t *weight, float eps,
                          const uint32_t *rows_idx, uint32_t rows, uint16_t *out,
                          hipStream_t stream) {
    if (rows == 0 || hidden == 0) return hipSuccess;
    KernelTimer timer("rmsnorm", stream);
    if (hidden % 8 == 0)
        hipLaunchKernelGGL((rmsnorm_kernel<true>), dim3(rows), dim3(kThreads), 0, stream, x, hidden,
                           weight, eps, rows_idx, out);
    else
        hipLaunchKernelGGL((rmsnorm_kernel<false>), dim3(rows), dim3(kThreads), 0, stream, x, hidden,
                           weight, eps, rows_idx, out);
    return hipGetLastError();
}

hipError_t launch_gather_rows(const void *x, uint32_t row_words, const uint32_t *rows,
                              uint32_t num_rows, void *out, bool vec4, hipStream_t stream) {
    if (num_rows == 0 || row_words == 0) return hipSuccess;
    KernelTimer timer("gather_rows", stream);
    const uint32_t *src = static_cast<const uint32_t *>(x);
    uint32_t *dst = static_cast<uint32_t *>(out);
    if (vec4)
        hipLaunchKernelGGL((gather_rows_kernel<true>), dim3(num_rows), dim3(kThreads), 0, stream, src,
                           row_words, rows, dst);
    else
        hipLaunchKernelGGL((gather_rows_kernel<false>), dim3(num_rows), dim3(kThreads), 0, stream,
                           src, row_words, rows, dst);
    return hipGetLastError();
}

hipError_t launch_add(float *sum, const void *x, bool x_bf16, uint64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    KernelTimer timer("add", stream);
    const uint32_t grid = grid_for(n);
    if (x_bf16)
        hipLaunchKernelGGL((add_kernel<true>), dim3(grid), dim3(kThreads), 0, stream, sum, x, n);
    else
        hipLaunchKernelGGL((add_kernel<false>), dim3(grid), dim3(kThreads), 0, stream, sum, x, n);
    return hipGetLastError();
}

hipError_t launch_silu_mul(const uint16_t *gate, uint32_t gate_ld, const uint16_t *up,
                           uint32_t up_ld, uint32_t rows, uint32_t cols, uint16_t *out,
                           uint32_t out_ld, bool vec8, hipStream_t stream) {
    if (rows == 0 || cols == 0) return hipSuccess;
    KernelTimer timer("silu_mul", stream);
    const uint64_t items = static_cast<uint64_t>(rows) * (vec8 ? cols / 8 : cols);
    const uint32_t grid = grid_for(items);
    if (vec8)
        hipLaunchKernelGGL((silu_mul_kernel<true>), dim3(grid), dim3(kThreads), 0, stream, gate,
                           gate_ld, up, up_ld, rows, cols, out, out_ld);
    else
        hipLaunchKernelGGL((silu_mul_kernel<false>), dim3(grid), dim3(kThreads), 0, stream, gate,
                           gate_ld, up, up_ld, rows, cols, out, out_ld);
    return hipGetLastError();
}

hipError_t launch_argmax(const void *logits, bool f32, uint32_t rows, uint32_t cols, uint32_t *ids,
                         hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    KernelTimer timer("argmax", stream);
    // 16-byte reads where every row starts on a 16-byte boundary; 1024 threads
    // once a row has a word for each.
    const uint32_t per_word = f32 ? 4 : 8;
    const bool wide = cols % per_word == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0;
#define VO_ARGMAX(F32, V, T) \
    hipLaunchKernelGGL((argmax_kernel<F32, V, T>), dim3(rows), dim3(T), 0, stream, logits, cols, ids)
    if (wide) {
        const bool large = cols / per_word >= 1024;
        if (f32 && large) VO_ARGMAX(true, 4, 1024);
        else if (f32) VO_ARGMAX(true, 4, 256);
        else if (large) VO_ARGMAX(false, 8, 1024);
        else VO_ARGMAX(false, 8, 256);
    } else {
        const bool large = cols >= 1024;
        if (f32 && large) VO_ARGMAX(true, 1, 1024);
        else if (f32) VO_ARGMAX(true, 1, 256);
        else if (large) VO_ARGMAX(false, 1, 1024);
        else VO_ARGMAX(false, 1, 256);
    }
#undef VO_ARGMAX
    return hipGetLastError();
}

}  // namespace kernels
}  // namespace vo

namespace vo {
namespace kernels {

hipError_t launch_matmul_generic(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t n,
                                 uint32_t k, void *out, bool out_f32, bool accumulate,
                                 hipStream_t stream) {
    const uint64_t items = static_cast<uint64_t>(rows) * n;
    if (items == 0) return hipSuccess;
    const uint64_t grid = (items + kThreads - 1) / kThreads;
    if (grid > 0x7fffffffull) return hipErrorInvalidValue;
    KernelTimer timer("matmul_generic", stream);
    if (out_f32)
        hipLaunchKernelGGL((matmul_generic_kernel<true>), dim3(static_cast<uint32_t>(grid)),
                           dim3(kThreads), 0, stream, x, w, rows, n, k, out, accumulate);
    else
        hipLaunchKernelGGL((matmul_generic_kernel<false>), dim3(static_cast<uint32_t>(grid)),
                           dim3(kThreads), 0, stream, x, w, rows, n, k, out, accumulate);
    return hipGetLastError();
}

}  // namespace kernels
}  // namespace vo

namespace vo {
namespace kernels {

namespace {

enum SkinnyKernel { kLibrary, kHalves, kWhole, kStream };

// Which kernel runs a product of few rows, from times of weights of 1024 to
// 128256 rows and 2048 to 28672 columns (GPU us a call, replayed from a graph
// over weights that are not cached; own kernel / library):
//  - skinny_gemm_kernel: small weights (above), and up to 4 rows of weights of
//    more than 4096 columns and 16384 to 65536 rows: 16384 x 8192, 1 row 51.8,
//    stream 64.7, library 65.5; 57344 x 8192 162, 187, 178; but 8192 x 28672
//    92.8, 85.6, 88.4, 10240 x 8192 38.1, 42.0, 36.0, 128256 x 8192, 4 rows
//    388, 360, 363.
//  - up to 16 rows stream_gemm_kernel: 4096 x 4096 9.9 / 12.7, 6144 x 4096
//    13.7 / 14.5, 16384 x 2048 14.9 / 17.7, 28672 x 4096 45.0 / 63.0, 8192 x
//    14336 45.9 / 51.7.  Not past 5120 columns where the tiles leave CUs idle
//    (6144 x 8192 24.8 / 23.2), or 4096 below 16384 rows (10240 x 8192 40.9 /
//    35.6) and past 32768 (128256 x 8192 372 / 359).  Up to 4096 weight rows
//    the library's 6 us more of host time a call count: an MLP, op by op, of
//    2048 x 8192 and 9 to 16 rows takes 45.8 us with this kernel (15.1 alone,
//    the library 13.1) and 54.6, though a whole decode step of 9 or 12
//    sequences, bound by the GPU, 1229 and 1165; 4096 x 14336, 12 rows 26.5 /
//    26.4, the MLP 73.2 and 74.0, 16 rows 27.8 / 27.0, 75.2 and 74.6.  (4096 x
//    11264, 12 rows, 21.7 / 20.1, is on the wrong side of that line.)
//  - 17 to 64 rows, where every workgroup stages more of x: the line is at
//    fewer columns the more rows there are.  4096 x 2048, 64 rows 10.9 / 12.0;
//    4096 x 4096, 32 rows 11.6 / 13.1, 33 rows 15.8 / 13.3; 6144 x 3072, 64
//    rows 16.6 / 17.5; 6144 x 4096, 48 rows 17.4 / 17.3, 64 rows 19.0 / 17.9;
//    8192 x 8192, 32 rows 31.7 / 30.2; 12288 x 4096, 32 rows 23.3 / 23.6, 48
//    rows 25.6 / 24.9; 28672 x 4096, 64 rows 50.9 / 56.0; 32768 x 5120, 32
//    rows 66.8 / 60.5; 128256 x 8192, 32 rows 349 / 381.
// The host time also decides 5120 .. 7168 x 4096 at 24 and 32 rows, where both
// are within 3%.
SkinnyKernel skinny_kernel(uint64_t rows, uint64_t n, uint64_t k) {
    if (rows < 1 || rows > 64 || n < 16 || n % 16 != 0 || n / 16 > 0x7fffffffull || k < 512 ||
        k % 512 != 0 || k > (1u << 24))
        return kLibrary;
    const bool small = n * k <= kSkinnyWeight;
    if (small && rows <= 8 && n <= kSkinnyHalfN && k % (kSkinnyWaves * 2 * 32 * 2) == 0) return kHalves;
    if (rows <= 4 && k % (kSkinnyWaves * 32 * 8) == 0 && (small || (n >= 16384 && n <= 65536 && k > 4096)))
        return kWhole;
    bool stream;
    if (rows <= 16) {
        if (n <= 4096)
            stream = k <= 8192 || rows <= 12;
        else if (n <= 8192)
            stream = k <= 5120 || n > 7168 || rows <= 4;
        else
            stream = k <= 4096 || (n >= 16384 && n <= 32768 && k <= 8192);
    } else if (k > 2 * n) {
        stream = false;
    } else if (n <= 4096) {
        stream = k <= (rows <= 32 ? 4096 : 2048);
    } else if (n <= 8192) {
        stream = k <= (rows <= 48 ? 4096 : 3072);
    } else if (n < 16384) {
        stream = k <= (rows <= 32 ? 4096 : 2048);
    } else {
        stream = k <= 4096 || n >= 98304;
    }
    return stream ? kStream : kLibrary;
}

}  // namespace

bool skinny_gemm_supported(uint64_t rows, uint64_t n, uint64_t k) {
    return skinny_kernel(rows, n, k) != kLibrary;
}

bool swiglu_gemm_supported(uint64_t rows, uint64_t ffn, uint64_t k) {
    const SkinnyKernel kernel = skinny_kernel(rows, 2 * ffn, k);
    return ffn % 16 == 0 && kernel != kLibrary && (kernel != kWhole || 2 * ffn * k <= kSkinnyWeight);
}

hipError_t launch_skinny_gemm(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t n,
                              uint32_t k, void *out, bool out_f32, bool accumulate,
                              hipStream_t stream) {
    const SkinnyKernel kernel = skinny_kernel(rows, n, k);
    if (kernel == kLibrary) return hipErrorInvalidValue;
    KernelTimer timer("matmul_skinny", stream);
    const int mode = !out_f32 ? 0 : (accumulate ? 2 : 1);
    if (kernel == kStream) return launch_stream_any(x, w, rows, n, k, out, mode, stream);
    const dim3 block(64 * kSkinnyWaves);
#define VO_SKINNY(P, U)                                                                          \
    do {                                                                                         \
        const dim3 grid(n / 16 * P);                                                             \
        if (mode == 0)                                                                           \
            hipLaunchKernelGGL((skinny_gemm_kernel<0, P, U>), grid, block, 0, stream, x, w, rows, \
                               n, k, out);                                                       \
        else if (mode == 1)                                                                      \
            hipLaunchKernelGGL((skinny_gemm_kernel<1, P, U>), grid, block, 0, stream, x, w, rows, \
                               n, k, out);                                                       \
        else                                                                                     \
            hipLaunchKernelGGL((skinny_gemm_kernel<2, P, U>), grid, block, 0, stream, x, w, rows, \
                               n, k, out);                                                       \
    } while (0)
    if (kernel == kHalves)
        VO_SKINNY(2, 2);
    else
        VO_SKINNY(1, 8);
#undef VO_SKINNY
    return hipGetLastError();
}

// Up to 8 rows of 2048 values, 4 for a weight of 8192 rows and more, where
// the product's own time hides less of them (figures at norm_gemm_kernel): as
// many as the workgroup has wavefronts.  Longer rows lose or gain nothing:
// 6144 x 4096, 1 and 4 rows, 19.3 and 20.2 us against 15.4 and 15.8 as two
// launches; 28672 x 4096 with SwiGLU 46.0 and 45.2 against 46.2 and 46.3, no
// more than runs differ.
bool norm_gemm_supported(uint64_t rows, uint64_t n, uint64_t k, bool swiglu) {
    const uint32_t kg = n >= 8192 ? 1 : swiglu ? 4 : 8;
    return rows >= 1 && rows <= (n >= 8192 ? 4 : kNormGemmRows) && k >= 512 && k <= kNormGemmK &&
           k % 512 == 0 && k % (256 * kg) == 0 && n >= 16 && n <= 0x7fffffffull &&
           n % (swiglu ? 32 : 16) == 0;
}

hipError_t launch_norm_gemm(const float *x, const uint16_t *norm, float eps, const uint16_t *w,
                            uint32_t rows, uint32_t n, uint32_t k, bool swiglu, uint16_t *out,
                            hipStream_t stream) {
    if (!norm_gemm_supported(rows, n, k, swiglu)) return hipErrorInvalidValue;
    KernelTimer timer("matmul_norm", stream);
#define VO_NORM(MODE, NW, KG)                                                                \
    hipLaunchKernelGGL((norm_gemm_kernel<MODE, NW, KG>), dim3((n + 16 * NW - 1) / (16 * NW)), \
                       dim3(64 * NW * KG), 0, stream, x, norm, eps, w, rows, n, k, out, QkvRope{})
    if (swiglu && n >= 8192) VO_NORM(3, 4, 1);
    else if (swiglu) VO_NORM(3, 2, 4);
    else if (n >= 8192) VO_NORM(0, 4, 1);
    else VO_NORM(0, 1, 8);
#undef VO_NORM
    return hipGetLastError();
}

hipError_t launch_norm_qkv_rope(const float *x, const uint16_t *norm, float eps, const uint16_t *w,
                                uint32_t rows, uint32_t k, const QkvRope &to, hipStream_t stream) {
    const uint64_t n = to.q_cols + 2ull * to.kv_heads * to.head_dim;
    if (!norm_gemm_supported(rows, n, k, false) || (to.head_dim != 64 && to.head_dim != 128) ||
        to.q_cols % to.head_dim != 0)
        return hipErrorInvalidValue;
    KernelTimer timer("matmul_norm", stream);
    const uint32_t tiles = static_cast<uint32_t>(n / 16);
    if (n >= 8192)
        hipLaunchKernelGGL((norm_gemm_kernel<4, 4, 1>), dim3((tiles + 3) / 4), dim3(256), 0, stream,
                           x, norm, eps, w, rows, static_cast<uint32_t>(n), k, nullptr, to);
    else
        hipLaunchKernelGGL((norm_gemm_kernel<4, 1, 8>), dim3(tiles), dim3(512), 0, stream, x, norm,
                           eps, w, rows, static_cast<uint32_t>(n), k, nullptr, to);
    return hipGetLastError();
}

hipError_t launch_swiglu_gemm(const uint16_t *x, const uint16_t *w, uint32_t rows, uint32_t ffn,
                              uint32_t k, uint16_t *out, hipStream_t stream) {
    if (!swiglu_gemm_supported(rows, ffn, k)) return hipErrorInvalidValue;
    KernelTimer timer("matmul_swiglu", stream);
    return launch_stream_any(x, w, rows, 2 * ffn, k, out, 3, stream);
}

}  // namespace kernels
}  // namespace vo
