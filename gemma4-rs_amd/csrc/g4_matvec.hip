// Mat-vecs over the GGUF weight formats the engine keeps (Q8_0, BF16, F32)
// and the activations fused into them (Gemma's GELU-gated FFN input, the
// logit soft-cap): crates/llm-backend-cpu/src/matvec.rs, ops.rs:79-103.
//
// Every kernel reproduces the reference's arithmetic exactly: the integer
// block dots are exact in any order, and every floating-point sum is taken
// in the reference's order -- a row's block products (Q8_0) or element
// products (BF16, F32, dequantized Q8_0) added one after another from -0.0,
// as Rust's `Iterator::sum` does.  Only tanh inside GELU and the soft-cap
// comes from the device's libm.
//
// Q8_0 with quantized activations (the engine's default numerics) is the
// HBM-bound hot path: a wavefront takes a run of rows, streams their bytes
// into LDS with 16-byte direct-to-LDS loads (rows of 34-byte blocks are
// 16-byte aligned when cols is a multiple of 256), and lane b then takes
// block b: its f16 scale and 32 int8 values against the activation's block b
// (held in the lane's registers for the whole kernel), 8 v_dot4 steps.  The
// block products go to a table in LDS that lane r then sums for row r in
// block order, so the run's sequential sums proceed side by side.  Matrices
// below the output head's size bring all their rows at once instead, with the
// activation quantized once per workgroup (f32 activations, the engine's
// comparison numerics, go the same way).  BF16 and F32 rows, one sum per
// element, split the loading and the adding over two wavefronts.  Many short
// rows take a lane each, in every format.

#include <algorithm>
#include <type_traits>

#include "g4_internal.h"

namespace g4 {
namespace {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

constexpr int kQ8Values = 32;  // values per Q8_0 block
constexpr int kQ8Bytes = 34;   // f16 scale + 32 int8
// Buffer resource (V#) word 3 for raw buffers on gfx950.
constexpr int kBufferWord3 = 0x00020000;
constexpr int kVmcntZero = 0x0F70;  // s_waitcnt vmcnt(0), other counters untouched

// Cache-policy operand of a buffer load: NT, non-temporal.  Large matrices
// stream their weights with it (output head 84.6 -> 78.9 us); small ones,
// which stay latency-bound, were 0.6 us slower with it.
constexpr int kNonTemporal = 2;

// One 16-byte load per active lane from `rsrc` at byte offset voff, written
// straight to LDS at lds + 16 * lane (lds is the same for the whole
// wavefront); AUX is the cache policy.
template <int AUX>
__device__ inline void load_to_lds(__amdgpu_buffer_rsrc_t rsrc, u32x4 *lds, uint32_t voff) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void *)lds, 16, voff, 0, 0, AUX);
#endif
}

__device__ inline float half_bits_to_float(unsigned bits) {
    return (float)__builtin_bit_cast(_Float16, (unsigned short)(bits & 0xffffu));
}

// f16 rounding of an f32 value (half::f16::from_f32).  The empty asm makes
// x opaque: otherwise the compiler fuses a product that feeds the conversion
// into one mixed-precision fma (v_fma_mixlo_f16 a, b, 0), which rounds the
// exact product to f16 once -- where the reference rounds it to f32 first --
// and turns a -0 product into +0.
__device__ inline float round_to_half(float x) {
    asm volatile("" : "+v"(x));
    return (float)(_Float16)x;
}

// Rust's `f32 as i8`: saturating, NaN -> 0.
__device__ inline int saturate_i8(float v) {
    if (v != v) return 0;
    return (int)fminf(fmaxf(v, -128.0f), 127.0f);
}

// ops.rs:85-89, evaluated left to right as rustc does (no contraction).
__device__ inline float gelu_tanh(float x) {
#pragma clang fp contract(off)
    return 0.5f * x * (1.0f + tanhf(0.7978846f * x * (1.0f + 0.044715f * x * x)));
}

// ops.rs:95-103
__device__ inline float gelu_tanh_fp16_table(float x) {
    if (x <= -10.0f) return 0.0f;
    if (x >= 10.0f) return x;
    return round_to_half(gelu_tanh(round_to_half(x)));
}

// quantize_q8_0 (matvec.rs:35-53): 32 lanes per block; max |x| over the
// block (NaN ignored, as f32::max does), scale = max/127 kept as its f16
// rounding, values x * (1/scale) rounded half to even and saturated.
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float *x, int64_t n, float *scales,
                                                            signed char *quants) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const float v = i < n ? x[i] : 0.0f;
    float m = fmaxf(0.0f, fabsf(v));
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 32));
    const float scale = m / 127.0f;
    const float inverse = scale == 0.0f ? 0.0f : 1.0f / scale;
    if (i >= n) return;
    if ((i & 31) == 0) scales[i >> 5] = round_to_half(scale);
    quants[i] = (signed char)saturate_i8(rintf(v * inverse));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Epilogues of the Q8_0 row kernel.
enum Epilogue : int { kPlain = 0, kSoftcap = 1, kGeglu = 2, kGegluFp16 = 3 };

// W @ x for Q8_0 rows against a Q8_0 activation (matvec.rs:55-102).  A
// workgroup is one wavefront and takes `rb` consecutive rows (rb <= 64), staged into
// LDS `g` rows at a time with direct-to-LDS 16-byte loads.  For each staged
// row, lane b computes block b's product (NS = blocks per lane: b = lane +
// 64 s) into a row-major product table in LDS; once all rows are done, lane
// r sums row r's products in block order -- up to 64 independent sequential
// sums at once, each exactly the reference's.  kGeglu* read a second matrix
// (up) beside the first (gate).  For large matrices: small workgroups, so
// that many are resident per CU (measured faster than double-buffering fewer
// of them).
template <int EPI, int NS>
__global__ __launch_bounds__(64) void matvec_q8_0_kernel(const unsigned char *__restrict__ w,
                                                         const unsigned char *__restrict__ w2, int64_t rows,
                                                         int nb, const float *__restrict__ xs,
                                                         const int *__restrict__ xq, float arg, int g, int rb,
                                                         float *__restrict__ out) {
#pragma clang fp contract(off)
    extern __shared__ u32x4 lds[];
    constexpr int NM = EPI >= kGeglu ? 2 : 1;  // matrices read
    const int lane = threadIdx.x;
    const int row_len = nb * kQ8Bytes;  // bytes, a multiple of 16
    const int chunks = row_len >> 4;    // 16-byte chunks per row
    const int pstride = nb + 1;         // product table row stride (odd: no bank conflicts)
    u32x4 *stage = lds;                                  // [g][NM][chunks]
    float *prod = (float *)(lds + (size_t)g * NM * chunks);  // [NM][rb][pstride]

    const int64_t row0 = (int64_t)blockIdx.x * rb;
    const int n_rows = (int)min((int64_t)rb, rows - row0);  // >= 1: the grid covers the rows exactly
    // Stage rows r0 .. r0 + min(g, n_rows - r0) - 1 of each matrix.
    auto stage_rows = [&](int r0) {
        const int nr = min(g, n_rows - r0);
        for (int r = 0; r < nr; ++r)
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                    (void *)((m == 0 ? w : w2) + (row0 + r0 + r) * row_len), 0, row_len, kBufferWord3);
                u32x4 *dst = stage + (r * NM + m) * chunks;
                for (int k = 0; k * 64 < chunks; ++k)
                    if (k * 64 + lane < chunks)
                        load_to_lds<kNonTemporal>(rs, dst + 64 * k, (uint32_t)(k * 64 + lane) * 16u);
            }
    };
    // The first rows' loads are in flight while the activation is read: this
    // lane's blocks, 8 packed int8 dwords and the scale each.
    stage_rows(0);
    int xqr[NS][8];
    float xsr[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int b = lane + 64 * s;
#pragma unroll
        for (int j = 0; j < 8; ++j) xqr[s][j] = 0;
        xsr[s] = 0.0f;
        if (b < nb) {
#pragma unroll
            for (int j = 0; j < 8; ++j) xqr[s][j] = xq[b * 8 + j];
            xsr[s] = xs[b];
        }
    }

    for (int r0 = 0; r0 < n_rows; r0 += g) {
        const int nr = min(g, n_rows - r0);
        if (r0 > 0) stage_rows(r0);
        __builtin_amdgcn_s_waitcnt(kVmcntZero);
        __syncthreads();
        for (int r = 0; r < nr; ++r)
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const unsigned *rw = (const unsigned *)(stage + (r * NM + m) * chunks);
                float *pr = prod + ((size_t)m * rb + r0 + r) * pstride;
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const int b = lane + 64 * s;
                    if (b < nb) {
                        // Block b starts at byte 34b: dword 17(b/2), offset 0
                        // (even b: scale in the low half, values from byte 2)
                        // or dword 17(b/2) + 8, offset 2 (odd b: scale in the
                        // high half, values dword-aligned after it).
                        const unsigned *d = rw + 17 * (b >> 1) + ((b & 1) ? 8 : 0);
                        unsigned raw[9];
#pragma unroll
                        for (int j = 0; j < 9; ++j) raw[j] = d[j];
                        int dot = 0;
                        float ws;
                        if (b & 1) {
                            ws = half_bits_to_float(raw[0] >> 16);
#pragma unroll
                            for (int j = 0; j < 8; ++j) dot = __builtin_amdgcn_sdot4((int)raw[j + 1], xqr[s][j], dot, false);
                        } else {
                            ws = half_bits_to_float(raw[0]);
#pragma unroll
                            for (int j = 0; j < 8; ++j)
                                dot = __builtin_amdgcn_sdot4((int)__builtin_amdgcn_alignbyte(raw[j + 1], raw[j], 2),
                                                             xqr[s][j], dot, false);
                        }
                        // matvec.rs:148: `dot as f32 * (w_scale * x_scale)`
                        pr[b] = (float)dot * (ws * xsr[s]);
                    }
                }
            }
        __syncthreads();  // the stage is refilled next; the products are complete
    }
    if (lane >= n_rows) return;
    // Lane r: row r's block products summed in block order.
    float acc[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const float *pr = prod + ((size_t)m * rb + lane) * pstride;
        float sum = -0.0f;
        for (int b = 0; b < nb; ++b) sum += pr[b];
        acc[m] = sum;
    }
    float v = acc[0];
    if constexpr (EPI == kSoftcap) v = tanhf(v * (1.0f / arg)) * arg;  // ops.rs:79-81
    if constexpr (EPI == kGeglu) v = gelu_tanh(acc[0]) * acc[NM - 1];
    if constexpr (EPI == kGegluFp16) v = gelu_tanh_fp16_table(acc[0]) * acc[NM - 1];
    out[row0 + lane] = v;
}

// LDS of matvec_q8_0_once_kernel, in bytes unless said: the activation, then
// per row wavefront the rows it brings (per matrix) and its product table.
struct Q8OnceLds {
    int padded, pstride;  // products per row: rounded up to 16, and apart
    int act, stage, wave;
    __host__ __device__ Q8OnceLds(int nb, int rw, int nm, int value_bytes, int act_block)
        : padded((nb + 15) / 16 * 16), pstride(padded + 16 / value_bytes), act((nb * act_block * 4 + 15) / 16 * 16),
          stage((rw * nb * kQ8Bytes + 2 + 15) / 16 * 16), wave(nm * (stage + rw * pstride * value_bytes)) {}
};

// What a block's product is: the integer dot of quantized activations, or
// the sequential f32 / f64 sum against f32 activations.
enum Dot : int { kInt8 = 0, kF32 = 1, kF64 = 2 };

// Largest of v over each run of 8 lanes (NaN ignored, as fmaxf does).
__device__ inline float max8(float v) {
    auto from = [](float x, auto ctrl) {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true));
    };
    v = fmaxf(v, from(v, std::integral_constant<int, 0xB1>()));  // quad_perm [1,0,3,2]
    v = fmaxf(v, from(v, std::integral_constant<int, 0x4E>()));  // quad_perm [2,3,0,1]
    return fmaxf(v, from(v, std::integral_constant<int, 0x141>()));  // row_half_mirror
}

// Dwords of an activation block in LDS: 8 of int8 values and the scale, or
// 32 f32 values, padded so that 16-byte reads by consecutive lanes spread
// over the banks.
template <int DOT> constexpr int kActBlock = DOT == kInt8 ? 12 : 36;

// The activation into LDS by nq wavefronts (t: thread among them), 8 lanes
// per block, 6 blocks of a lane group in flight: quantized here when it
// comes as f32 (the arithmetic of quantize_q8_0_kernel), else copied.
template <int DOT>
__device__ inline void stage_activation(float *act, int nb, const float *xs, const int *xq, const float *xf, int t,
                                        int nq) {
#pragma clang fp contract(off)
    const int j = t & 7, step = 8 * nq;
    if (DOT == kInt8 && xs) {
        for (int b = t >> 3; b < nb; b += step) {
            ((int *)act)[b * 12 + j] = xq[b * 8 + j];
            if (j == 0) act[b * 12 + 8] = xs[b];
        }
        return;
    }
    constexpr int NF = 6;
    const bool aligned = ((uintptr_t)xf & 15) == 0;
    for (int b0 = t >> 3; b0 < nb; b0 += NF * step) {
        f32x4 v[NF];
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            const float *src = xf + kQ8Values * min(b0 + i * step, nb - 1) + 4 * j;
            if (aligned)
                v[i] = *(const f32x4 *)src;
            else
                v[i] = f32x4{src[0], src[1], src[2], src[3]};
        }
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            const int b = b0 + i * step;
            if (b >= nb) break;
            if constexpr (DOT == kInt8) {
                float m = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k) m = fmaxf(m, fabsf(v[i][k]));
                const float scale = max8(m) / 127.0f;
                const float inverse = scale == 0.0f ? 0.0f : 1.0f / scale;
                unsigned packed = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    packed |= ((unsigned)saturate_i8(rintf(v[i][k] * inverse)) & 0xffu) << (8 * k);
                ((int *)act)[b * 12 + j] = (int)packed;
                if (j == 0) act[b * 12 + 8] = round_to_half(scale);
            } else {
                *(f32x4 *)(act + b * 36 + 4 * j) = v[i];
            }
        }
    }
}

// W @ x for Q8_0 rows, the matrices that do not fill the chip for long
// (everything but a whole output head).  They are bound by one trip to memory,
// so every byte is asked for at once: about one workgroup per CU, whose nw
// row wavefronts each bring rw consecutive rows (one run of bytes, per
// matrix) into LDS with 16-byte direct-to-LDS loads, while nq further
// wavefronts load the activation, quantize it once for the workgroup and
// leave it in LDS.  Those are other wavefronts because load counters
// complete in order: a row wavefront that also read the activation would
// wait for its rows first.  Then lane b of a row wavefront forms block b's
// product of each of its rows (b = lane, lane + 64, ...) in a table, and
// lane r sums row r's products in block order.  Rows need not be 16-byte
// aligned: a run is loaded from the dword its first byte lies in, its last
// bytes (fewer than 16) as 2-byte values.
// Weights from HBM, activation as f32 (one wavefront per two or three rows
// that quantized the activation for itself, before -> here): 2048 x 1536
// 5.4 -> 4.0 us, 4096 x 1536 6.3 -> 5.0, 1536 x 6144 11.3 -> 7.1, gate and up
// of 6144 x 1536 (20.1 MB) 10.3 -> 7.6; a plain read of 16 MiB takes 4.7.
// f32 activations, one lane per row before: 2048 x 1536 27 -> 3.8 us,
// 1536 x 6144 172 -> 7.0.
template <int EPI, int DOT>
__global__ __launch_bounds__(768) void matvec_q8_0_once_kernel(const unsigned char *__restrict__ w,
                                                               const unsigned char *__restrict__ w2, int64_t rows,
                                                               int nb, const float *__restrict__ xs,
                                                               const int *__restrict__ xq,
                                                               const float *__restrict__ xf, float arg, int nw, int nq,
                                                               int rw, float *__restrict__ out) {
#pragma clang fp contract(off)
    using T = typename std::conditional<DOT == kF64, double, float>::type;
    typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
    constexpr int NM = EPI >= kGeglu ? 2 : 1;  // matrices read
    constexpr int V = 16 / sizeof(T);          // products per 16-byte read
    extern __shared__ u32x4 lds[];
    float *act = (float *)lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Q8OnceLds at(nb, rw, NM, (int)sizeof(T), kActBlock<DOT>);
    if (wave >= nw) {
        stage_activation<DOT>(act, nb, xs, xq, xf, threadIdx.x - 64 * nw, nq);
        __syncthreads();
        return;
    }
    unsigned char *mine = (unsigned char *)lds + at.act + (size_t)wave * at.wave;  // this wavefront's rows and products
    T *prod = (T *)(mine + NM * at.stage);                                         // [NM][rw][pstride]
    const int row_len = nb * kQ8Bytes;
    const int64_t row0 = ((int64_t)blockIdx.x * nw + wave) * rw;
    const int n = (int)max((int64_t)0, min((int64_t)rw, rows - row0));
    const int64_t first = row0 * row_len;
    const int skew = (int)(first & 3);  // 0 or 2
    if (n > 0) {
        const int bytes = n * row_len + skew, chunks = bytes >> 4, rest = bytes & 15;
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const unsigned char *src = (m == 0 ? w : w2) + (first - skew);
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc((void *)src, 0, chunks * 16, kBufferWord3);
            u32x4 *dst = (u32x4 *)(mine + m * at.stage);
            for (int k = 0; k < chunks; k += 64)
                if (k + lane < chunks) load_to_lds<0>(rs, dst + k, (uint32_t)(k + lane) * 16u);
            if (2 * lane < rest)
                ((unsigned short *)(dst + chunks))[lane] = ((const unsigned short *)(src + chunks * 16))[lane];
        }
    }
    __builtin_amdgcn_s_waitcnt(kVmcntZero);
    __syncthreads();
    if (n <= 0) return;

    for (int b = lane; b < at.padded; b += 64) {
        int xi[8];
        float xr[DOT == kInt8 ? 1 : kQ8Values];
        if constexpr (DOT == kInt8) {
            const int *src = (const int *)act + min(b, nb - 1) * 12;
#pragma unroll
            for (int j = 0; j < 8; ++j) xi[j] = src[j];
            xr[0] = ((const float *)src)[8];
        } else {
            const float *src = act + min(b, nb - 1) * 36;
#pragma unroll
            for (int j = 0; j < kQ8Values; ++j) xr[j] = src[j];
        }
        for (int r = 0; r < n; ++r)
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                T *pr = prod + (m * rw + r) * at.pstride + b;
                if (b >= nb) {  // every sum keeps -0.0
                    *pr = (T)-0.0;
                    continue;
                }
                // The block's scale is in its first two bytes, the values
                // follow: in 9 dwords, one half left over.
                const int off = skew + r * row_len + kQ8Bytes * b;
                const unsigned *d = (const unsigned *)(mine + m * at.stage) + (off >> 2);
                unsigned raw[9], q[8];
#pragma unroll
                for (int j = 0; j < 9; ++j) raw[j] = d[j];
                const bool high = off & 2;
                const float ws = half_bits_to_float(high ? raw[0] >> 16 : raw[0]);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    q[j] = high ? raw[j + 1] : __builtin_amdgcn_alignbyte(raw[j + 1], raw[j], 2);
                if constexpr (DOT == kInt8) {
                    int dot = 0;
#pragma unroll
                    for (int j = 0; j < 8; ++j) dot = __builtin_amdgcn_sdot4((int)q[j], xi[j], dot, false);
                    *pr = (float)dot * (ws * xr[0]);  // matvec.rs:148
                } else {  // matvec.rs:153-176: the 32 products in order, then the scale
                    T dot = (T)-0.0;
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            dot += (T)(int)(signed char)(q[j] >> (8 * k)) * (T)xr[4 * j + k];
                    *pr = dot * (T)ws;
                }
            }
    }
    // Lane m*rw + r sums row r of matrix m, 16 products at a time with the
    // next 32 on their way: 16 adds are shorter than an LDS read (1536 x
    // 6144 with only 16 ahead 7.5 us, 7.1 so; five layers' calls 167.7 ->
    // 163.2).
    T sum = (T)-0.0;
    if (lane < NM * rw) {
        const vec *pr = (const vec *)(prod + lane * at.pstride);
        const int groups = at.padded / 16;
        vec v[3][16 / V];
        auto read = [&](int g, vec (&dst)[16 / V]) {
#pragma unroll
            for (int i = 0; i < 16 / V; ++i) dst[i] = pr[min(g, groups - 1) * (16 / V) + i];
        };
        read(0, v[0]);
        read(1, v[1]);
        for (int g = 0; g < groups; g += 3) {
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                if (g + p >= groups) break;
                read(g + p + 2, v[(p + 2) % 3]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int i = 0; i < 16 / V; ++i)
#pragma unroll
                    for (int k = 0; k < V; ++k) sum += v[p][i][k];
            }
        }
    }
    float v = (float)sum;
    if constexpr (EPI == kSoftcap) v = tanhf(v * (1.0f / arg)) * arg;  // ops.rs:79-81
    if constexpr (NM == 2) {
        const float up = __shfl(v, lane + rw);
        v = (EPI == kGeglu ? gelu_tanh(v) : gelu_tanh_fp16_table(v)) * up;
    }
    if (lane < n) out[row0 + lane] = v;
}

// Reads the 34-byte Q8_0 block at byte `off` of a row (2-byte aligned):
// its f16 scale and the 32 values packed 4 to a dword.
__device__ inline float load_q8_block(const unsigned short *row16, int64_t off, unsigned (&q)[8]) {
    const unsigned short *p = row16 + off / 2;
    const float scale = half_bits_to_float(p[0]);
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = (unsigned)p[1 + 2 * j] | ((unsigned)p[2 + 2 * j] << 16);
    return scale;
}

// Q8_0 against a Q8_0 activation, one lane per row (any cols multiple of 32):
// the same block products and order as matvec_q8_0_kernel.
template <int EPI>
__global__ __launch_bounds__(256) void matvec_q8_0_rowwise_kernel(const unsigned char *__restrict__ w,
                                                                  const unsigned char *__restrict__ w2,
                                                                  int64_t rows, int nb, const float *__restrict__ xs,
                                                                  const int *__restrict__ xq, float arg,
                                                                  float *__restrict__ out) {
#pragma clang fp contract(off)
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    constexpr int NM = EPI >= kGeglu ? 2 : 1;
    const int64_t row_len = (int64_t)nb * kQ8Bytes;
    float acc[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        const unsigned short *r16 = (const unsigned short *)((m == 0 ? w : w2) + row * row_len);
        float sum = -0.0f;
        for (int b = 0; b < nb; ++b) {
            unsigned q[8];
            const float ws = load_q8_block(r16, (int64_t)b * kQ8Bytes, q);
            int dot = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) dot = __builtin_amdgcn_sdot4((int)q[j], xq[b * 8 + j], dot, false);
            sum += (float)dot * (ws * xs[b]);
        }
        acc[m] = sum;
    }
    float v = acc[0];
    if constexpr (EPI == kSoftcap) v = tanhf(v * (1.0f / arg)) * arg;
    if constexpr (EPI == kGeglu) v = gelu_tanh(acc[0]) * acc[NM - 1];
    if constexpr (EPI == kGegluFp16) v = gelu_tanh_fp16_table(acc[0]) * acc[NM - 1];
    out[row] = v;
}

// matvec_q8_0_f32 / matvec_q8_0_f64_sums (matvec.rs:104-122, 153-176): f32
// activations against dequantized blocks, one lane per row.  Per block the
// 32 products summed in order, times the scale; the blocks summed in order
// (F64: every sum in f64, one rounding at the end).
template <bool F64>
__global__ __launch_bounds__(256) void matvec_q8_0_f32_kernel(const unsigned char *__restrict__ w, int64_t rows,
                                                              int nb, const float *__restrict__ x,
                                                              float *__restrict__ out) {
#pragma clang fp contract(off)
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    const unsigned short *r16 = (const unsigned short *)(w + row * (int64_t)nb * kQ8Bytes);
    using T = typename std::conditional<F64, double, float>::type;
    T sum = (T)-0.0;
    for (int b = 0; b < nb; ++b) {
        unsigned q[8];
        const float scale = load_q8_block(r16, (int64_t)b * kQ8Bytes, q);
        T dot = (T)-0.0;
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int v = (int)(signed char)(q[j] >> (8 * k));
                dot += (T)v * (T)x[b * kQ8Values + 4 * j + k];
            }
        sum += dot * (T)scale;
    }
    out[row] = (float)sum;
}

// matvec.rs:196-204 (f32_to_bf16) and 192-194.
__device__ inline float round_to_bf16(float value) {
    const unsigned bits = __float_as_uint(value);
    unsigned h;
    if (value != value)
        h = (bits >> 16) | 64u;
    else
        h = (bits + (0x7fffu + ((bits >> 16) & 1u))) >> 16;
    return __uint_as_float(h << 16);
}

// A value of a BF16 or F32 row as f32, and the activation it meets
// (matvec_bf16 rounds x to bf16 first).
__device__ inline float weight_value(unsigned short w) { return __uint_as_float((unsigned)w << 16); }
__device__ inline float weight_value(float w) { return w; }
__device__ inline float activation_value(unsigned short, float x) { return round_to_bf16(x); }
__device__ inline float activation_value(float, float x) { return x; }

// Waits for this wavefront's LDS work, then the workgroup barrier; loads in
// flight stay in flight (__syncthreads would wait for them too).
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// matvec_bf16 / matvec_f32 (matvec.rs:124-136, 178-184): every row is one
// sequential f32 sum of its rounded products, so what bounds a row is its
// chain of adds (one VALU issue, 4 cycles, per element: 2.6 us for 1536
// columns), and everything else has to stay off the wavefront that adds.  A
// workgroup of two wavefronts takes R rows.  The first loads them kDenseCols
// columns at a time (16 bytes per lane, P chunks in flight in registers) and
// puts the products into one of two tables in LDS; in the other, lane r of
// the second adds row r's products in order, four to a 16-byte read.
// Products past the row's end are -0.0, which every sum keeps.  8960 x 1536
// (weights from HBM) takes 9.9 us in bf16 and 13.9 in f32, against 213 us in
// bf16 with one lane walking each row in memory (its loads are a row apart)
// and 14.0 / 14.7 us with one wavefront doing both parts.
// VEC: rows are read with 16-byte loads through buffer resources: whole loads
// per row, a matrix on a 4-byte boundary and offsets below 2^31; otherwise
// value by value.
constexpr int kDenseCols = 256;

template <typename W, int R, int P, bool VEC>
__global__ __launch_bounds__(128) void matvec_dense_kernel(const W *__restrict__ w, int64_t rows, int64_t cols,
                                                           const float *__restrict__ x, float *__restrict__ out) {
#pragma clang fp contract(off)
    constexpr int E = 16 / sizeof(W);    // values per load
    constexpr int LPR = kDenseCols / E;  // lanes per row and chunk
    constexpr int RPI = 64 / LPR;        // rows per load
    constexpr int NLD = R / RPI;
    constexpr int TS = kDenseCols + 4;   // table row stride: rows 4 banks apart
    static_assert(R % RPI == 0 && R <= 64, "whole loads; a lane per row");
    __shared__ f32x4 table[2][R * TS / 4];
    const int lane = threadIdx.x & 63;
    const int64_t row0 = (int64_t)blockIdx.x * R;
    const int n_rows = (int)min((int64_t)R, rows - row0);
    const int chunks = (int)((cols + kDenseCols - 1) / kDenseCols);

    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) {  // the products
        const int sub = lane / LPR, g = lane % LPR;
        const W *base = w + row0 * cols;
        const uint32_t row_bytes = (uint32_t)(cols * sizeof(W));  // VEC: R * row_bytes < 2^31
        const __amdgpu_buffer_rsrc_t ws =
            __builtin_amdgcn_make_buffer_rsrc((void *)base, 0, n_rows * row_bytes, kBufferWord3);
        const __amdgpu_buffer_rsrc_t xs =
            __builtin_amdgcn_make_buffer_rsrc((void *)x, 0, (int)(cols * sizeof(float)), kBufferWord3);
        u32x4 wb[P][NLD];
        f32x4 xb[P][E / 4];
        // Chunk c of the rows and of x.  Loads past the last row's end read
        // zeros, past another's end the next row: the column test replaces
        // their products.
        auto load = [&](int c, u32x4 (&wv)[NLD], f32x4 (&xv)[E / 4]) {
            const int64_t col = (int64_t)c * kDenseCols + E * g;
            if constexpr (VEC) {
#pragma unroll
                for (int j = 0; j < E / 4; ++j)
                    xv[j] = __builtin_bit_cast(
                        f32x4, __builtin_amdgcn_raw_buffer_load_b128(xs, (uint32_t)(col + 4 * j) * 4u, 0, 0));
#pragma unroll
                for (int j = 0; j < NLD; ++j)
                    wv[j] = __builtin_amdgcn_raw_buffer_load_b128(
                        ws, (uint32_t)(j * RPI + sub) * row_bytes + (uint32_t)col * (uint32_t)sizeof(W), 0, 0);
            } else {
#pragma unroll
                for (int j = 0; j < E / 4; ++j)
#pragma unroll
                    for (int k = 0; k < 4; ++k) xv[j][k] = col + 4 * j + k < cols ? x[col + 4 * j + k] : 0.0f;
#pragma unroll
                for (int j = 0; j < NLD; ++j) {
                    W v[E];
                    const int r = j * RPI + sub;
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        v[e] = r < n_rows && col + e < cols ? base[r * cols + col + e] : (W)0;
                    wv[j] = __builtin_bit_cast(u32x4, v);
                }
            }
        };
        auto products = [&](int c, const u32x4 (&wv)[NLD], const f32x4 (&xv)[E / 4], auto whole) {
            float xa[E];
#pragma unroll
            for (int e = 0; e < E; ++e) xa[e] = activation_value(W(), xv[e / 4][e % 4]);
            float *t = (float *)table[c & 1] + sub * TS + E * g;
#pragma unroll
            for (int j = 0; j < NLD; ++j) {
                W v[E];
                __builtin_memcpy(v, &wv[j], 16);
#pragma unroll
                for (int q = 0; q < E / 4; ++q) {
                    f32x4 pr;
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int e = 4 * q + k;
                        pr[k] = weight_value(v[e]) * xa[e];
                        if (!decltype(whole)::value && (int64_t)c * kDenseCols + E * g + e >= cols) pr[k] = -0.0f;
                    }
                    *(f32x4 *)(t + j * RPI * TS + 4 * q) = pr;
                }
            }
        };
#pragma unroll
        for (int p = 0; p < P; ++p) load(p, wb[p], xb[p]);
        for (int c0 = 0; c0 < chunks; c0 += P) {
#pragma unroll
            for (int p = 0; p < P; ++p) {
                const int c = c0 + p;
                if (c >= chunks) break;
                if ((int64_t)(c + 1) * kDenseCols <= cols)
                    products(c, wb[p], xb[p], std::true_type());
                else
                    products(c, wb[p], xb[p], std::false_type());
                load(c + P, wb[p], xb[p]);
                lds_barrier();  // chunk c is in its table; chunk c - 1 has been added
            }
        }
        return;
    }
    float sum = -0.0f;
    for (int c = 0; c < chunks; ++c) {
        lds_barrier();
        const f32x4 *tr = table[c & 1] + (lane % R) * (TS / 4);
        const int n = (int)min((int64_t)kDenseCols, cols - (int64_t)c * kDenseCols);
        // 32 products read ahead of the 32 being added.
        f32x4 a[8], b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = tr[i];
#pragma unroll
        for (int s = 0; s < kDenseCols / 32; s += 2) {
            if (32 * s >= n) break;
#pragma unroll
            for (int i = 0; i < 8; ++i) b[i] = tr[8 * (s + 1) + i];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k) sum += a[i][k];
            __builtin_amdgcn_sched_barrier(0);
            if (s + 2 < kDenseCols / 32) {
#pragma unroll
                for (int i = 0; i < 8; ++i) a[i] = tr[8 * (s + 2) + i];
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int k = 0; k < 4; ++k) sum += b[i][k];
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    if (lane < n_rows) out[row0 + lane] = sum;
}

// The same, one lane per row: for many rows of a few values, of which the
// kernel above uses one lane in eight or fewer.
template <typename W>
__global__ __launch_bounds__(256) void matvec_dense_narrow_kernel(const W *__restrict__ w, int64_t rows, int64_t cols,
                                                                  const float *__restrict__ x,
                                                                  float *__restrict__ out) {
#pragma clang fp contract(off)
    const int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= rows) return;
    const W *r = w + row * cols;
    float sum = -0.0f;
    for (int64_t i = 0; i < cols; ++i) sum += weight_value(r[i]) * activation_value(W(), x[i]);
    out[row] = sum;
}

template <int EPI, int NS>
int launch_q8_rows(const MatvecArgs &a, int g, int rb, hipStream_t stream) {
    constexpr int NM = EPI >= kGeglu ? 2 : 1;
    const int nb = (int)(a.cols / kQ8Values);
    const size_t lds = (size_t)g * NM * (nb * kQ8Bytes) + (size_t)NM * rb * (nb + 1) * sizeof(float);
    const int64_t groups = (a.rows + rb - 1) / rb;
    hipLaunchKernelGGL((matvec_q8_0_kernel<EPI, NS>), dim3((unsigned)groups), dim3(64), lds, stream, a.w, a.w2, a.rows,
                       nb, a.xs, (const int *)a.xq, a.arg, g, rb, a.out);
    G4_HIP(hipGetLastError());
    return G4_OK;
}

// Launches matvec_q8_0_once_kernel, or says (*done) that the shape does not
// suit it: a matrix off a 4-byte boundary, no blocks, rows too long for a
// CU's LDS, or more workgroups than a launch takes.
template <int EPI, int DOT>
int launch_q8_once(g4_ctx *ctx, const MatvecArgs &a, hipStream_t stream, bool *done) {
    constexpr int NM = EPI >= kGeglu ? 2 : 1;
    constexpr int kValue = DOT == kF64 ? 8 : 4;
    *done = false;
    const int64_t nb64 = a.cols / kQ8Values;
    if (nb64 <= 0 || nb64 > 8192 || (uintptr_t)a.w % 4 != 0 || (NM == 2 && (uintptr_t)a.w2 % 4 != 0)) return G4_OK;
    const int nb = (int)nb64;
    // One workgroup per CU with a row wavefront per row, up to 8, then more
    // rows per wavefront.  Where that does not fit a CU's LDS, rounds of
    // smaller workgroups, of 4 row wavefronts and five to a CU, whose loads,
    // products and sums overlap (84,752 x 768 17.2 us, 49,152 x 1536 17.8;
    // 8 wavefronts and two to a CU 20.9 and 20.0; three 17.8 and 20.1).
    constexpr size_t kLds = 160 * 1024;
    auto bytes = [&](int nw, int rw) {
        const Q8OnceLds at(nb, rw, NM, kValue, kActBlock<DOT>);
        return (size_t)at.act + (size_t)nw * at.wave;
    };
    const int64_t per_cu = std::min<int64_t>(8 * (64 / NM), (a.rows + ctx->num_cus - 1) / ctx->num_cus);
    int nw = (int)std::min<int64_t>(8, per_cu), rw = (int)((per_cu + nw - 1) / nw);
    if (bytes(nw, rw) > kLds) {
        nw = std::min(nw, 4);
        while (rw > 1 && bytes(nw, rw) > kLds / 5) --rw;
        while (nw > 1 && bytes(nw, rw) > kLds / 5) --nw;
        if (bytes(nw, rw) > kLds) return G4_OK;
    }
    const int nq = std::min(4, (nb + 23) / 24);
    const int64_t groups = (a.rows + (int64_t)nw * rw - 1) / ((int64_t)nw * rw);
    if (groups > (1LL << 22)) return G4_OK;  // a launch holds fewer than 2^32 threads
    hipLaunchKernelGGL((matvec_q8_0_once_kernel<EPI, DOT>), dim3((unsigned)groups), dim3(64 * (nw + nq)),
                       bytes(nw, rw), stream, a.w, a.w2, a.rows, nb, DOT == kInt8 ? a.xs : nullptr,
                       (const int *)a.xq, a.x, a.arg, nw, nq, rw, a.out);
    G4_HIP(hipGetLastError());
    *done = true;
    return G4_OK;
}

// Whether one lane per row is faster than matvec_q8_0_once_kernel, whose
// wavefronts take a lane per block: where rows are so short that most lanes
// idle and so many that the workgroups run in rounds, or so long that a CU's
// LDS holds only a few.  Measured (us, lane per row / at once; the activation
// quantized by a launch of its own in the first):
//   int8 96 columns: 16,384 rows 6.2 / 5.8, 25,000 6.0 / 6.8, 100,000 7.1 / 13.5,
//     262,144 9.8 / 29.9; 224: 32,768 8 / 7, 50,000 8 / 9; 256: 50,000 8 / 9,
//     180,000 20 / 20; 16,384: 32,768 464 / 414, 40,000 467 / 503
//   f32 512: 25,000 11.9 / 11.9, 65,536 14 / 23; 640: 32,768 13 / 14; 768: 50,000
//     18 / 18, 100,000 31 / 28; 8192: 32,768 231 / 198, 50,000 243 / 304
//   f64 256: 8192 10 / 9, 16,384 10 / 12, 262,144 14 / 84; 512: 32,768 13 / 16; 800:
//     50,000 27 / 25, 131,072 40 / 52; 1024: 180,000 69 / 71, 262,144 115 / 101;
//     4096: 32,768 116 / 93, 50,000 118 / 138
template <int DOT, int NM>
bool q8_lane_per_row(int64_t rows, int64_t nb, int64_t num_cus) {
    const int64_t per_cu = rows / num_cus;
    if (DOT == kInt8) {
        if (nb > 256) return nb * rows > (NM == 2 ? 3LL << 23 : 1LL << 24);
        return nb < 8 && per_cu >= 20 * std::max<int64_t>(nb, 4);
    }
    if (nb >= (DOT == kF32 ? 256 : 128)) return per_cu >= 160;
    return nb <= (DOT == kF32 ? 20 : 28) && per_cu >= 8 * std::max<int64_t>(nb, DOT == kF32 ? 10 : 8);
}

template <int EPI>
int launch_q8(g4_ctx *ctx, MatvecArgs a, hipStream_t stream) {
    constexpr int NM = EPI >= kGeglu ? 2 : 1;
    const int num_cus = ctx->num_cus;
    const int64_t nb = a.cols / kQ8Values;
    // Rows start 16-byte aligned when cols is a multiple of 256 and the
    // matrices are (GGUF aligns tensor data to 32 bytes).  An empty row
    // (cols == 0) takes the row-wise kernel, which reads no block.
    const bool aligned = (uintptr_t)a.w % 16 == 0 && (NM == 1 || (uintptr_t)a.w2 % 16 == 0);
    const bool staged = a.cols % 256 == 0 && nb > 0 && nb <= 256 && aligned;
    // Rows per workgroup: up to 16, the product table under 16 KB.
    const int64_t rb_max = std::min<int64_t>(16, std::max<int64_t>(1, 16384 / (NM * (nb + 1) * 4)));
    // The streaming kernel, which needs its activation quantized by a launch
    // of its own, pays from some 128 MB on: 33,017 x 1024 (36 MB) 13.3 us
    // against 11.0 at once, 84,752 x 768 (69 MB) 20.4 against 17.2, 131,072 x
    // 1280 (178 MB) 35.3 against 35.0, the output head (429 MB) 71.0 against
    // 72.1; and earlier where rows at once leave too few bytes in flight
    // (weights from HBM): 32,768 x 2816 (98 MB) 22.9 against 24.8, x 3072 (107
    // MB) 24.1 against 40.5, 40,000 x 3072 31.6 against 44.0.
    const bool large = staged && a.rows >= rb_max * 8 * num_cus &&
                       (a.rows * nb * kQ8Bytes * NM > (512LL << 10) * num_cus || nb > 80);
    // The other two kernels read a quantized activation; a graph capture that
    // finds no workspace for one can allocate none, and takes this one.
    const size_t sbytes = ((size_t)nb * sizeof(float) + 255) / 256 * 256;
    if (!(large || q8_lane_per_row<kInt8, NM>(a.rows, nb, num_cus)) ||
        (!a.xs && ctx->ws.bytes < sbytes + (size_t)a.cols && capturing(stream))) {
        bool done = false;
        const int rc = launch_q8_once<EPI, kInt8>(ctx, a, stream, &done);
        if (rc != G4_OK || done) return rc;
    }
    if (!a.xs) {
        // An f32 activation for a kernel that reads a quantized one:
        // quantize_q8_0 into the context's workspace first.
        const int rc = ensure_workspace(ctx, sbytes + (size_t)a.cols, stream);
        if (rc != G4_OK) return rc;
        a.xs = (const float *)ctx->ws.ptr;
        a.xq = (const signed char *)ctx->ws.ptr + sbytes;
        const int rq = launch_quantize_q8_0(a.x, a.cols, (float *)a.xs, (signed char *)a.xq, stream);
        if (rq != G4_OK) return rq;
    }
    if (large) {
        // 8 rows per workgroup, staged two at a time, so that the workgroups
        // are small and many are resident per CU, each with two rows in
        // flight.  Output head (262,144 x 1536, quantize included): 75.5 us
        // with 16 rows staged one at a time, 71.5 with 8 (or 4) staged two at
        // a time, 87 with 8 staged eight at a time, 97-142 with 64 rows per
        // workgroup.
        const int rb = (int)std::min<int64_t>(8, rb_max), g = std::min(2, rb);
        switch ((nb + 63) / 64) {
        case 1: return launch_q8_rows<EPI, 1>(a, g, rb, stream);
        case 2: return launch_q8_rows<EPI, 2>(a, g, rb, stream);
        case 3: return launch_q8_rows<EPI, 3>(a, g, rb, stream);
        default: return launch_q8_rows<EPI, 4>(a, g, rb, stream);
        }
    }
    hipLaunchKernelGGL((matvec_q8_0_rowwise_kernel<EPI>), dim3((unsigned)((a.rows + 255) / 256)), dim3(256), 0,
                       stream, a.w, a.w2, a.rows, (int)nb, a.xs, (const int *)a.xq, a.arg, a.out);
    G4_HIP(hipGetLastError());
    return G4_OK;
}

template <int DOT>
int launch_q8_f32(g4_ctx *ctx, const MatvecArgs &a, hipStream_t stream) {
    if (!q8_lane_per_row<DOT, 1>(a.rows, a.cols / kQ8Values, ctx->num_cus)) {
        bool done = false;
        const int rc = launch_q8_once<kPlain, DOT>(ctx, a, stream, &done);
        if (rc != G4_OK || done) return rc;
    }
    hipLaunchKernelGGL(matvec_q8_0_f32_kernel<DOT == kF64>, dim3((unsigned)((a.rows + 255) / 256)), dim3(256), 0,
                       stream, a.w, a.rows, (int)(a.cols / kQ8Values), a.x, a.out);
    G4_HIP(hipGetLastError());
    return G4_OK;
}

template <typename W, int R, int P, bool VEC>
int launch_dense_rows(const MatvecArgs &a, hipStream_t stream) {
    constexpr int64_t kRows = (int64_t)R << 24;  // a launch holds fewer than 2^32 threads
    for (int64_t r0 = 0; r0 < a.rows; r0 += kRows) {
        const int64_t rows = std::min(kRows, a.rows - r0);
        hipLaunchKernelGGL((matvec_dense_kernel<W, R, P, VEC>), dim3((unsigned)((rows + R - 1) / R)), dim3(128), 0,
                           stream, (const W *)a.w + r0 * a.cols, rows, a.cols, a.x, a.out + r0);
        G4_HIP(hipGetLastError());
    }
    return G4_OK;
}

// Short rows take a lane each where the two-wavefront kernel, whose time does
// not fall with the columns below 256, would take longer, and the whole matrix
// is small enough that the lanes' scattered reads hit a cache.  Measured (us,
// lane per row / two wavefronts): bf16 off the 16-byte loads 2048 x 7 4 / 5,
// 8192 x 33 5 / 6, 16,384 x 33 5 / 8, 32,768 x 50 7 / 12, 100,000 x 50 16 / 27, 200,000
// x 33 18 / 51, 50,000 x 100 17 / 18; with them 16,384 x 32 6 / 5, 32,768 x 32 6 /
// 8, 262,144 x 32 18 / 38; f32 off them 32,768 x 50 8 / 9, 100,000 x 50 (20 MB) 22
// / 20, 200,000 x 39 (31 MB) 46 / 42; with them 500,000 x 32 (64 MB) 257 / 73.
template <typename W>
bool dense_lane_per_row(const MatvecArgs &a, bool vec, int64_t num_cus) {
    const int64_t per_cu = a.rows / num_cus;
    if (a.cols <= 0 || a.rows > (1LL << 30) || a.rows * a.cols * (int64_t)sizeof(W) > (32LL << 20)) return false;
    if (a.cols <= 40) return per_cu >= (vec ? 128 : 64) || (!vec && a.cols <= 16);
    return !vec && a.cols <= 64 && per_cu >= 128 && a.rows * a.cols * (int64_t)sizeof(W) <= (16LL << 20);
}

// Rows per workgroup of the BF16 / F32 mat-vecs.  Up to eight rows per CU
// every wavefront has a SIMD of its own with 4 rows, and the shorter loads
// start the chain sooner (1024 x 1536 bf16: 6.6 us against 7.2 with 16).
// Beyond that the adding wavefronts share SIMDs, and an add costs the same
// for 4 rows as for 16 (8960 x 1536: 14.3 us with 4, 11.3 with 8, 9.9 with 16).
template <typename W>
int launch_dense(g4_ctx *ctx, const MatvecArgs &a, hipStream_t stream) {
    const bool vec = (uintptr_t)a.w % 4 == 0 && a.cols * sizeof(W) % 16 == 0 && a.cols < (1LL << 24);
    if (dense_lane_per_row<W>(a, vec, ctx->num_cus)) {
        hipLaunchKernelGGL(matvec_dense_narrow_kernel<W>, dim3((unsigned)((a.rows + 255) / 256)), dim3(256), 0, stream,
                           (const W *)a.w, a.rows, a.cols, a.x, a.out);
        G4_HIP(hipGetLastError());
        return G4_OK;
    }
    if (!vec) return launch_dense_rows<W, 4, 2, false>(a, stream);
    if (a.rows <= 8LL * ctx->num_cus) return launch_dense_rows<W, 4, 4, true>(a, stream);
    return launch_dense_rows<W, 16, 3, true>(a, stream);
}

}  // namespace

int launch_quantize_q8_0(const float *x, int64_t n, float *scales, signed char *quants, hipStream_t stream) {
    if (n <= 0) return G4_OK;
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, x, n, scales,
                       quants);
    G4_HIP(hipGetLastError());
    return G4_OK;
}

int launch_matvec(g4_ctx *ctx, const MatvecArgs &a, hipStream_t stream) {
    if (a.rows <= 0) return G4_OK;
    switch (a.kind) {
    case MatvecKind::Q8: return launch_q8<kPlain>(ctx, a, stream);
    case MatvecKind::Q8Softcap: return launch_q8<kSoftcap>(ctx, a, stream);
    case MatvecKind::Q8Geglu: return launch_q8<kGeglu>(ctx, a, stream);
    case MatvecKind::Q8GegluFp16: return launch_q8<kGegluFp16>(ctx, a, stream);
    case MatvecKind::Q8F32: return launch_q8_f32<kF32>(ctx, a, stream);
    case MatvecKind::Q8F64: return launch_q8_f32<kF64>(ctx, a, stream);
    case MatvecKind::Bf16: return launch_dense<unsigned short>(ctx, a, stream);
    case MatvecKind::F32: return launch_dense<float>(ctx, a, stream);
    }
    return G4_OK;
}

}  // namespace g4
