// Prefill: quantised-weight GEMM  Y[M,N] = X[M,K] . W[N,K]^T  on the matrix cores (gfx950 MFMA).
//
// The reference has no such kernel: for M > 1 rows matmul_q runs M independent GEMVs
// (torch/io/gguf_model.h:7029-7036, :7056-7061), re-reading the weights M times.  Two families:
//   * exact kernels (below): the GEMV's arithmetic per output row, each weight tile read once per 64 rows of X;
//   * a fast kernel (second half of this file): fp16 MFMA on weights dequantised in registers.
//
// Q4_K (reference row semantics: torch/io/cpu_quant_gemv.h:505-685)
//   rows of X are quantised to Q8 blocks of 32 (same rule as the GEMV), and for every 32-wide sub-block
//   v_mfma_i32_16x16x32_i8 produces the exact integer dots of a 16x16 (m x n) tile: K = 32 of the
//   instruction is exactly one sub-block, so each result is scaled on the VALU by
//   fma(d*sc*dx[m], isum, -(dmin*mn*sx[m])) and added to the even/odd sub-block chains in the
//   reference's order (the result is bit-identical to the reference's per-row GEMV).
//   4-bit weights are unpacked in registers (an 8-byte slice of qs gives the B fragments of the low-
//   and high-nibble sub-blocks), Q8 activations of a 64-row x 256-column chunk are staged in LDS.
// Q6_K (reference row semantics: cpu_quant_gemv.h:883-1020, fp32 activations)
//   v_mfma_f32_16x16x16_bf16: K = 16 is exactly one scale group of Q6_K.  (q - 32) is exact in bf16 and
//   X is bf16 by contract, so products are exact; each 16-group sum is scaled by d*scale[n] in fp32.
#include "gemm_tile.h"
#include "ptm_common.h"

#include <mutex>
#include <type_traits>

namespace ptm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));

enum { QG_NT = 2, QG_MT = 4, QG_MCHUNK = 16 * QG_MT, QG_NBLOCK = 4 * 16 * QG_NT, QG_PITCH8 = 256 + 8, QG_PITCH16 = 512 + 8 };

__device__ __forceinline__ float bf16_to_f32(uint32_t bits16) { return __uint_as_float(bits16 << 16); }
__host__ __device__ inline int qg_mpad(int M) { return (M + QG_MCHUNK - 1) / QG_MCHUNK * QG_MCHUNK; }

// ---- rows of X (bf16) -> Q8 blocks: qs[Mpad][K], dT[K/32][Mpad], sT[K/32][Mpad]; rows >= M are zero ----
__global__ __launch_bounds__(256) void qgemm_quantize_rows_kernel(const uint16_t* __restrict__ X, int8_t* __restrict__ qs,
                                                                  float* __restrict__ dT, float* __restrict__ sT, int M,
                                                                  int Mpad, int K) {
    const int m = blockIdx.x;
    const int n4 = K / 4;
    for (int i = threadIdx.x; i < n4; i += 256) {  // K % 256 == 0: whole waves stay together
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < M) {
            const uint2 raw = *reinterpret_cast<const uint2*>(X + (int64_t)m * K + 4 * i);
            v.x = bf16_to_f32(raw.x & 0xffffu);
            v.y = bf16_to_f32(raw.x >> 16);
            v.z = bf16_to_f32(raw.y & 0xffffu);
            v.w = bf16_to_f32(raw.y >> 16);
        }
        float d, s;
        const uint32_t packed = q8_quantize4(v, d, s);
        reinterpret_cast<uint32_t*>(qs + (int64_t)m * K)[i] = packed;
        if ((threadIdx.x & 7) == 0) {
            dT[(int64_t)(i >> 3) * Mpad + m] = d;
            sT[(int64_t)(i >> 3) * Mpad + m] = s;
        }
    }
}

// ---- Q4_K x Q8 on int8 MFMA ----------------------------------------------------------------------
// grid (ceil(N/128), Mpad/64), 256 threads; wave w owns columns [128*bx + 32*w, +32) as two 16-wide tiles.
__global__ __launch_bounds__(256) void qgemm_q4k_kernel(const uint8_t* __restrict__ W, int64_t stride,
                                                        const int8_t* __restrict__ qs, const float* __restrict__ dT,
                                                        const float* __restrict__ sT, float* __restrict__ Y, int M,
                                                        int Mpad, int K, int N) {
    __shared__ __align__(16) uint8_t s_x[QG_MCHUNK * QG_PITCH8];
    __shared__ __align__(16) float s_d[8][QG_MCHUNK];
    __shared__ __align__(16) float s_s[8][QG_MCHUNK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, kq = lane >> 4;  // MFMA: lane = (row or column) + 16 * (k / 8)
    const int m0 = blockIdx.y * QG_MCHUNK;
    const int nblk = K / 256;
    int ncol[QG_NT];
    const uint8_t* wrow[QG_NT];
#pragma unroll
    for (int t = 0; t < QG_NT; ++t) {
        ncol[t] = blockIdx.x * QG_NBLOCK + wave * (16 * QG_NT) + 16 * t + col;
        wrow[t] = W + (int64_t)min(ncol[t], N - 1) * stride;
    }
    float acc_a[QG_NT][QG_MT][4], acc_b[QG_NT][QG_MT][4];
#pragma unroll
    for (int t = 0; t < QG_NT; ++t)
#pragma unroll
        for (int mt = 0; mt < QG_MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc_a[t][mt][r] = acc_b[t][mt][r] = 0.0f;

    for (int b = 0; b < nblk; ++b) {
        // weights of this super-block for the lane's two columns
        uint4 hdr[QG_NT];
        uint2 raw[QG_NT][4];
#pragma unroll
        for (int t = 0; t < QG_NT; ++t) {
            const uint8_t* p = wrow[t] + (int64_t)b * 144;
            hdr[t] = *reinterpret_cast<const uint4*>(p);
#pragma unroll
            for (int g = 0; g < 4; ++g) raw[t][g] = *reinterpret_cast<const uint2*>(p + 16 + 32 * g + 8 * kq);
        }
        __syncthreads();  // previous chunk fully consumed
        // Q8 activations of rows [m0, m0+64), columns [256b, 256b+256): 64 x 256 B, 16 B per thread x 4
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            const int row = (tid >> 4) + 16 * it, cb = (tid & 15) * 16;
            *reinterpret_cast<uint4*>(s_x + row * QG_PITCH8 + cb) =
                *reinterpret_cast<const uint4*>(qs + (int64_t)(m0 + row) * K + b * 256 + cb);
        }
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int e = tid + 256 * it, sb = e >> 6, m = e & 63;
            s_d[sb][m] = dT[(int64_t)(b * 8 + sb) * Mpad + m0 + m];
            s_s[sb][m] = sT[(int64_t)(b * 8 + sb) * Mpad + m0 + m];
        }
        __syncthreads();

        float dsc[QG_NT][8], dmn[QG_NT][8];
#pragma unroll
        for (int t = 0; t < QG_NT; ++t) {
            const float d = h2f(hdr[t].x), dmin = h2f(hdr[t].x >> 16);
#pragma unroll
            for (int sb = 0; sb < 8; ++sb) {
                int sc, mn;
                q4k_scale_min(hdr[t].y, hdr[t].z, hdr[t].w, sb, sc, mn);
                dsc[t][sb] = d * (float)sc;
                dmn[t][sb] = dmin * (float)mn;
            }
        }
#pragma unroll
        for (int sb = 0; sb < 8; ++sb) {
            const int g = sb >> 1;
            long bfrag[QG_NT];
#pragma unroll
            for (int t = 0; t < QG_NT; ++t) {
                const uint32_t lo = (sb & 1) ? ((raw[t][g].x >> 4) & 0x0f0f0f0fu) : (raw[t][g].x & 0x0f0f0f0fu);
                const uint32_t hi = (sb & 1) ? ((raw[t][g].y >> 4) & 0x0f0f0f0fu) : (raw[t][g].y & 0x0f0f0f0fu);
                bfrag[t] = (long)(((uint64_t)hi << 32) | lo);
            }
#pragma unroll
            for (int mt = 0; mt < QG_MT; ++mt) {
                const long afrag = *reinterpret_cast<const long*>(s_x + (mt * 16 + col) * QG_PITCH8 + sb * 32 + 8 * kq);
                const float4 dx = *reinterpret_cast<const float4*>(&s_d[sb][mt * 16 + 4 * kq]);
                const float4 sx = *reinterpret_cast<const float4*>(&s_s[sb][mt * 16 + 4 * kq]);
                const float dxr[4] = {dx.x, dx.y, dx.z, dx.w}, sxr[4] = {sx.x, sx.y, sx.z, sx.w};
#pragma unroll
                for (int t = 0; t < QG_NT; ++t) {
                    const v4i zero = {0, 0, 0, 0};
                    const v4i c = __builtin_amdgcn_mfma_i32_16x16x32_i8(afrag, bfrag[t], zero, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float w = dsc[t][sb] * dxr[r];
                        const float cm = dmn[t][sb] * sxr[r];
                        const float term = fmaf(w, (float)c[r], -cm);
                        if (sb & 1) acc_b[t][mt][r] += term;
                        else acc_a[t][mt][r] += term;
                    }
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < QG_NT; ++t)
#pragma unroll
        for (int mt = 0; mt < QG_MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + mt * 16 + 4 * kq + r;
                if (m < M && ncol[t] < N) Y[(int64_t)m * N + ncol[t]] = acc_a[t][mt][r] + acc_b[t][mt][r];
            }
}

// ---- Q6_K x bf16 on bf16 MFMA --------------------------------------------------------------------
__device__ __forceinline__ uint32_t ld_u32_a2(const uint8_t* p) {
    struct __attribute__((packed, aligned(2))) u32a2 { uint32_t v; };
    return reinterpret_cast<const u32a2*>(p)->v;
}
// two (q - 32) values (bytes b0, b1 of q in 0..63) as a packed pair of bf16
__device__ __forceinline__ uint32_t q_pair_bf16(uint32_t b0, uint32_t b1) {
    const float f0 = (float)(int)b0 - 32.0f, f1 = (float)(int)b1 - 32.0f;
    return (__float_as_uint(f0) >> 16) | (__float_as_uint(f1) & 0xffff0000u);
}

__global__ __launch_bounds__(256) void qgemm_q6k_kernel(const uint8_t* __restrict__ W, int64_t stride,
                                                        const uint16_t* __restrict__ X, float* __restrict__ Y, int M,
                                                        int K, int N) {
    __shared__ __align__(16) uint8_t s_x[QG_MCHUNK * QG_PITCH16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 15, kq = lane >> 4;  // MFMA 16x16x16: lane = (row or column) + 16 * (k / 4)
    const int m0 = blockIdx.y * QG_MCHUNK;
    const int nblk = K / 256;
    int ncol[QG_NT];
    const uint8_t* wrow[QG_NT];
#pragma unroll
    for (int t = 0; t < QG_NT; ++t) {
        ncol[t] = blockIdx.x * QG_NBLOCK + wave * (16 * QG_NT) + 16 * t + col;
        wrow[t] = W + (int64_t)min(ncol[t], N - 1) * stride;
    }
    float acc[QG_NT][QG_MT][4];
#pragma unroll
    for (int t = 0; t < QG_NT; ++t)
#pragma unroll
        for (int mt = 0; mt < QG_MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][mt][r] = 0.0f;

    for (int b = 0; b < nblk; ++b) {
        // B fragments: for scale group s (16 weights) the lane holds elements 16s + 4kq + {0..3} of column n
        v4s bfrag[QG_NT][16];
        float fsc[QG_NT][16];
#pragma unroll
        for (int t = 0; t < QG_NT; ++t) {
            const uint8_t* p = wrow[t] + (int64_t)b * 210;
            const float d = h2f(reinterpret_cast<const u16_a2*>(p + 208)->v);
#pragma unroll
            for (int s = 0; s < 16; ++s) {
                const int e = 16 * s + 4 * kq;  // first of the lane's four consecutive elements
                const int half = e >> 7, r = e & 127, grp = r >> 5, l5 = r & 31;
                const uint32_t ql = ld_u32_a2(p + 64 * half + 32 * (grp & 1) + l5);
                const uint32_t qh = ld_u32_a2(p + 128 + 32 * half + l5);
                const uint32_t q4 = (ql >> (4 * (grp >> 1))) & 0x0f0f0f0fu;
                const uint32_t q = q4 | (((qh >> (2 * grp)) & 0x03030303u) << 4);
                const uint32_t p01 = q_pair_bf16(q & 0xffu, (q >> 8) & 0xffu);
                const uint32_t p23 = q_pair_bf16((q >> 16) & 0xffu, q >> 24);
                v4s f;
                f[0] = (short)(p01 & 0xffffu); f[1] = (short)(p01 >> 16);
                f[2] = (short)(p23 & 0xffffu); f[3] = (short)(p23 >> 16);
                bfrag[t][s] = f;
                // scale index of element e: 8*half + 2*grp + l5/16
                fsc[t][s] = d * (float)(int)(int8_t)p[192 + 8 * half + 2 * grp + (l5 >> 4)];
            }
        }
        __syncthreads();
        // bf16 activations of rows [m0, m0+64), columns [256b, +256): 64 x 512 B, 16 B per thread x 8
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int row = (tid >> 5) + 8 * it, cb = (tid & 31) * 16;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (m0 + row < M) v = *reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(X) + ((int64_t)(m0 + row) * K + b * 256) * 2 + cb);
            *reinterpret_cast<uint4*>(s_x + row * QG_PITCH16 + cb) = v;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < 16; ++s) {
#pragma unroll
            for (int mt = 0; mt < QG_MT; ++mt) {
                const v4s afrag = *reinterpret_cast<const v4s*>(s_x + (mt * 16 + col) * QG_PITCH16 + (16 * s + 4 * kq) * 2);
#pragma unroll
                for (int t = 0; t < QG_NT; ++t) {
                    const v4f zero = {0.f, 0.f, 0.f, 0.f};
                    const v4f c = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(afrag, bfrag[t][s], zero, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[t][mt][r] = fmaf(fsc[t][s], c[r], acc[t][mt][r]);
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < QG_NT; ++t)
#pragma unroll
        for (int mt = 0; mt < QG_MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = m0 + mt * 16 + 4 * kq + r;
                if (m < M && ncol[t] < N) Y[(int64_t)m * N + ncol[t]] = acc[t][mt][r];
            }
}

// =================================================================================================
// Fast path: fp16 MFMA on dequantised weights.
//   Activations: each row of X is rounded to the reference's Q8 values (d * q per block of 32, the rounding the
//   CPU GEMV applies) and stored as fp16, scaled by a power of two per row so that it cannot overflow.
//   Weights: dequantised in registers to their exact fp32 value, then rounded to fp16 (round toward zero, one
//   instruction per pair).  v_mfma_f32_32x32x16_f16 accumulates in fp32 over the whole K, so there is NO per-sub-
//   block epilogue: VALU work is the dequantisation only, and it is amortised over the 128 rows of X a workgroup
//   owns.  Result = reference GEMV up to fp16 rounding of the operands (relative 2^-12 per element).
//   Workgroup: 32 to 256 rows of X x 256 (128) columns, a 32-column strip a wave; the rows of X are shared through LDS
//   (double-buffered) and each wave dequantises only its own columns.
//   The summation index of the MFMA is free to permute: lane half kh takes the 16 CONSECUTIVE elements
//   [16 kh, 16 kh + 16) of a 32-wide sub-block (first 8 in k-step 0, next 8 in k-step 1), for A and B alike, so a
//   lane's weights of one sub-block come from one 16-byte load.
// =================================================================================================
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// LDS holds the fp16 X tile of a whole super-block step: 128 rows x 256 k, row pitch 528 B (16 consecutive lanes
// x 16 B then hit all 64 banks once), double-buffered: 2 x 66 KB of the CU's 160 KB.
enum { QF_TM = 128, QF_TN = 256, QF_PITCH = 528 };
// LDS of a launch in tiles of 128, 192 and 256 rows: two X tiles and the row scales of 128 rows, which take more than those of 256 (qgemm_f16_tall_body)
enum { QF_ROWS_LDS = 2 * 128 * QF_PITCH + 4 * 128 };

__host__ __device__ inline int qf_mpad(int M) { return (M + QF_TM - 1) / QF_TM * QF_TM; }

// rows of X (bf16, or fp32 when XF32) -> fp16 rows Xh[Mpad][K] (Q8ROUND: first rounded to the reference's Q8 values d*q per block of
// 32, the rounding its Q4_K GEMV applies; otherwise the bf16 value itself, as its Q6_K GEMV uses), divided by a
// power of two per row (returned in rowscale) so that fp16 cannot overflow
template <bool XF32>
__device__ __forceinline__ float4 load_x4(const void* row, int i) {
    if constexpr (XF32) {
        return reinterpret_cast<const float4*>(row)[i];
    } else {
        const uint2 raw = reinterpret_cast<const uint2*>(row)[i];
        return make_float4(bf16_to_f32(raw.x & 0xffffu), bf16_to_f32(raw.x >> 16), bf16_to_f32(raw.y & 0xffffu),
                           bf16_to_f32(raw.y >> 16));
    }
}

template <bool Q8ROUND, bool XF32>
__global__ __launch_bounds__(256) void qgemm_prepare_rows_f16_kernel(const void* __restrict__ X, _Float16* __restrict__ Xh,
                                                                     float* __restrict__ rowscale, int M, int K) {
    __shared__ float red[4];
    const int m = blockIdx.x, tid = threadIdx.x;
    const int n4 = K / 4;
    _Float16* dst = Xh + (int64_t)m * K;
    if (m >= M) {  // padding rows: zeros
        for (int i = tid; i < n4; i += 256) reinterpret_cast<uint2*>(dst)[i] = make_uint2(0, 0);
        return;
    }
    const void* src = static_cast<const uint8_t*>(X) + (int64_t)m * K * (XF32 ? 4 : 2);
    float amax = 0.0f;
    for (int i = tid; i < n4; i += 256) {
        const float4 v = load_x4<XF32>(src, i);
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    amax = max64(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    // power of two that brings the row below 2^14 (fp16 tops out at 65504); 1 for ordinary activations
    int e = 0;
    if (amax > 16384.0f) { (void)frexpf(amax, &e); e -= 14; }
    const float down = ldexpf(1.0f, -e);
    if (tid == 0) rowscale[m] = ldexpf(1.0f, e);
    for (int i = tid; i < n4; i += 256) {  // K % 256 == 0: whole waves, aligned groups of 8 lanes = one Q8 block
        float4 v = load_x4<XF32>(src, i);
        if constexpr (Q8ROUND) {
            float d, sm;
            const uint32_t pk = q8_quantize4(v, d, sm);
            v.x = d * (float)(int)(int8_t)(pk & 0xff);
            v.y = d * (float)(int)(int8_t)((pk >> 8) & 0xff);
            v.z = d * (float)(int)(int8_t)((pk >> 16) & 0xff);
            v.w = d * (float)(int)(int8_t)(pk >> 24);
        }
        union { _Float16 h[4]; uint2 u; } o;
        o.h[0] = (_Float16)(v.x * down);  // power-of-two scaling: exact
        o.h[1] = (_Float16)(v.y * down);
        o.h[2] = (_Float16)(v.z * down);
        o.h[3] = (_Float16)(v.w * down);
        reinterpret_cast<uint2*>(dst)[i] = o.u;
    }
}

// silu(g) u and gelu(g) u in the arithmetic of silu_mul_kernel and gelu_mul_kernel
__device__ __forceinline__ float silu_mul(float g, float u) {
    float ng = 0.0f - g;
    ng = fminf(fmaxf(ng, -88.0f), 88.0f);
    return (g * (1.0f / (1.0f + expf(ng)))) * u;
}
__device__ __forceinline__ float gelu_mul(float g, float u) {
    const float x3 = g * g * g;
    const float t = tanhf(0.7978845608028654f * (g + 0.044715f * x3));
    return 0.5f * g * (1.0f + t) * u;
}

// The same conversion fused with what precedes a projection in the prompt pass, so that the fp32 intermediate is never
// written: PRE 1 = RMSNorm of the row (x * rs * (gamma + add_one), the arithmetic and reduction order of
// rms_norm_kernel), PRE 2 = SiLU(gate) * up (the arithmetic of silu_mul_kernel), or tanh-GELU(gate) * up (that of
// gelu_mul_kernel) when add_one, which has no other meaning for PRE 2, is set.  Writes the Q8-rounded form (for Q4_K
// matrices) and / or the plain form (for Q6_K matrices) in one pass; either output may be NULL.
// PRE 2 has 1024 threads per row (256: 512 rows of 9728 16.9 us, 12.8 so; 2048 of 14336 69 -> 57, 252 MB), PRE 1 the 256 whose order
// the RMSNorm's sum has.
template <int PRE, int THREADS = PRE == 2 ? 1024 : 256>
__global__ __launch_bounds__(THREADS) void qgemm_prepare_fused_kernel(const float* __restrict__ X, const float* __restrict__ X2,
                                                                  float eps, int add_one, _Float16* __restrict__ Xh_round,
                                                                  float* __restrict__ rs_round, _Float16* __restrict__ Xh_plain,
                                                                  float* __restrict__ rs_plain, int M, int K) {
    static_assert(PRE == 2 || THREADS == 256, "the RMSNorm sum keeps the 256-thread reduction order");
    __shared__ float red[4];
    __shared__ float red2[THREADS / 64];
    const int m = blockIdx.x, tid = threadIdx.x;
    const int n4 = K / 4;
    if (m >= M) {  // padding rows: zeros
        for (int i = tid; i < n4; i += THREADS) {
            if (Xh_round) reinterpret_cast<uint2*>(Xh_round + (int64_t)m * K)[i] = make_uint2(0, 0);
            if (Xh_plain) reinterpret_cast<uint2*>(Xh_plain + (int64_t)m * K)[i] = make_uint2(0, 0);
        }
        return;
    }
    const float* x = X + (int64_t)m * K;
    const float* x2 = PRE == 2 ? X2 + (int64_t)m * K : X2;
    float rs = 1.0f;
    const float one = add_one ? 1.0f : 0.0f;
    if constexpr (PRE == 1) {
        float ss = 0.0f;
        for (int i = tid; i < K; i += THREADS) ss = fmaf(x[i], x[i], ss);
        ss = block_sum256(ss, red);
        rs = 1.0f / sqrtf(ss / (float)K + eps);
    }
    const bool gelu = PRE == 2 && add_one != 0;
    auto value = [&](float4 a, float4 b) {
        float4 r;
        if constexpr (PRE == 1) {
            r.x = a.x * rs * (b.x + one); r.y = a.y * rs * (b.y + one); r.z = a.z * rs * (b.z + one); r.w = a.w * rs * (b.w + one);
        } else {
            if (gelu) { r.x = gelu_mul(a.x, b.x); r.y = gelu_mul(a.y, b.y); r.z = gelu_mul(a.z, b.z); r.w = gelu_mul(a.w, b.w); }
            else { r.x = silu_mul(a.x, b.x); r.y = silu_mul(a.y, b.y); r.z = silu_mul(a.z, b.z); r.w = silu_mul(a.w, b.w); }
        }
        return r;
    };
    auto value4 = [&](int i) { return value(reinterpret_cast<const float4*>(x)[i], reinterpret_cast<const float4*>(x2)[i]); };
    // Rows of up to 16384 values are computed once and kept in registers between the maximum and the store pass: all of a
    // thread's loads go out together, and the exponentials of PRE 2 are paid once (the pass is otherwise two dependent
    // sweeps over 2 x 4 K bytes per row).
    constexpr int HOLD = 4096 / THREADS;
    const bool held = n4 <= HOLD * THREADS;
    float4 hv[HOLD];
    float amax = 0.0f;
    if (held) {
        float4 hx[HOLD];
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {  // the loads go out together
            const int i = tid + THREADS * u;
            hv[u] = hx[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < n4) {
                hv[u] = reinterpret_cast<const float4*>(x)[i];
                hx[u] = reinterpret_cast<const float4*>(x2)[i];
            }
        }
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            hv[u] = tid + THREADS * u < n4 ? value(hv[u], hx[u]) : make_float4(0.f, 0.f, 0.f, 0.f);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(hv[u].x), fabsf(hv[u].y)), fmaxf(fabsf(hv[u].z), fabsf(hv[u].w))));
        }
    } else {
        for (int i = tid; i < n4; i += THREADS) {
            const float4 v = value4(i);
            amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    }
    amax = max64(amax);
    if ((tid & 63) == 0) red2[tid >> 6] = amax;
    __syncthreads();
    {
        float t = red2[0];
#pragma unroll
        for (int w = 1; w < THREADS / 64; ++w) t = fmaxf(t, red2[w]);
        amax = t;
    }
    int e = 0;
    if (amax > 16384.0f) { (void)frexpf(amax, &e); e -= 14; }
    const float down = ldexpf(1.0f, -e);
    if (tid == 0) {
        if (rs_round) rs_round[m] = ldexpf(1.0f, e);
        if (rs_plain) rs_plain[m] = ldexpf(1.0f, e);
    }
    auto store4 = [&](_Float16* dst, int i, float4 v) {
        union { _Float16 h[4]; uint2 u; } o;
        o.h[0] = (_Float16)(v.x * down);
        o.h[1] = (_Float16)(v.y * down);
        o.h[2] = (_Float16)(v.z * down);
        o.h[3] = (_Float16)(v.w * down);
        reinterpret_cast<uint2*>(dst)[i] = o.u;
    };
    auto emit4 = [&](int i, float4 v) {  // K % 256 == 0: whole waves, aligned groups of 8 lanes = one Q8 block
        if (Xh_plain) store4(Xh_plain + (int64_t)m * K, i, v);
        if (Xh_round) {
            float d, sm;
            const uint32_t pk = q8_quantize4(v, d, sm);
            float4 q;
            q.x = d * (float)(int)(int8_t)(pk & 0xff);
            q.y = d * (float)(int)(int8_t)((pk >> 8) & 0xff);
            q.z = d * (float)(int)(int8_t)((pk >> 16) & 0xff);
            q.w = d * (float)(int)(int8_t)(pk >> 24);
            store4(Xh_round + (int64_t)m * K, i, q);
        }
    };
    if (held) {
#pragma unroll
        for (int u = 0; u < HOLD; ++u) {
            const int i = tid + THREADS * u;
            if (i < n4) emit4(i, hv[u]);  // wave-uniform: n4 is a multiple of 64
        }
    } else {
        for (int i = tid; i < n4; i += THREADS) emit4(i, value4(i));
    }
}

// The K-split partial sums of a projection into the residual stream, folded into the conversion that follows it:
// X[m] (+)= P[0][m] + P[1][m] + ... (the order of qgemm_split_reduce_kernel), then RMSNorm of the new row and its fp16
// forms as qgemm_prepare_fused_kernel<1> produces them (same arithmetic, same reduction order: the row is staged in LDS
// and walked with that kernel's two lane mappings).  One launch and one pass over the row instead of a reduction launch
// and three sweeps of the conversion.
template <int B, int THREADS>  // partial sums fetched per batch
__global__ __launch_bounds__(THREADS) void qgemm_reduce_norm_prepare_kernel(const float* __restrict__ P, int splits, float* __restrict__ X,
                                                                        int accumulate, const float* __restrict__ gamma, float eps,
                                                                        int add_one, _Float16* __restrict__ Xh_round,
                                                                        float* __restrict__ rs_round, _Float16* __restrict__ Xh_plain,
                                                                        float* __restrict__ rs_plain, int M, int K) {
    extern __shared__ __align__(16) float rn_row[];  // K floats
    __shared__ float red[4];
    __shared__ float red2[THREADS / 64];
    const int m = blockIdx.x, tid = threadIdx.x;
    const int n4 = K / 4;
    // the norm weights of a thread's first two pieces go out with the slabs: behind the sums they were a round trip of their own (2048 rows of 4096,
    // two slabs, 29.2 -> 26.8 us; 19 rows in 72 launches of a prompt 2830 -> 2811)
    float4 g[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) g[u] = reinterpret_cast<const float4*>(gamma)[min(tid + THREADS * u, n4 - 1)];
    issue_order_fence();
    const int64_t total = (int64_t)M * K;
    float4* x4 = reinterpret_cast<float4*>(X + (int64_t)m * K);
    for (int i = tid; i < n4; i += THREADS) {
        // B partial sums per batch, fetched unconditionally (the index clamped) so that they are in flight together; B = 4
        // where there are at most four slabs (half the clamped re-reads of the last one)
        const float4 o = accumulate ? x4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int z0 = 0; z0 < splits; z0 += B) {
            float4 b[B];
#pragma unroll
            for (int u = 0; u < B; ++u) b[u] = reinterpret_cast<const float4*>(P + min(z0 + u, splits - 1) * total + (int64_t)m * K)[i];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (z0 + u == 0) a = b[u];
                else if (z0 + u < splits) { a.x += b[u].x; a.y += b[u].y; a.z += b[u].z; a.w += b[u].w; }
            }
        }
        if (accumulate) { a.x += o.x; a.y += o.y; a.z += o.z; a.w += o.w; }
        x4[i] = a;
        reinterpret_cast<float4*>(rn_row)[i] = a;
    }
    __syncthreads();
    // the order of 256 threads whatever their number
    float ss = 0.0f;
    if (tid < 256) {
        for (int i = tid; i < K; i += 256) ss = fmaf(rn_row[i], rn_row[i], ss);
        ss = sum64(ss);
        if ((tid & 63) == 0) red[tid >> 6] = ss;
    }
    __syncthreads();
    ss = (red[0] + red[1]) + (red[2] + red[3]);
    const float rs = 1.0f / sqrtf(ss / (float)K + eps);
    const float one = add_one ? 1.0f : 0.0f;
    auto value4 = [&](int i, const float4& b) {
        const float4 a = reinterpret_cast<const float4*>(rn_row)[i];
        float4 r;
        r.x = a.x * rs * (b.x + one); r.y = a.y * rs * (b.y + one); r.z = a.z * rs * (b.z + one); r.w = a.w * rs * (b.w + one);
        return r;
    };
    // every piece of a thread: the two whose weights are here, then the rest
    auto pieces = [&](auto take) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (tid + THREADS * u < n4) take(tid + THREADS * u, value4(tid + THREADS * u, g[u]));
        for (int i = tid + 2 * THREADS; i < n4; i += THREADS) take(i, value4(i, reinterpret_cast<const float4*>(gamma)[i]));
    };
    float amax = 0.0f;
    pieces([&](int, const float4& v) {
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    });
    amax = max64(amax);
    if ((tid & 63) == 0) red2[tid >> 6] = amax;
    __syncthreads();
    amax = red2[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) amax = fmaxf(amax, red2[w]);
    int e = 0;
    if (amax > 16384.0f) { (void)frexpf(amax, &e); e -= 14; }
    const float down = ldexpf(1.0f, -e);
    if (tid == 0) {
        if (rs_round) rs_round[m] = ldexpf(1.0f, e);
        if (rs_plain) rs_plain[m] = ldexpf(1.0f, e);
    }
    auto store4 = [&](_Float16* dst, int i, float4 v) {
        union { _Float16 h[4]; uint2 u; } o;
        o.h[0] = (_Float16)(v.x * down);
        o.h[1] = (_Float16)(v.y * down);
        o.h[2] = (_Float16)(v.z * down);
        o.h[3] = (_Float16)(v.w * down);
        reinterpret_cast<uint2*>(dst)[i] = o.u;
    };
    pieces([&](int i, const float4& v) {  // K % 256 == 0: whole waves, aligned groups of 8 lanes = one Q8 block
        if (Xh_plain) store4(Xh_plain + (int64_t)m * K, i, v);
        if (Xh_round) {
            float d, sm;
            const uint32_t pk = q8_quantize4(v, d, sm);
            float4 q;
            q.x = d * (float)(int)(int8_t)(pk & 0xff);
            q.y = d * (float)(int)(int8_t)((pk >> 8) & 0xff);
            q.z = d * (float)(int)(int8_t)((pk >> 16) & 0xff);
            q.w = d * (float)(int)(int8_t)(pk >> 24);
            store4(Xh_round + (int64_t)m * K, i, q);
        }
    });
}

// SiLU(gate) . up (gelu: tanh-GELU) of a short prompt's rows, gate and up still `sg` / `su` slabs of K splits each, into the fp16 rows of the down
// projection (rounded: to Q8 blocks first).  A workgroup has `chunk` values of a row, those of one K split of that projection, and they have
// a scale of their own at rowscale[split * scale_stride + row]: nothing needs the whole row, which one workgroup a row had to
// walk (19 rows: 19 CUs, behind a launch that summed the slabs on all).  What bounds it is one round trip for the slabs: 19 rows of 9728, three
// slabs each, 4.1 us (the two launches 4.0 + 5.8).
constexpr int ACT_CHUNK = 4096;  // values a workgroup holds
__global__ __launch_bounds__(256) void qgemm_act_rows_kernel(const float* __restrict__ G, const float* __restrict__ U, int sg, int su, int gelu,
                                                             int rounded, _Float16* __restrict__ Xh, float* __restrict__ rowscale,
                                                             int scale_stride, int chunk, int M, int K) {
    read_now(G, Xh, K);
    __shared__ float red[4];
    const int m = blockIdx.y, split = blockIdx.x, tid = threadIdx.x;
    const int first = split * chunk, n4 = min(chunk, K - first) / 4;  // both multiples of 256
    const int64_t total = (int64_t)M * K, at = (int64_t)m * K + first;
    constexpr int HOLD = ACT_CHUNK / 1024, B = 4;
    auto sum = [&](const float* P, int slabs, int i) {
        float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int z0 = 0; z0 < slabs; z0 += B) {
            float4 b[B];
#pragma unroll
            for (int u = 0; u < B; ++u) b[u] = reinterpret_cast<const float4*>(P + min(z0 + u, slabs - 1) * total + at)[i];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (z0 + u == 0) a = b[u];
                else if (z0 + u < slabs) { a.x += b[u].x; a.y += b[u].y; a.z += b[u].z; a.w += b[u].w; }
            }
        }
        return a;
    };
    float4 v[HOLD];
    float amax = 0.0f;
#pragma unroll
    for (int h = 0; h < HOLD; ++h) {
        const int i = tid + 256 * h;
        v[h] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < n4) {  // whole waves: n4 is a multiple of 64
            const float4 g = sum(G, sg, i), u = sum(U, su, i);
            if (gelu) v[h] = make_float4(gelu_mul(g.x, u.x), gelu_mul(g.y, u.y), gelu_mul(g.z, u.z), gelu_mul(g.w, u.w));
            else v[h] = make_float4(silu_mul(g.x, u.x), silu_mul(g.y, u.y), silu_mul(g.z, u.z), silu_mul(g.w, u.w));
        }
        amax = fmaxf(amax, fmaxf(fmaxf(fabsf(v[h].x), fabsf(v[h].y)), fmaxf(fabsf(v[h].z), fabsf(v[h].w))));
    }
    amax = max64(amax);
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    int e = 0;
    if (amax > 16384.0f) { (void)frexpf(amax, &e); e -= 14; }
    const float down = ldexpf(1.0f, -e);
    if (tid == 0) rowscale[split * scale_stride + m] = ldexpf(1.0f, e);
#pragma unroll
    for (int h = 0; h < HOLD; ++h) {
        const int i = tid + 256 * h;
        if (i >= n4) break;
        float4 q = v[h];
        if (rounded) {
            float d, sm;
            const uint32_t pk = q8_quantize4(q, d, sm);
            q = make_float4(d * (float)(int)(int8_t)(pk & 0xff), d * (float)(int)(int8_t)((pk >> 8) & 0xff), d * (float)(int)(int8_t)((pk >> 16) & 0xff),
                            d * (float)(int)(int8_t)(pk >> 24));
        }
        union { _Float16 h4[4]; uint2 u2; } o;
        o.h4[0] = (_Float16)(q.x * down);
        o.h4[1] = (_Float16)(q.y * down);
        o.h4[2] = (_Float16)(q.z * down);
        o.h4[3] = (_Float16)(q.w * down);
        reinterpret_cast<uint2*>(Xh + at)[i] = o.u2;
    }
}

// 16 small integers (4 dwords of bytes, each < 1024) -> two fragments of 8 fp16 holding (byte - bias) * scale + offset.
// A byte b becomes the fp16 number 1024 + b by writing it under the exponent byte 0x64 (one v_perm per pair); the
// subtraction of 1024 + bias is exact, and one packed fp16 FMA applies scale and offset: 2.5 instructions per pair.
__device__ __forceinline__ void bytes_to_frags(const uint32_t (&b)[4], float bias, float scale, float offset, h8& f0, h8& f1) {
    const h2 sub = {(_Float16)(1024.0f + bias), (_Float16)(1024.0f + bias)};
    const h2 sc = {(_Float16)scale, (_Float16)scale};
    const h2 of = {(_Float16)offset, (_Float16)offset};
    uint32_t o[8];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t hq = __builtin_amdgcn_perm(0x64646464u, b[w], p ? 0x04030402u : 0x04010400u);
            h2 q;
            __builtin_memcpy(&q, &hq, 4);
            const h2 v = __builtin_elementwise_fma(q - sub, sc, of);
            __builtin_memcpy(&o[2 * w + p], &v, 4);
        }
    }
    __builtin_memcpy(&f0, &o[0], 16);
    __builtin_memcpy(&f1, &o[4], 16);
}

__device__ __forceinline__ void pin4(uint4& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z), "+v"(v.w)); }

// ---- per-type weight access: what a lane (column n, element half kh) fetches of a 256-wide super-block ----
struct Q4Half;
struct Q6Half;
struct Q4Tile {  // Q4_K: header + the lane's 16 bytes of each of the 4 groups of 64
    uint4 hdr;
    uint4 qs[4];
    __device__ __forceinline__ void load(const uint8_t* blk, int kh) {
        hdr = *reinterpret_cast<const uint4*>(blk);
#pragma unroll
        for (int g = 0; g < 4; ++g) qs[g] = *reinterpret_cast<const uint4*>(blk + 16 + 32 * g + 16 * kh);
    }
    // sub-block s (0..7) of the block -> two fragments
    __device__ __forceinline__ void frags(int s, int /*kh*/, h8& f0, h8& f1) const {
        int sc, mn;
        q4k_scale_min(hdr.y, hdr.z, hdr.w, s, sc, mn);
        const float dsc = h2f(hdr.x) * (float)sc, dmn = h2f(hdr.x >> 16) * (float)mn;
        const uint4 r = qs[s >> 1];
        const int sh = 4 * (s & 1);
        const uint32_t b[4] = {(r.x >> sh) & 0x0f0f0f0fu, (r.y >> sh) & 0x0f0f0f0fu, (r.z >> sh) & 0x0f0f0f0fu,
                               (r.w >> sh) & 0x0f0f0f0fu};
        bytes_to_frags(b, 0.0f, dsc, -dmn, f0, f1);  // (d*sc)*q - dmin*m, the dequantised value (gguf_dequant.h:304-341)
    }
    // Nothing computed from these registers may be scheduled above this point: without it the scheduler fills the vector
    // slots behind the first MFMAs of a block with the scale arithmetic of the block that was requested an instant
    // before, and every block starts with a wait for its successor's weights.
    __device__ __forceinline__ void pin() {
        pin4(hdr);
#pragma unroll
        for (int g = 0; g < 4; ++g) pin4(qs[g]);
    }
    static constexpr int kBlockBytes = 144;
    static constexpr bool kQ8Round = true;
    typedef Q4Half Half;
};
struct Q6Tile {  // Q6_K: the lane's 16 bytes of ql for each (half, pair), of qh for each half, scales, d
    uint4 ql[4], qh[2], sc;
    uint32_t d;
    __device__ __forceinline__ void load(const uint8_t* blk, int kh) {
#pragma unroll
        for (int c = 0; c < 4; ++c) ql[c] = ld16_a2(blk + 64 * (c >> 1) + 32 * (c & 1) + 16 * kh);
#pragma unroll
        for (int h = 0; h < 2; ++h) qh[h] = ld16_a2(blk + 128 + 32 * h + 16 * kh);
        sc = ld16_a2(blk + 192);
        d = reinterpret_cast<const u16_a2*>(blk + 208)->v;
    }
    // step s (0..7): elements 32 s + 16 kh + (0..15) = half s/4, group gq = s%4, one scale (index 2 s + kh)
    __device__ __forceinline__ void frags(int s, int kh, h8& f0, h8& f1) const {
        const int half = s >> 2, gq = s & 3;
        const uint4 l = ql[2 * half + (gq & 1)], hq = qh[half];
        const int lsh = 4 * (gq >> 1), hsh = 2 * gq;
        const uint32_t lw[4] = {l.x, l.y, l.z, l.w}, hw[4] = {hq.x, hq.y, hq.z, hq.w};
        uint32_t b[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) b[w] = ((lw[w] >> lsh) & 0x0f0f0f0fu) | ((((hw[w] >> hsh) & 0x03030303u)) << 4);
        const uint32_t scw[4] = {sc.x, sc.y, sc.z, sc.w};
        const uint32_t pair = scw[s >> 1] >> (16 * (s & 1));            // scales 2s and 2s+1
        const int sv = (int)(int8_t)((kh ? pair >> 8 : pair) & 0xffu);
        bytes_to_frags(b, 32.0f, h2f(d) * (float)sv, 0.0f, f0, f1);     // d*scale*(q-32) (gguf_dequant.h:395-430)
    }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int c = 0; c < 4; ++c) pin4(ql[c]);
        pin4(qh[0]); pin4(qh[1]); pin4(sc);
        asm volatile("" : "+v"(d));
    }
    static constexpr int kBlockBytes = 210;
    static constexpr bool kQ8Round = false;
    typedef Q6Half Half;
};

// Where a workgroup's accumulators go.
// C layout of the 32x32 tile: column j = lane % 32, rows 8 (r / 4) + 4 (lane / 32) + r % 4.  The row scales come from
// LDS (staged in the prologue) four at a time, and a value's place is the lane's first plus rows that are the same for the wave: 64-bit products
// per value, each behind its own read of a scale and its own branches, were 42 instructions and a wait where this has three (EDGE: six).
// ADD: the 16 old values of a tile are fetched together before its 16
// stores: a load issued behind a store the compiler cannot tell apart from it is one serial memory round trip per value,
// more than the main loop of a launch with few blocks per workgroup takes.
// p: the lane's column in row m0 + 4 kh, `left` rows from there on; rows: M < m0 + 32 MT or N within the workgroup's columns (EDGE).
// Few rows' sums are read by the next kernel from the caches, where plain stores leave them (19 rows of 36 layers 2823 -> 2749 us); many
// rows' pass by them (509 rows: 8353 us plain, 8248 so).
template <int MT, bool EDGE, bool ADD>
__device__ __forceinline__ void qf_store_rows(const f32x16 (&acc)[MT], const float* s_rs, float* p, int N, int left, bool n_ok, int kh) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        float4 sc[4];
        float old[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) sc[q] = *reinterpret_cast<const float4*>(s_rs + 32 * mt + 8 * q + 4 * kh);
        if constexpr (ADD) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 32 * mt + 8 * (r >> 2) + (r & 3);
                old[r] = p[(int64_t)(EDGE ? min(row, left - 1) : row) * N];
            }
            issue_order_fence();
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int row = 32 * mt + 8 * (r >> 2) + (r & 3);
            const float4 s4 = sc[r >> 2];
            float v = acc[mt][r] * ((r & 3) == 0 ? s4.x : (r & 3) == 1 ? s4.y : (r & 3) == 2 ? s4.z : s4.w);
            if constexpr (ADD) v = old[r] + v;
            if (!EDGE || (row < left && n_ok)) {
                if constexpr (MT == 1) p[(int64_t)row * N] = v;
                else __builtin_nontemporal_store(v, &p[(int64_t)row * N]);
            }
        }
    }
}
template <int MT>
__device__ __forceinline__ void qf_store(const f32x16 (&acc)[MT], const float* s_rs, float* Y, float* partials, int accumulate, int M, int N, int m0, int n_base,
                                         int j, int kh, int bz) {
    const int n = n_base + j, left = M - m0 - 4 * kh;
    float* p = (partials ? partials + (int64_t)bz * M * N : Y) + (int64_t)(m0 + 4 * kh) * N + min(n, N - 1);
    const bool add = !partials && accumulate, edge = MT == 1 || m0 + 32 * MT > M || __builtin_amdgcn_readfirstlane(n_base) + 32 > N;
    if (edge) {
        if (add) qf_store_rows<MT, true, true>(acc, s_rs, p, N, left, n < N, kh);
        else qf_store_rows<MT, true, false>(acc, s_rs, p, N, left, n < N, kh);
    } else {
        if (add) qf_store_rows<MT, false, true>(acc, s_rs, p, N, left, true, kh);
        else qf_store_rows<MT, false, false>(acc, s_rs, p, N, left, true, kh);
    }
}

// Up to 32 rows and up to four super-blocks of a K split: 128 columns, four waves of one strip.  Such a workgroup's time is its requests' round trips,
// one per block where the next block's are out while this one is worked on (half a microsecond's work).  Here all of its blocks, of X
// (into LDS) and of the weights (registers, up to 120), are requested before any is waited for.  Same sums in the same order.
// 19 rows, 2560 x 9728 in 13 splits of three: Q6_K 21.6 -> 16.6 us, Q4_K 12.4 -> 11.0; 2 x 9728 x 2560 in three of four 15.8 -> 15.2 (weights in memory order
// through LDS 17.1; eight waves, 256 columns 17.0).  Then its time is unpacking, behind the weights: 2 x 9728 x 2560 12.3 us without X and stores, 7.3 with one
// line of weights for all.  Up to two blocks three of them fit a SIMD: 36 layers of 19 rows 2749 -> 2728 us, most of it in q / k / v and o.
template <typename Tile, int NB>
__device__ __forceinline__ void qgemm_f16_short_body(const uint8_t* W, int64_t stride, const _Float16* Xh, const float* __restrict__ rowscale, float* Y, int M,
                                                     int K, int N, int accumulate, int blocks_per_split, float* partials, int bx, int bz, uint8_t* s_a,
                                                     int scale_stride) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 31, kh = lane >> 5;
    const int n_base = bx * 128 + wave * 32;
    const int blk0 = bz * blocks_per_split, nblk = min(K / 256 - blk0, blocks_per_split);
    const uint8_t* wrow = W + (int64_t)min(n_base + j, N - 1) * stride + (int64_t)blk0 * Tile::kBlockBytes;
    const uint8_t* x_src = reinterpret_cast<const uint8_t*>(Xh) + (int64_t)blk0 * 512 + 16 * (tid & 31);
    float* s_rs = reinterpret_cast<float*>(s_a + NB * 32 * QF_PITCH);
    // rows past the last repeat it: their sums are not stored
    u32x4 x[4 * NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int p = 0; p < 4; ++p)
            x[4 * b + p] = *reinterpret_cast<const u32x4*>(x_src + (int64_t)min((tid >> 5) + 8 * p, M - 1) * K * 2 + min(b, nblk - 1) * 512);
    issue_order_fence();
    Tile w[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) w[b].load(wrow + (int64_t)min(b, nblk - 1) * Tile::kBlockBytes, kh);
    issue_order_fence();
    if (tid < 32) s_rs[tid] = rowscale[bz * scale_stride + min(tid, M - 1)];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int p = 0; p < 4; ++p) *reinterpret_cast<u32x4*>(s_a + (b * 32 + (tid >> 5) + 8 * p) * QF_PITCH + 16 * (tid & 31)) = x[4 * b + p];
    __syncthreads();
    f32x16 acc[1];
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[0][r] = 0.0f;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (b >= nblk) break;  // workgroup-uniform
        w[b].pin();
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            h8 bf[2];
            w[b].frags(s, kh, bf[0], bf[1]);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const h8 af = *reinterpret_cast<const h8*>(s_a + (b * 32 + j) * QF_PITCH + 64 * s + 32 * kh + 16 * ks);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, bf[ks], acc[0], 0, 0, 0);
            }
        }
    }
    qf_store<1>(acc, s_rs, Y, partials, accumulate, M, N, 0, n_base, j, kh, bz);
}
// Whether it serves a launch whose longest split has `blocks`
constexpr int QF_SHORT_BLOCKS = 4;
static inline bool qf_short(int M, int blocks) { return M <= 32 && blocks <= QF_SHORT_BLOCKS; }
static inline size_t qf_short_lds(int nb) { return (size_t)nb * 32 * QF_PITCH + 4 * 32; }

// X tile of a super-block step in LDS.  The pieces a thread owns of the NEXT block's tile are fetched during the first
// steps of the current block, followed by the next block's weights, and written to the other LDS buffer during the
// later steps, so the block ends with the next tile complete behind the only workgroup barrier of the block.  (After the
// last block the same code re-fetches the last tile into the idle buffer: no conditionals in the steady-state loop.)
// WAVES = 8: waves w and w + 4 own one 32-column strip each of the same 64 columns and all MT row tiles, so a SIMD holds two waves
// and one's dequantisation and LDS reads run under the other's MFMAs (the two pipes of a single wave barely overlap); no weight is
// dequantised twice.  WAVES = 4, up to 64 rows: 128 columns, one strip a wave.  There a workgroup's time is unpacking and requests (64
// lanes are 64 rows of W), not MFMAs, and half as many columns on twice as many CUs halve it where 256 columns leave CUs idle.
// (bx, by, bz) = (column tile, row tile, K split) of this workgroup; s_a = its dynamic LDS
template <typename Tile, int MT, int WAVES>
__device__ __forceinline__ void qgemm_f16_body(const uint8_t* W, int64_t stride, const _Float16* Xh,
                                               const float* __restrict__ rowscale, float* Y, int M, int K, int N,
                                               int accumulate, int blocks_per_split, float* partials, int bx, int by, int bz,
                                               uint8_t* s_a, int scale_stride) {
    // W and Xh are deliberately not __restrict__: loads through a restrict pointer may be moved across the
    // compiler fences below, and the prefetch distance of this loop depends on those fences
    constexpr int TM = 32 * MT;                     // rows of X per workgroup (MT tiles of 32)
    constexpr int TN = 32 * WAVES;                  // columns per workgroup
    constexpr int RS = 2 * WAVES;                   // rows of the X tile that one fetch instruction of the workgroup covers
    constexpr int NPIECE = TM / RS;                 // 16-byte pieces of the X tile per thread
    static_assert((WAVES == 4 && (MT == 1 || MT == 2)) || (WAVES == 8 && (MT == 2 || MT == 4)), "wave layouts");
    static_assert(NPIECE == 4 || NPIECE == 8, "pieces per thread");
    const int tid = threadIdx.x, lane = tid & 63, wave = (tid >> 6) & 3;  // s_a: [2][TM * QF_PITCH]
    const int j = lane & 31, kh = lane >> 5;
    const int m0 = by * TM;
    const int n_base = bx * TN + (WAVES == 8 ? wave * 64 + 32 * (tid >> 8) : wave * 32);
    // split K: workgroup z of the grid sums super-blocks [blk0, blk0 + nblk) into its own M x N partial
    const int blk0 = bz * blocks_per_split;
    const int nblk = min(K / 256 - blk0, blocks_per_split);
    const uint8_t* wrow = W + (int64_t)min(n_base + j, N - 1) * stride + (int64_t)blk0 * Tile::kBlockBytes;

    f32x16 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mt][r] = 0.0f;

    // X tile of a block = TM rows x 512 B in pieces of 16 B; piece q = 64 WAVES i + tid (i < NPIECE) is row q / 32, bytes 16 (q % 32): a
    // wave fetches two whole rows per instruction and writes LDS without bank conflicts
    const int64_t x_row_bytes = (int64_t)K * 2;
    const uint8_t* x_src = reinterpret_cast<const uint8_t*>(Xh) + (int64_t)(m0 + (tid >> 5)) * x_row_bytes + 16 * (tid & 31) +
                           (int64_t)blk0 * 512;
    uint8_t* x_dst = s_a + (tid >> 5) * QF_PITCH + 16 * (tid & 31);
    float* s_rs = reinterpret_cast<float*>(s_a + 2 * TM * QF_PITCH);  // the tile's TM row scales (of rows past M, like the rows, anything: their sums are not stored)
    if (tid < TM) s_rs[tid] = rowscale[bz * scale_stride + m0 + tid];  // scale_stride 0: a row has one scale, not one per K split
    // the pieces of the next tile in flight (scalars, not an array: they must stay in registers)
    uint4 x0, x1, x2, x3, x4, x5, x6, x7;
    // prologue: tile of block 0 -> LDS buffer 0, weights of block 0, fragments of step 0.  The weight loads go out behind
    // the tile's, before anything waits: one memory round trip for both, not two (a launch of two or three blocks per
    // workgroup, as the K splits of the narrow projections are, is mostly this prologue)
#define QF_LD0(p) (*reinterpret_cast<const uint4*>(x_src + RS * (p) * x_row_bytes))
#define QF_ST0(p, v) (*reinterpret_cast<uint4*>(x_dst + RS * (p) * QF_PITCH) = (v))
    x0 = QF_LD0(0); x1 = QF_LD0(1); x2 = QF_LD0(2); x3 = QF_LD0(3);
    if constexpr (NPIECE == 8) { x4 = QF_LD0(4); x5 = QF_LD0(5); x6 = QF_LD0(6); x7 = QF_LD0(7); }
    issue_order_fence();
    Tile cur, nxt;
    cur.load(wrow, kh);
    issue_order_fence();
    QF_ST0(0, x0); QF_ST0(1, x1); QF_ST0(2, x2); QF_ST0(3, x3);
    if constexpr (NPIECE == 8) { QF_ST0(4, x4); QF_ST0(5, x5); QF_ST0(6, x6); QF_ST0(7, x7); }
#undef QF_LD0
#undef QF_ST0
    h8 bf[2], bn[2];
    cur.frags(0, kh, bf[0], bf[1]);
    __syncthreads();

    for (int blk = 0; blk < nblk; ++blk) {
        const int nb = min(blk + 1, nblk - 1);  // block whose tile and weights are fetched during this one
        const uint8_t* a_cur = s_a + (blk & 1) * (TM * QF_PITCH);
        uint8_t* x_nxt = x_dst + ((blk & 1) ^ 1) * (TM * QF_PITCH);
        const uint8_t* x_from = x_src + (int64_t)nb * 512;
        h8 af[2][MT];  // X fragments of step 0 of this block (the tile became visible at the barrier)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                af[ks][mt] = *reinterpret_cast<const h8*>(a_cur + (mt * 32 + j) * QF_PITCH + 32 * kh + 16 * ks);
#pragma unroll
        for (int s = 0; s < 8; ++s) {  // unrolled: the sub-block index selects registers
#define QF_LD(p) (*reinterpret_cast<const uint4*>(x_from + RS * (p) * x_row_bytes))
#define QF_ST(p, v) (*reinterpret_cast<uint4*>(x_nxt + RS * (p) * QF_PITCH) = (v))
            // Where a thread has eight pieces the fetches of the next block are spread over steps 0..3 and the LDS stores of the tile pieces
            // over steps 4..7: issued in one burst at step 0 they held up the vector-memory path for everything behind them
            // (512 x 4096 x 14336: 75.6 -> 72.1 us; a 2048-token prompt 26.3 -> 25.6 ms; prompts of up to 64 rows were 2 % slower
            // with their four pieces spread, so those keep the burst; the 64-row tile of four waves has eight, and the same time either
            // way: 64 rows, four layers of Qwen3-4B shapes, 537 ... 553 us spread, 549 in a burst).  Tile pieces go FIRST and the weights last (step 3):
            // loads return in order, so a wait for a piece must not have the weight loads (HBM latency, one cache line per
            // lane) in front of it; the weights are first needed at step 7.
            if constexpr (NPIECE == 8) {
                if (s == 0) { x0 = QF_LD(0); x1 = QF_LD(1); }
                if (s == 1) { x2 = QF_LD(2); x3 = QF_LD(3); }
                if (s == 2) { x4 = QF_LD(4); x5 = QF_LD(5); }
                if (s == 3) { x6 = QF_LD(6); x7 = QF_LD(7); issue_order_fence(); nxt.load(wrow + (int64_t)nb * Tile::kBlockBytes, kh); }
                if (s == 4) { QF_ST(0, x0); QF_ST(1, x1); }
                if (s == 5) { QF_ST(2, x2); QF_ST(3, x3); }
                if (s == 6) { QF_ST(4, x4); QF_ST(5, x5); }
                if (s == 7) { QF_ST(6, x6); QF_ST(7, x7); }
            } else {
                if (s == 0) {
                    x0 = QF_LD(0); x1 = QF_LD(1); x2 = QF_LD(2); x3 = QF_LD(3);
                    issue_order_fence();
                    nxt.load(wrow + (int64_t)nb * Tile::kBlockBytes, kh);
                }
                if (s == 3) { QF_ST(0, x0); QF_ST(1, x1); QF_ST(2, x2); QF_ST(3, x3); }
            }
#undef QF_LD
#undef QF_ST
            issue_order_fence();  // the fetches stay HERE, two steps ahead of their use (the compiler would sink them to it)
            // This step's X fragments were read from LDS during the previous step; nothing that consumes them may be hoisted
            // above this point.  (An MFMA is no memory operation: without this the scheduler moves each MFMA up to right
            // behind the LDS read of its operand, the fragments share ONE register quad, and every MFMA waits out the
            // LDS latency of its own operand.)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(af[ks][mt]));
            // X fragments of the NEXT step are read from LDS now and weight fragments of the next step are prepared
            // while this step's MFMAs (all operands already in registers) run
            h8 an[2][MT];
            if (s < 7) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt)
                        an[ks][mt] = *reinterpret_cast<const h8*>(a_cur + (mt * 32 + j) * QF_PITCH + 64 * (s + 1) + 32 * kh + 16 * ks);
            }
            if (s < 7) cur.frags(s + 1, kh, bn[0], bn[1]);
            else { nxt.pin(); nxt.frags(0, kh, bn[0], bn[1]); }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[ks][mt], bf[ks], acc[mt], 0, 0, 0);
            bf[0] = bn[0];
            bf[1] = bn[1];
            if (s < 7) {
#pragma unroll
                for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) af[ks][mt] = an[ks][mt];
            }
        }
        cur = nxt;
        __syncthreads();  // next tile complete, this tile no longer read
    }
    qf_store<MT>(acc, s_rs, Y, partials, accumulate, M, N, m0, n_base, j, kh, bz);
}

// ---- 256 and 192 rows x 256 columns ----
// A wave has one strip of 32 columns and all 256 rows (128 accumulators), so each unpacked weight serves twice the products of the 128-row tile, whose
// time is its matrix and its unpacking instructions one after the other.  A stage is half a super-block: X goes from memory to LDS directly, two stages
// of 64 KB, and the loop is laid out by hand: behind every MFMA the read of the fragment eight MFMAs on into the registers it has just freed, a
// piece of the next sub-block's weights behind every fourth, and one barrier a stage, between the last reads of its LDS and the first of the
// next, with MFMAs on either side.  The same products in the same order as in the 128-row tile: same bits.  With 192 rows, for launches that would
// leave CUs idle, everything is three quarters of that but the unpacking.
// What bounds it: 2048 x 14336 x 4096 in 236 us (276 in 128-row tiles), Q6_K 257 to 291 (427), 1020 TFLOP/s; the matrix cores are busy 67 % of the time that
// a workgroup is there (59 % in 128-row tiles), at which the card lowers its clock (1.8 GHz; 1.6 at 2048 x 28672 x 4096).  Where the barrier lies, when the weights are
// requested and how the pieces are spread change it by less than 1 %.  The same loop for 128 rows is 1 to 5 % slower than qgemm_f16_body.

// What a lane (column n, element half kh) holds of half a super-block, and the fragments of its four sub-blocks, four pieces each.
struct Q4Half {
    uint4 hdr, qs[2];
    uint32_t sc4, mn4;
    __device__ __forceinline__ void load(const uint8_t* blk, int half, int kh) {
        hdr = *reinterpret_cast<const uint4*>(blk);
#pragma unroll
        for (int g = 0; g < 2; ++g) qs[g] = *reinterpret_cast<const uint4*>(blk + 16 + 64 * half + 32 * g + 16 * kh);
    }
    // scales and mins of the four sub-blocks, a byte each (q4k_scale_min)
    __device__ __forceinline__ void arrive(int half, int) {
        pin4(hdr); pin4(qs[0]); pin4(qs[1]);
        sc4 = half ? (hdr.w & 0x0f0f0f0fu) | ((hdr.y >> 2) & 0x30303030u) : hdr.y & 0x3f3f3f3fu;
        mn4 = half ? ((hdr.w >> 4) & 0x0f0f0f0fu) | ((hdr.z >> 2) & 0x30303030u) : hdr.z & 0x3f3f3f3fu;
    }
    __device__ __forceinline__ void scale(int s, h2& sc, h2& of) const {
        const float dsc = h2f(hdr.x) * (float)((sc4 >> (8 * s)) & 0xffu), dmn = h2f(hdr.x >> 16) * (float)((mn4 >> (8 * s)) & 0xffu);
        sc = {(_Float16)dsc, (_Float16)dsc};
        of = {(_Float16)-dmn, (_Float16)-dmn};
    }
    __device__ __forceinline__ uint32_t bytes(int s, int w) const {
        const uint32_t r[4] = {qs[s >> 1].x, qs[s >> 1].y, qs[s >> 1].z, qs[s >> 1].w};
        return (r[w] >> (4 * (s & 1))) & 0x0f0f0f0fu;
    }
    static constexpr float kBias = 0.0f;
    static constexpr int kBlockBytes = 144;
};
struct Q6Half {
    uint4 ql[2], qh;
    uint32_t s0, s1, d;
    __device__ __forceinline__ void load(const uint8_t* blk, int half, int kh) {
#pragma unroll
        for (int c = 0; c < 2; ++c) ql[c] = ld16_a2(blk + 64 * half + 32 * c + 16 * kh);
        qh = ld16_a2(blk + 128 + 32 * half + 16 * kh);
        s0 = ld_u32_a2(blk + 192 + 8 * half);
        s1 = ld_u32_a2(blk + 196 + 8 * half);
        d = reinterpret_cast<const u16_a2*>(blk + 208)->v;
    }
    __device__ __forceinline__ void arrive(int, int kh) {
        pin4(ql[0]); pin4(ql[1]); pin4(qh);
        asm volatile("" : "+v"(s0), "+v"(s1), "+v"(d));
        s0 >>= 8 * kh;  // scales 2 s + kh in bytes 0 and 2
        s1 >>= 8 * kh;
    }
    __device__ __forceinline__ void scale(int s, h2& sc, h2& of) const {
        const int sv = (int)(int8_t)(((s >> 1 ? s1 : s0) >> (16 * (s & 1))) & 0xffu);
        const float v = h2f(d) * (float)sv;
        sc = {(_Float16)v, (_Float16)v};
        of = {(_Float16)0.0f, (_Float16)0.0f};
    }
    __device__ __forceinline__ uint32_t bytes(int s, int w) const {
        const uint32_t l[4] = {ql[s & 1].x, ql[s & 1].y, ql[s & 1].z, ql[s & 1].w}, h[4] = {qh.x, qh.y, qh.z, qh.w};
        return ((l[w] >> (4 * (s >> 1))) & 0x0f0f0f0fu) | (((h[w] >> (2 * s)) & 0x03030303u) << 4);
    }
    static constexpr float kBias = 32.0f;
    static constexpr int kBlockBytes = 210;
};


template <typename Half, int MT>
__device__ __forceinline__ void qgemm_f16_tall_body(const uint8_t* W, int64_t stride, const _Float16* Xh, const float* __restrict__ rowscale, float* Y,
                                                    int M, int K, int N, int accumulate, int blocks_per_split, float* partials, int bx, int by,
                                                    int bz, uint8_t* s_a, int scale_stride) {
    static_assert(MT == 8 || MT == 6, "row tiles of 32");
    constexpr int TM = 32 * MT, STAGE = TM * 256, H = MT / 2;
    static_assert(2 * STAGE + 4 * TM <= QF_ROWS_LDS, "two stages and the row scales");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kh = lane >> 5;
    const int m0 = by * TM, n_base = bx * 256 + 64 * (wave & 3) + 32 * (wave >> 2);
    const int blk0 = bz * blocks_per_split, nblk = min(K / 256 - blk0, blocks_per_split), nst = 2 * nblk;
    const uint8_t* wrow = W + (int64_t)min(n_base + j, N - 1) * stride + (int64_t)blk0 * Half::kBlockBytes;

    // X: row r of a stage is 256 bytes of LDS, its sixteen 16-byte pieces at piece ^ (r % 16).  A wave's instruction fetches four rows.
    const uint32_t row_bytes = (uint32_t)K * 2, last = min(M - 1 - m0, TM - 1), r0 = 4 * wave + (lane >> 4);
    const uint32_t piece = ((lane & 15) ^ (r0 & 15)) << 4;
    gt_i4 xs = gt_buffer(reinterpret_cast<const uint8_t*>(Xh) + (int64_t)m0 * K * 2 + (int64_t)blk0 * 512);
    xs[0] = __builtin_amdgcn_readfirstlane(xs[0]);  // the compiler does not always see that they are the same in every lane
    xs[1] = __builtin_amdgcn_readfirstlane(xs[1]);
    const uint32_t lds0 = (uint32_t)(uintptr_t)s_a + wave * 1024;
    auto fetch = [&](int st, int i) { gt_to_lds(lds0 + (st & 1) * STAGE + i * 8192, (int)(min(r0 + 32 * i, last) * row_bytes + piece), xs, st * 256); };

    float* s_rs = reinterpret_cast<float*>(s_a + 2 * STAGE);
    f32x16 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mt][r] = 0.0f;
    Half w[2];
    for (int i = 0; i < MT; ++i) fetch(0, i);
    w[0].load(wrow, 0, kh);
    issue_order_fence();
    for (int i = 0; i < MT; ++i) fetch(1, i);
    if (tid < TM) s_rs[tid] = rowscale[bz * scale_stride + m0 + min(tid, (int)last)];
    h2 sc, of;
    uint32_t bf[2][8];  // [buffer][two fragments of four]
    auto dequant = [&](const Half& h, int s, int q, uint32_t (&out)[8]) {
        const h2 sub = {(_Float16)(1024.0f + Half::kBias), (_Float16)(1024.0f + Half::kBias)};
        const uint32_t b = h.bytes(s, q);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t hq = __builtin_amdgcn_perm(0x64646464u, b, p ? 0x04030402u : 0x04010400u);
            h2 x;
            __builtin_memcpy(&x, &hq, 4);
            const h2 v = __builtin_elementwise_fma(x - sub, sc, of);
            __builtin_memcpy(&out[2 * q + p], &v, 4);
        }
    };
    w[0].arrive(0, kh);
    w[0].scale(0, sc, of);
#pragma unroll
    for (int q = 0; q < 4; ++q) dequant(w[0], 0, q, bf[0]);
    gt_arrived<0>();
    const int a0 = j * 256 + (((2 * kh) ^ (j & 15)) << 4);
    h8 af[MT];
    auto read = [&](int from, int mt) { af[mt] = *reinterpret_cast<const h8*>(s_a + from + mt * 8192); };
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) read(a0, mt);

    auto stage = [&](int st, auto half_) {  // 8 groups of MT MFMAs: 16 values of K each
        constexpr int half = decltype(half_)::value;
        Half& cur = w[half];
        Half& nxt = w[half ^ 1];
        constexpr int at = half * STAGE;
#pragma unroll
        for (int g = 0; g < 8; ++g) {
            const int s = g >> 1, ks = g & 1;
            // where the fragments of the next 16 values of K lie (in assembly: hoisted out of the loop, the sixteen places cost as many registers)
            int from;
            asm volatile("v_xor_b32 %0, %1, %2" : "=v"(from) : "v"(a0), "s"(((4 * (((g + 1) >> 1) & 3) + ((g + 1) & 1)) << 4) | (g < 7 ? at : STAGE - at)));
            h8 b;
            __builtin_memcpy(&b, &bf[s & 1][4 * ks], 16);
            if (g == 6) nxt.arrive(half ^ 1, kh);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                __builtin_amdgcn_sched_barrier(0);
                acc[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[mt], b, acc[mt], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if (g < 7) read(from, mt);
                else if (mt >= H) { read(from, 2 * (mt - H)); read(from, 2 * (mt - H) + 1); }
                // weights of the next sub-block
                const Half& src = s < 3 ? cur : nxt;
                const int slot = MT * ks + mt, sn = (s + 1) & 3;
                if (slot == 0) src.scale(sn, sc, of);
                if (slot % H == H / 2) dequant(src, sn, slot / H, bf[(s + 1) & 1]);
                // the stage after the next, into the half of LDS this one is read from; the next half block of weights
                if (g == 7 && mt == H - 1) gt_arrived<0>();
                if (g == 7 && mt >= H && st + 2 < nst) fetch(st + 2, mt - H);
                if (g == 0 && mt < H && st > 0 && st + 1 < nst) fetch(st + 1, mt + H);
                if (g == 2 && mt == 0) nxt.load(wrow + (int64_t)min((st + 1) >> 1, nblk - 1) * Half::kBlockBytes, half ^ 1, kh);
            }
        }
    };
    for (int st = 0; st < nst; st += 2) {
        stage(st, std::integral_constant<int, 0>{});
        stage(st + 1, std::integral_constant<int, 1>{});
    }
    qf_store<MT>(acc, s_rs, Y, partials, accumulate, M, N, m0, n_base, j, kh, bz);
}

// Which tile a workgroup takes.  The hardware deals consecutive workgroup ids round-robin to the 8 XCDs, each with its own
// L2; taken as they come, the workgroups of one XCD are scattered over all column tiles, row tiles and K splits and share
// almost nothing (the down projection of a 512-row prompt, 10 x 4 tiles x 6 splits, then pulls 200 MB through the L2s for
// 30 MB of operands).  Here the workgroups an XCD receives form one contiguous run of the order "row tile fastest, then
// column tile (or slot) within a band of 4 row tiles, then band, then K split": the 32 or so workgroups an XCD runs at a time
// are then about 4 row tiles x 8 column tiles, so each weight piece serves 4 of them and each X tile 8 from one L2.
__device__ __forceinline__ int qf_xcd_order(int hw, int nwg) {
    const int xcd = hw & 7, slot = hw >> 3, per = nwg >> 3, rem = nwg & 7;
    return xcd * per + (xcd < rem ? xcd : rem) + slot;
}
// position L of that order -> (column tile or slot, row tile, K split) on a gx x gy x gz grid
__device__ __forceinline__ void qf_tile_of(int L, int gx, int gy, int& bx, int& by, int& bz) {
    const int plane = gx * gy;
    bz = L / plane;
    const int r = L - bz * plane;
    const int band = r / (4 * gx);
    const int rows = min(4, gy - 4 * band);
    const int within = r - band * 4 * gx;
    by = 4 * band + within % rows;
    bx = within / rows;
}

// The first `tall` workgroups of a launch take 256 rows each, in that order of pairs of row tiles; the tiles of 128 rows that are left, two from
// each pair, follow (qf_tall).  QF_192: all take 192.  False: a row tile past the last.
constexpr int QF_192 = -1;
__device__ __forceinline__ bool qf_place(int hw, int nwg, int gx, int M, int tall, int& bx, int& by, int& bz) {
    const int gy = tall == QF_192 ? (M + 191) / 192 : (M + QF_TM - 1) / QF_TM;
    if (tall <= 0) {
        qf_tile_of(qf_xcd_order(hw, nwg), gx, gy, bx, by, bz);
        return true;
    }
    const int rest = hw - tall, L = rest < 0 ? qf_xcd_order(hw, tall) : qf_xcd_order(rest, nwg - tall);
    qf_tile_of(rest < 0 ? L : tall + (L >> 1), gx, (gy + 1) >> 1, bx, by, bz);
    if (rest >= 0) by = 2 * by + (L & 1);
    return rest < 0 || by < gy;
}

// tiles of 128, 192 and 256 rows by 256 columns
template <typename Tile>
__global__ __launch_bounds__(512, 1) void qgemm_f16_rows_kernel(const uint8_t* W, int64_t stride, const _Float16* Xh, const float* __restrict__ rowscale,
                                                                float* Y, int M, int K, int N, int accumulate, int blocks_per_split, float* partials,
                                                                int scale_stride, int tall) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(W, M);
    int bx, by, bz;
    if (!qf_place(blockIdx.x, gridDim.x, (N + QF_TN - 1) / QF_TN, M, tall, bx, by, bz)) return;
    if (tall == QF_192)
        qgemm_f16_tall_body<typename Tile::Half, 6>(W, stride, Xh, rowscale, Y, M, K, N, accumulate, blocks_per_split, partials, bx, by, bz, qf_lds, scale_stride);
    else if ((int)blockIdx.x < tall)
        qgemm_f16_tall_body<typename Tile::Half, 8>(W, stride, Xh, rowscale, Y, M, K, N, accumulate, blocks_per_split, partials, bx, by, bz, qf_lds, scale_stride);
    else
        qgemm_f16_body<Tile, 4, 8>(W, stride, Xh, rowscale, Y, M, K, N, accumulate, blocks_per_split, partials, bx, by, bz, qf_lds, scale_stride);
}

template <typename Tile, int MT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, (WAVES == 8 ? 1 : 2)) void qgemm_f16_kernel(const uint8_t* W, int64_t stride, const _Float16* Xh,
                                                        const float* __restrict__ rowscale, float* Y, int M, int K, int N,
                                                        int accumulate, int blocks_per_split, float* partials, int scale_stride) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(W, M);
    const int hw = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int L = qf_xcd_order(hw, gridDim.x * gridDim.y * gridDim.z);
    int bx, by, bz;
    qf_tile_of(L, gridDim.x, gridDim.y, bx, by, bz);
    qgemm_f16_body<Tile, MT, WAVES>(W, stride, Xh, rowscale, Y, M, K, N, accumulate, blocks_per_split, partials, bx, by, bz, qf_lds, scale_stride);
}

// up to 32 rows, NB super-blocks per split
template <typename Tile, int NB>
__global__ __launch_bounds__(256, (NB <= 2 ? 3 : 2)) void qgemm_f16_short_kernel(const uint8_t* W, int64_t stride, const _Float16* Xh, const float* __restrict__ rowscale,
                                                                 float* Y, int M, int K, int N, int accumulate, int blocks_per_split, float* partials,
                                                                 int scale_stride) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(W, M);
    const int L = qf_xcd_order(blockIdx.x, gridDim.x), tiles = (N + 127) / 128;
    qgemm_f16_short_body<Tile, NB>(W, stride, Xh, rowscale, Y, M, K, N, accumulate, blocks_per_split, partials, L % tiles, L / tiles, qf_lds, scale_stride);
}

// Up to three projections of the same rows in ONE launch, its tile chosen as below for a single matrix (q, k, v of a layer: in a Q4_K_M
// file two Q4_K matrices and a Q6_K one).  Each matrix brings its own prepared rows (Q8-rounded for Q4_K, plain for
// Q6_K), column tiles and K splits; blockIdx.x walks the (column tile, split) slots of the matrices one after the other.
// Three narrow launches of two or three blocks per workgroup are mostly launch, prologue and epilogue; one launch pays
// them once and fills the chip.
struct QfMat {
    const uint8_t* W;
    int64_t stride;
    const _Float16* Xh;
    const float* rowscale;
    float* Y;
    float* partials;  // NULL: one split, written to Y
    int N, bps, ntiles, slot_end, q6;
};
struct QfMulti { QfMat m[3]; int n_mat; };

template <int MT, int WAVES>
__global__ __launch_bounds__(64 * WAVES, (WAVES == 8 ? 1 : 2)) void qgemm_f16_multi_kernel(const QfMulti a, int M, int K) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(a.m[0].W, a.m[1].W, a.m[2].W, a.n_mat);
    const int L = qf_xcd_order(blockIdx.x + gridDim.x * blockIdx.y, gridDim.x * gridDim.y);
    int sx, by, unused;
    qf_tile_of(L, gridDim.x, gridDim.y, sx, by, unused);  // sx: the (matrix, split, column tile) slot
    int i = 0;
    if (a.n_mat > 1 && sx >= a.m[0].slot_end) i = 1;
    if (a.n_mat > 2 && sx >= a.m[1].slot_end) i = 2;
    const QfMat& q = i == 0 ? a.m[0] : (i == 1 ? a.m[1] : a.m[2]);
    const int local = sx - (i == 0 ? 0 : (i == 1 ? a.m[0].slot_end : a.m[1].slot_end));
    const int bx = local % q.ntiles, bz = local / q.ntiles;
    if (q.q6) qgemm_f16_body<Q6Tile, MT, WAVES>(q.W, q.stride, q.Xh, q.rowscale, q.Y, M, K, q.N, 0, q.bps, q.partials, bx, by, bz, qf_lds, 0);
    else qgemm_f16_body<Q4Tile, MT, WAVES>(q.W, q.stride, q.Xh, q.rowscale, q.Y, M, K, q.N, 0, q.bps, q.partials, bx, by, bz, qf_lds, 0);
}

// the same in tiles of 128, 192 and 256 rows
__global__ __launch_bounds__(512, 1) void qgemm_f16_rows_multi_kernel(const QfMulti a, int M, int K, int slots, int tall) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(a.m[0].W, a.m[1].W, a.m[2].W, a.n_mat);
    int sx, by, unused;
    if (!qf_place(blockIdx.x, gridDim.x, slots, M, tall, sx, by, unused)) return;
    int i = 0;
    if (a.n_mat > 1 && sx >= a.m[0].slot_end) i = 1;
    if (a.n_mat > 2 && sx >= a.m[1].slot_end) i = 2;
    const QfMat& q = i == 0 ? a.m[0] : (i == 1 ? a.m[1] : a.m[2]);
    const int local = sx - (i == 0 ? 0 : (i == 1 ? a.m[0].slot_end : a.m[1].slot_end));
    const int bx = local % q.ntiles, bz = local / q.ntiles;
#define PTM_QR(BODY) BODY(q.W, q.stride, q.Xh, q.rowscale, q.Y, M, K, q.N, 0, q.bps, q.partials, bx, by, bz, qf_lds, 0)
    if (tall == QF_192) {
        if (q.q6) PTM_QR((qgemm_f16_tall_body<Q6Half, 6>));
        else PTM_QR((qgemm_f16_tall_body<Q4Half, 6>));
    } else if ((int)blockIdx.x < tall) {
        if (q.q6) PTM_QR((qgemm_f16_tall_body<Q6Half, 8>));
        else PTM_QR((qgemm_f16_tall_body<Q4Half, 8>));
    } else {
        if (q.q6) PTM_QR((qgemm_f16_body<Q6Tile, 4, 8>));
        else PTM_QR((qgemm_f16_body<Q4Tile, 4, 8>));
    }
#undef PTM_QR
}

// the same for up to 32 rows and up to NB super-blocks per split
template <int NB>
__global__ __launch_bounds__(256, (NB <= 2 ? 3 : 2)) void qgemm_f16_short_multi_kernel(const QfMulti a, int M, int K) {
    extern __shared__ __align__(16) uint8_t qf_lds[];
    read_now(a.m[0].W, a.m[1].W, a.m[2].W, a.n_mat);
    const int sx = qf_xcd_order(blockIdx.x, gridDim.x);
    int i = 0;
    if (a.n_mat > 1 && sx >= a.m[0].slot_end) i = 1;
    if (a.n_mat > 2 && sx >= a.m[1].slot_end) i = 2;
    const QfMat& q = i == 0 ? a.m[0] : (i == 1 ? a.m[1] : a.m[2]);
    const int local = sx - (i == 0 ? 0 : (i == 1 ? a.m[0].slot_end : a.m[1].slot_end));
    const int bx = local % q.ntiles, bz = local / q.ntiles;
#define PTM_QS(TILE, B) qgemm_f16_short_body<TILE, B>(q.W, q.stride, q.Xh, q.rowscale, q.Y, M, K, q.N, 0, q.bps, q.partials, bx, bz, qf_lds, 0)
    if constexpr (NB <= 2) {
        if (q.q6) {
            if (q.bps == 1) PTM_QS(Q6Tile, 1);
            else PTM_QS(Q6Tile, 2);
        } else {
            if (q.bps == 1) PTM_QS(Q4Tile, 1);
            else PTM_QS(Q4Tile, 2);
        }
    } else if (q.q6) {
        if (q.bps <= 2) PTM_QS(Q6Tile, 2);
        else if (q.bps == 3) PTM_QS(Q6Tile, 3);
        else PTM_QS(Q6Tile, 4);
    } else {
        if (q.bps <= 2) PTM_QS(Q4Tile, 2);
        else if (q.bps == 3) PTM_QS(Q4Tile, 3);
        else PTM_QS(Q4Tile, 4);
    }
#undef PTM_QS
}

// Y (+)= partials[0] + partials[1] + ... in that fixed order (deterministic, unlike atomics)
__global__ __launch_bounds__(256) void qgemm_split_reduce_kernel(const float* __restrict__ P, int splits, float* __restrict__ Y,
                                                                 int64_t total, int accumulate) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= total) return;
    if (i + 4 <= total && (total & 3) == 0) {
        float4 a = *reinterpret_cast<const float4*>(P + i);
        for (int z = 1; z < splits; ++z) {
            const float4 b = *reinterpret_cast<const float4*>(P + z * total + i);
            a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
        }
        float4* y = reinterpret_cast<float4*>(Y + i);
        if (accumulate) { const float4 o = *y; a.x += o.x; a.y += o.y; a.z += o.z; a.w += o.w; }
        *y = a;
    } else {
        for (int64_t e = i; e < total && e < i + 4; ++e) {
            float a = P[e];
            for (int z = 1; z < splits; ++z) a += P[z * total + e];
            Y[e] = accumulate ? Y[e] + a : a;
        }
    }
}

// the same for the matrices of a multi-matrix launch: blockIdx.x walks the segments' 1024-element pieces
struct QfRedSeg { const float* P; float* Y; int64_t total; int splits, blk_end; };
struct QfRedMulti { QfRedSeg s[3]; int n; };
__global__ __launch_bounds__(256) void qgemm_split_reduce_multi_kernel(const QfRedMulti a) {
    int k = 0;
    if (a.n > 1 && (int)blockIdx.x >= a.s[0].blk_end) k = 1;
    if (a.n > 2 && (int)blockIdx.x >= a.s[1].blk_end) k = 2;
    const QfRedSeg& g = k == 0 ? a.s[0] : (k == 1 ? a.s[1] : a.s[2]);
    const int b = (int)blockIdx.x - (k == 0 ? 0 : (k == 1 ? a.s[0].blk_end : a.s[1].blk_end));
    const int64_t i = ((int64_t)b * 256 + threadIdx.x) * 4;
    if (i >= g.total) return;
    if (i + 4 <= g.total && (g.total & 3) == 0) {
        float4 v = *reinterpret_cast<const float4*>(g.P + i);
        for (int z = 1; z < g.splits; ++z) {
            const float4 w = *reinterpret_cast<const float4*>(g.P + z * g.total + i);
            v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
        }
        *reinterpret_cast<float4*>(g.Y + i) = v;
    } else {
        for (int64_t e = i; e < g.total && e < i + 4; ++e) {
            float v = g.P[e];
            for (int z = 1; z < g.splits; ++z) v += g.P[z * g.total + e];
            g.Y[e] = v;
        }
    }
}

// Row classes of the split rules: up to 128 rows, up to 256, up to 1024, more (2048-row chunks of long prompts: with 16 row
// tiles per column tile, as many splits as a 512-row launch wants only multiply the partial sums).
enum { QF_MAX_SPLITS = 16 };
static inline int qf_row_class(int M) { return M <= 128 ? 1 : (M <= 256 ? 2 : (M <= 1024 ? 4 : 8)); }

// K splits for an N x K weight matrix and M rows: enough workgroups to fill the chip when N alone gives few column
// tiles (a 2560-wide projection is 10 tiles).  M enters only through its class, so
// that the summation order of a row does not change with how many rows share the launch within a class; short
// prompts (one row tile) get up to 16 splits, because there the launch is bound by how many workgroups stream weights.
// Where workgroups have 128 columns (below), a few more of them than a round of the chip double what some CUs do: then more
// blocks a split (2560 x 9728, 19 rows: 13 splits of three blocks, 260 workgroups, Q6_K 15.9 us, Q4_K 10.1; 247 of them 11.3 and 8.1; ten of four, 200, 13.5 and 9.4;
// 19 of two 11.8 and 8.4, but as many more sums for the next kernel).  18 layers of Qwen3-4B shapes, 19 rows 1364 -> 1343 us, 40 rows 1676 -> 1606, 64
// rows 1713 -> 1645, 100 rows 2181 and 2185, 128 rows 2222 and 2237; 12 of Gemma-3-4B shapes, 30 rows 1276 -> 1254.
int qgemm_f16_splits(int N, int K, int M) {
    const int ntiles = (N + QF_TN - 1) / QF_TN, nblk = K / 256;
    const int row_tiles = qf_row_class(M);
    int s = 256 / (ntiles * row_tiles);
    const int cap = row_tiles == 1 ? QF_MAX_SPLITS : 8;
    s = s > cap ? cap : s;
    s = s > nblk / 2 ? nblk / 2 : s;
    s = s < 1 ? 1 : s;
    if (M <= 128 && s > 1) {
        const int tiles = (N + 127) / 128, from = (nblk + s - 1) / s;
        auto blocks = [&](int bps) { return (tiles * ((nblk + bps - 1) / bps) + 255) / 256 * bps; };
        int best = from;
        for (int bps = from + 1; bps <= QF_SHORT_BLOCKS; ++bps)
            if (blocks(bps) < blocks(best)) best = bps;
        s = (nblk + best - 1) / best;
    }
    return s;
}

// K splits of the matrices of a multi-matrix launch.  All (column tile, split) slots of all matrices must fit one round of
// the chip (256 workgroups over the row tiles of M's class, as above), and the launch lasts as long as its slowest
// workgroup: starting from one split each, the matrix whose workgroups have the most work (blocks per split, a Q6_K block
// weighing 1.6 Q4_K blocks: measured 8 against 5 us) gets its next split count until the slots run out.  A function of
// the shapes, the types and M's class only, like qgemm_f16_splits.
// (A split more where workgroups of 128 columns would do a fifth less on the busiest CU: 2 x 22016 x 4096, 5 / 32 rows 49.3 / 50.8 -> 45.3 / 48.8 us, but the rows of
// a class share their splits: 40 / 100 / 128 rows 57.0 / 66.6 / 68.8 -> 67.0 / 87.6 / 90.5; 2 x 24576 x 2048, 32 / 128 rows 30.9 / 43.9 -> 34.1 / 66.3.)
void qgemm_f16_multi_plan(int n, const int* N, const uint32_t* types, int K, int M, int* splits) {
    const int nblk = K / 256;
    const int row_tiles = qf_row_class(M);
    const int budget = 256 / row_tiles;
    const int cap = (row_tiles == 1 ? 16 : 8) < nblk / 2 ? (row_tiles == 1 ? 16 : 8) : (nblk / 2 < 1 ? 1 : nblk / 2);
    int ntile[3], slots = 0;
    for (int i = 0; i < n; ++i) { splits[i] = 1; ntile[i] = (N[i] + QF_TN - 1) / QF_TN; slots += ntile[i]; }
    for (;;) {
        int j = -1;
        float worst = 0.0f;
        for (int i = 0; i < n; ++i) {
            const float est = (float)((nblk + splits[i] - 1) / splits[i]) * (types[i] == PTM_TYPE_Q6_K ? 1.6f : 1.0f);
            if (est > worst) { worst = est; j = i; }
        }
        if (j < 0) break;
        const int bps = (nblk + splits[j] - 1) / splits[j];
        if (bps <= 1) break;
        const int next = (nblk + bps - 2) / (bps - 1);  // the fewest splits with fewer blocks each
        if (next > cap || slots + ntile[j] * (next - splits[j]) > budget) break;
        slots += ntile[j] * (next - splits[j]);
        splits[j] = next;
    }
}

// Which tiles of a launch of gx column tiles (slots) and gz K splits have 256 rows: the first `tall` pairs of row tiles in qf_tile_of's order, in whole
// rounds of the chip or all of them - or whether all tiles have 192 - whichever lets the launch end first; returns its time in rounds of 128-row tiles.  A tile of 256 rows takes 1.75
// times (Q6_K, more to unpack: 1.5 times) as long as one of 128, and where its last round leaves CUs idle, 128-row tiles run there; a tile of 192 rows
// 1.4 to 1.6 times (Q6_K 1.35), by how much of the chip the other tiles leave idle, that is to say how far they let it clock.  In us, all of 128 rows, all
// of 256, whole rounds of 256 and 128 behind them, 192, and by this rule (a run of its own: the same plan again differs by up to 12 %; since then
// qf_store takes 3 to 10 us less of each):
//   509 x 19456 x 2560     82  79   -   68   63 (192)        Q6_K  107  77   -   70   72 (192)
//   953 x 19456 x 2560    133 154  129 120  123 (256, 128)
//   953 x 28672 x 4096    273 234  254 265  238 (256)
//   953 x 14336 x 4096    131 120   -  167  118 (256)        Q6_K  170 124   -  199  125 (256)
//   2048 x 9728 x 2560    132 147  123 121  122 (256, 128)
//   2048 x 14336 x 4096   276 236  256 269  237 (256)        Q6_K  427 257  314 322  291 (256)
//   2048 x 28672 x 4096   496 471  451 477  459 (256, 128)
//   300 x 14336 x 4096     59  94   -   74   59 (128)        953 x 18944 x 3584, Q6_K  236 214  195 188  195 (256, 128)
//   384 x 28672 x 4096    121 117   -   93   92 (192)        2048 x 4096 x 14336, Q6_K 317 350   -  314  300 (128)
// A launch of several matrices counts as Q6_K where one of them is (v beside q and k): up to 50 column tiles and 2048 rows both counts choose the same.
static float qf_tall(int gx, int gz, int M, bool q4, int* tall) {
    const int gy = (M + QF_TM - 1) / QF_TM, pairs = (gy + 1) / 2, plane = gx * pairs, all = plane * gz;
    const float ratio = q4 ? 1.75f : 1.5f;
    // 128-row tiles in the pairs from place t of that order on: two each, but one in the last pair of an odd number of row tiles
    auto left = [&](int t) {
        const int last_band = (pairs - 1) / 4 * 4, r = t % plane - last_band * gx;
        const int single = gy & 1 ? gx * gz - (t / plane * gx + (r > 0 ? r / (pairs - last_band) : 0)) : 0;
        return 2 * (all - t) - single;
    };
    float best = (float)((left(0) + 255) / 256);
    *tall = 0;
    for (int t : {all / 256 * 256, all}) {
        if (t == 0) continue;
        const int rounds = (t + 255) / 256, rest = left(t) - (256 * rounds - t);
        const float cost = ratio * (float)rounds + (float)(rest > 0 ? (rest + 255) / 256 : 0);
        if (cost < best) { best = cost; *tall = t; }
    }
    const float cost = (q4 ? 1.5f : 1.35f) * (float)((gx * gz * ((M + 191) / 192) + 255) / 256);
    if (cost < best) { best = cost; *tall = QF_192; }
    return best;
}
static int qf_workgroups(int gx, int gz, int M, int tall) {
    const int gy = (M + QF_TM - 1) / QF_TM;
    return tall == QF_192 ? gx * ((M + 191) / 192) * gz : tall ? tall + 2 * (gx * ((gy + 1) / 2) * gz - tall) : gx * gy * gz;
}

// rounds of a launch of matrices with `tiles` column tiles and K splits together
float qgemm_f16_rounds(int tiles, int M, bool q4) {
    int tall;
    return qf_tall(tiles, 1, M, q4, &tall);
}

// Workgroups of 128 columns (and up to 64 rows): always up to 32 rows, up to 64 where the chip then has a CU for each, with more rows where two
// of them fit every CU: half the columns and half the rows are half the unpacking and a quarter of the products of a workgroup that leaves CUs idle.  Prompts of
// 19 / 32 / 50 / 64 tokens, Qwen3-4B shapes, 256 columns, this rule, 128 always: 3.53 / 3.67 / 3.97 / 4.12 ms, 3.32 / 3.45 / 3.89 / 4.00, 3.32 / 3.45 / 3.86 / 3.97;
// Llama-3-8B shapes in 16 layers, 60 tokens: 2.28, 2.28, 2.31; in 8 layers, 5 / 19 / 32 tokens, 256 columns and so: 1.05 / 1.10 / 1.13, 1.00 / 1.05 /
// 1.09.  Up to 32 rows a single product is 10 to 25 % faster where 256 columns are up to 128 workgroups, and the same within -3 to 3 % where they are
// more (32 x 4096 x 14336 22.5 -> 23.2 us, 2 x 9728 x 16384 41.7 -> 40.7).  More than 64 rows, 256 columns and so, and with three of them to two CUs: 70 / 128 rows,
// 18 layers of Qwen3-4B shapes 2039 / 2191 -> 1978 / 2122 us, 16 of width 1024 (66, 128, 250, 600, 1500 rows) 1183 1164 1415 1707 2868 -> 896 921 1157 1592 2818, the
// last three then 1141 1585 2925; 12 layers of Qwen3-4B, 160 / 250 rows 1898 / 2088, 1847 / 2078, 1909 / 2204; 6 of Llama-3-8B, 190 rows 1301, 1296, 1457.
// A row's sum does not depend on the choice.
static bool qf_narrow(int M, int wide_workgroups) { return M <= 32 || (M <= 64 ? wide_workgroups <= 128 : (int64_t)wide_workgroups * ((M + 63) / 64) <= 256); }

// Q4_K products of one split (where K may be split, 257 to 384 rows of 8193 to 10752 columns): where workgroups of 64 rows and 256 columns leave no CU two and would be more than half
// the chip, but ones of 128 rows would not be, they are faster than twice as many of 128 columns, whose X each needs again: 280 / 384 rows, 9728 x 2560 31.4 / 33.2 ->
// 29.4 / 32.2 us, x 4096 45.3 / 48.1 -> 43.2 / 46.7, 9216 x 1024 16.6 / 16.9 -> 15.6 / 16.6; of 512 values and of 8192 up to 4 % slower, of 14336
// 3 % either way.  (Q6_K, more to unpack, 9728 x 2560: 54 us so, 46 narrow.)
static bool qf_flat(int M, int K, int wide_workgroups) {
    return M > 64 && K >= 1024 && K <= 4096 && wide_workgroups * ((M + 127) / 128) < 128 && (int64_t)wide_workgroups * ((M + 63) / 64) > 128;
}

static int qgemm_check(const void* W, const void* X, const void* Y, int M, int K, int N, int64_t stride, int blk_bytes) {
    if (!W || !X || !Y) return PTM_E_NULL;
    if (M <= 0 || N <= 0 || K <= 0 || (K % 256) != 0) return PTM_E_SHAPE;
    if (stride < (int64_t)(K / 256) * blk_bytes) return PTM_E_SHAPE;
    if (!aligned16(X) || (reinterpret_cast<uintptr_t>(Y) & 3u)) return PTM_E_ALIGN;
    if ((int64_t)qg_mpad(M) / QG_MCHUNK > 65535) return PTM_E_UNSUPPORTED;
    return PTM_OK;
}

// room in a row workspace for a scale per row and K split
int64_t qgemm_f16_split_scale_bytes(int M) { return (int64_t)QF_MAX_SPLITS * qf_mpad(M) * 4; }

// where the M rows of K values and their scales lie in a row workspace
void qgemm_f16_row_workspace(void* workspace, int M, int K, void** rows, float** rowscale) {
    *rows = workspace;
    *rowscale = reinterpret_cast<float*>(static_cast<_Float16*>(workspace) + (int64_t)qf_mpad(M) * K);
}

// super-blocks per K split of qgemm_f16_impl with that much room for partial sums
int qgemm_f16_blocks_per_split(int N, int K, int M, size_t split_ws_bytes) {
    int splits = split_ws_bytes ? qgemm_f16_splits(N, K, M) : 1;
    while (splits > 1 && (size_t)splits * M * N * sizeof(float) > split_ws_bytes) --splits;
    return (K / 256 + splits - 1) / splits;
}

// Y (+)= X . W^T with X bf16 or fp32 rows; shared by the C entry points and the prefill runtime.
int qgemm_f16_impl(uint32_t ggml_type, const void* W, const void* X, bool x_is_f32, float* Y, int M, int K, int N,
                   int64_t stride, void* workspace, bool accumulate, float* split_ws, size_t split_ws_bytes, bool reuse_rows,
                   hipStream_t s, int* deferred_splits, bool split_scales) {
    // split_scales (with reuse_rows): the workspace holds a scale per row and K split (qgemm_f16_act_rows)
    // deferred_splits (optional): where K was split, the partial sums are left in split_ws for the caller's next kernel to
    // fold in (qgemm_f16_reduce_norm_prepare) and their count is returned here; 0 = Y is complete
    // reuse_rows: the workspace already holds these rows of X prepared by the previous call for a matrix of the
    // same type (same rounding rule), so the conversion pass is skipped
    if (ggml_type != PTM_TYPE_Q4_K && ggml_type != PTM_TYPE_Q6_K) return PTM_E_UNSUPPORTED;
    const int blk = ggml_type == PTM_TYPE_Q4_K ? 144 : 210;
    const int rc = qgemm_check(W, X, Y, M, K, N, stride, blk);
    if (rc != PTM_OK) return rc;
    if (!workspace) return PTM_E_NULL;
    if (!aligned16(workspace)) return PTM_E_ALIGN;
    if (ggml_type == PTM_TYPE_Q4_K ? (!aligned16(W) || (stride & 15)) : ((stride & 1) || (reinterpret_cast<uintptr_t>(W) & 1u)))
        return PTM_E_ALIGN;
    const int mp = qf_mpad(M);
    if (mp / 32 > 65535) return PTM_E_UNSUPPORTED;
    _Float16* Xh = static_cast<_Float16*>(workspace);
    float* rowscale = reinterpret_cast<float*>(Xh + (int64_t)mp * K);
    const int nblk = K / 256;
    const int bps = qgemm_f16_blocks_per_split(N, K, M, split_ws ? split_ws_bytes : 0);
    const int splits = (nblk + bps - 1) / bps;  // no empty split
    const int scale_stride = split_scales ? mp : 0;
    float* partials = splits > 1 ? split_ws : nullptr;
    const int acc = accumulate ? 1 : 0;
    const bool q4 = ggml_type == PTM_TYPE_Q4_K;
    if (!reuse_rows) {
        if (q4 && x_is_f32) hipLaunchKernelGGL((qgemm_prepare_rows_f16_kernel<true, true>), dim3(mp), dim3(256), 0, s, X, Xh, rowscale, M, K);
        else if (q4) hipLaunchKernelGGL((qgemm_prepare_rows_f16_kernel<true, false>), dim3(mp), dim3(256), 0, s, X, Xh, rowscale, M, K);
        else if (x_is_f32) hipLaunchKernelGGL((qgemm_prepare_rows_f16_kernel<false, true>), dim3(mp), dim3(256), 0, s, X, Xh, rowscale, M, K);
        else hipLaunchKernelGGL((qgemm_prepare_rows_f16_kernel<false, false>), dim3(mp), dim3(256), 0, s, X, Xh, rowscale, M, K);
    }
    const int wide = (N + QF_TN - 1) / QF_TN * splits;
    const bool flat = q4 && splits == 1 && qf_flat(M, K, wide);
    const bool narrow = !flat && qf_narrow(M, wide);
    const int MT = M <= 32 ? 1 : M <= 64 || narrow || flat ? 2 : 4;  // tiles of 32 rows
    const int tm = 32 * MT;
    const size_t lds = 2 * (size_t)tm * QF_PITCH + 4 * (size_t)tm;  // two X tiles (64 rows: 66 KB) and the row scales: above the default 64 KB cap of dynamic LDS
    static std::once_flag raised;  // two host threads may get here at once: the second waits until the caps are raised
    std::call_once(raised, [] {
        const int small = 2 * 64 * QF_PITCH + 4 * 64;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_short_kernel<Q4Tile, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)qf_short_lds(4));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_short_kernel<Q6Tile, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)qf_short_lds(4));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_rows_kernel<Q4Tile>), hipFuncAttributeMaxDynamicSharedMemorySize, QF_ROWS_LDS);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_rows_kernel<Q6Tile>), hipFuncAttributeMaxDynamicSharedMemorySize, QF_ROWS_LDS);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_kernel<Q4Tile, 2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, small);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_kernel<Q6Tile, 2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, small);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_kernel<Q4Tile, 2, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, small);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_kernel<Q6Tile, 2, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, small);
    });
    const int tn = narrow ? 128 : QF_TN;
    const dim3 grid((N + tn - 1) / tn, (M + tm - 1) / tm, splits);
    const uint8_t* Wb = static_cast<const uint8_t*>(W);
    // 256 columns run with eight waves (two per SIMD, one 32-column strip each): against four waves owning two strips each, 512 x 4096 x
    // 14336 104 -> 92 us (128 rows), 512 x 4096 x 4096 59.8 -> 45.3 us and 96 x 4096 x 2560 57.0 -> 42.7 us (64 rows).  128 columns have
    // four waves of one strip.
    if (qf_short(M, bps)) {
        const size_t short_lds = qf_short_lds(bps);
#define PTM_QS(TILE, NB) hipLaunchKernelGGL((qgemm_f16_short_kernel<TILE, NB>), dim3(grid.x * grid.z), dim3(256), short_lds, s, Wb, stride, Xh, rowscale, Y, M, K, N, acc, bps, partials, scale_stride)
        if (q4) {
            if (bps == 1) PTM_QS(Q4Tile, 1);
            else if (bps == 2) PTM_QS(Q4Tile, 2);
            else if (bps == 3) PTM_QS(Q4Tile, 3);
            else PTM_QS(Q4Tile, 4);
        } else {
            if (bps == 1) PTM_QS(Q6Tile, 1);
            else if (bps == 2) PTM_QS(Q6Tile, 2);
            else if (bps == 3) PTM_QS(Q6Tile, 3);
            else PTM_QS(Q6Tile, 4);
        }
#undef PTM_QS
    } else if (MT == 4) {
        int tall;
        qf_tall(grid.x, splits, M, q4, &tall);
#define PTM_QR(TILE) hipLaunchKernelGGL((qgemm_f16_rows_kernel<TILE>), dim3(qf_workgroups(grid.x, splits, M, tall)), dim3(512), QF_ROWS_LDS, s, Wb, stride, Xh, rowscale, Y, M, K, N, acc, bps, partials, scale_stride, tall)
        if (q4) PTM_QR(Q4Tile);
        else PTM_QR(Q6Tile);
#undef PTM_QR
    } else {
#define PTM_QF(TILE, MTV, WV) hipLaunchKernelGGL((qgemm_f16_kernel<TILE, MTV, WV>), grid, dim3(64 * WV), lds, s, Wb, stride, Xh, rowscale, Y, M, K, N, acc, bps, partials, scale_stride)
    if (q4) {
        if (MT == 2 && narrow) PTM_QF(Q4Tile, 2, 4);
        else if (MT == 2) PTM_QF(Q4Tile, 2, 8);
        else PTM_QF(Q4Tile, 1, 4);
    } else {
        if (MT == 2 && narrow) PTM_QF(Q6Tile, 2, 4);
        else if (MT == 2) PTM_QF(Q6Tile, 2, 8);
        else PTM_QF(Q6Tile, 1, 4);
    }
#undef PTM_QF
    }
    if (deferred_splits) *deferred_splits = partials ? splits : 0;
    if (partials && !deferred_splits) {
        const int64_t total = (int64_t)M * N;
        hipLaunchKernelGGL(qgemm_split_reduce_kernel, dim3((unsigned)((total + 1023) / 1024)), dim3(256), 0, s, partials, splits,
                           Y, total, acc);
    }
    return launch_status();
}

// X (+)= the `splits` partial sums a deferred qgemm_f16_impl left in P, then RMSNorm(X; gamma) into the row workspaces
// (ws_round for Q4_K matrices, ws_plain for Q6_K ones; either may be NULL), as qgemm_f16_prepare_fused(1, ...) fills them.
int qgemm_f16_reduce_norm_prepare(const float* P, int splits, float* X, bool accumulate, const float* gamma, float eps,
                                  int add_one, void* ws_round, void* ws_plain, int M, int K, hipStream_t s) {
    if (!P || !X || !gamma || (!ws_round && !ws_plain)) return PTM_E_NULL;
    if (M <= 0 || K <= 0 || (K % 256) != 0 || splits < 1) return PTM_E_SHAPE;
    if (K > 12288) return PTM_E_UNSUPPORTED;  // the row is staged in LDS (48 KB, within the default cap)
    if (!aligned16(P) || !aligned16(X) || !aligned16(gamma) || !aligned16(ws_round) || !aligned16(ws_plain)) return PTM_E_ALIGN;
    const int mp = qf_mpad(M);
    _Float16* hr = static_cast<_Float16*>(ws_round);
    _Float16* hp = static_cast<_Float16*>(ws_plain);
    float* rr = hr ? reinterpret_cast<float*>(hr + (int64_t)mp * K) : nullptr;
    float* rp = hp ? reinterpret_cast<float*>(hp + (int64_t)mp * K) : nullptr;
#define PTM_RN(B, T) hipLaunchKernelGGL((qgemm_reduce_norm_prepare_kernel<B, T>), dim3(M), dim3(T), (size_t)K * 4, s, P, splits, X, accumulate ? 1 : 0, gamma, eps, add_one, hr, rr, hp, rp, M, K)
    // up to 128 rows the launch lasts as long as one row's chain of requests: as many threads as the row has pieces (4 / 8 / 16 slabs of 2560
    // values 9.4 -> 6.5 us).  Beyond, 512 (953 rows of 4096, two slabs: 256 threads 22.6 us, 512 20.8, 1024 22.3; 509 of 2560, six: 12.1,
    // 11.6, 13.5)
    if (M <= 128 && K > 2048) PTM_RN(16, 1024);
    else if (M <= 128 && K > 1024) PTM_RN(16, 512);
    else if (splits <= 4) PTM_RN(4, 512);
    else PTM_RN(8, 512);
#undef PTM_RN
    return launch_status();
}

// Y[i] = X . W[i]^T for up to three Q4_K / Q6_K matrices over the same K whose rows are already prepared (ws_round for the
// Q4_K ones, ws_plain for the Q6_K ones, as qgemm_f16_prepare_fused leaves them), in one launch plus one reduction.
size_t qgemm_f16_multi_split_bytes(int n, const int* N, const uint32_t* types, int K, int M) {
    int sp[3];
    qgemm_f16_multi_plan(n, N, types, K, M, sp);
    size_t e = 0;
    for (int i = 0; i < n; ++i) if (sp[i] > 1) e += (size_t)sp[i] * M * N[i];
    return 4 * e;
}

// deferred_P / deferred_splits (optional, n entries each): instead of the reduction launch, where matrix i's partial sums lie
// (its finished rows Y[i] when it was not split) and how many slabs there are, for the caller's next kernel to fold in.
int qgemm_f16_multi(int n, const uint32_t* types, const void* const* W, const int64_t* strides, const int* N, float* const* Y,
                    int M, int K, void* ws_round, void* ws_plain, float* split_ws, size_t split_ws_bytes, hipStream_t s,
                    const float** deferred_P, int* deferred_splits) {
    if (n < 1 || n > 3) return PTM_E_SHAPE;
    if (M <= 0 || K <= 0 || (K % 256) != 0) return PTM_E_SHAPE;
    const int mp = qf_mpad(M);
    if (mp / 128 > 65535) return PTM_E_UNSUPPORTED;
    if (qgemm_f16_multi_split_bytes(n, N, types, K, M) > split_ws_bytes || !split_ws) return PTM_E_SHAPE;
    int sp[3];
    qgemm_f16_multi_plan(n, N, types, K, M, sp);
    const int nblk = K / 256;
    int wide = 0, most = 0;  // super-blocks of the longest split
    for (int i = 0; i < n; ++i) most = (nblk + sp[i] - 1) / sp[i] > most ? (nblk + sp[i] - 1) / sp[i] : most;
    for (int i = 0; i < n; ++i) wide += (N[i] + QF_TN - 1) / QF_TN * sp[i];
    const bool narrow = qf_narrow(M, wide);
    const int tn = narrow ? 128 : QF_TN;
    QfMulti a{};
    QfRedMulti r{};
    a.n_mat = n;
    int slots = 0, red_blocks = 0;
    float* part = split_ws;
    // the Q6_K matrices first: their workgroups take longest and should be the first ones placed
    int order[3], k = 0;
    for (int i = 0; i < n; ++i) if (types[i] == PTM_TYPE_Q6_K) order[k++] = i;
    for (int i = 0; i < n; ++i) if (types[i] != PTM_TYPE_Q6_K) order[k++] = i;
    for (int o = 0; o < n; ++o) {
        const int i = order[o];
        const bool q6 = types[i] == PTM_TYPE_Q6_K;
        if (!q6 && types[i] != PTM_TYPE_Q4_K) return PTM_E_UNSUPPORTED;
        void* ws = q6 ? ws_plain : ws_round;
        if (!W[i] || !Y[i] || !ws) return PTM_E_NULL;
        if (N[i] <= 0 || strides[i] < (int64_t)nblk * (q6 ? 210 : 144)) return PTM_E_SHAPE;
        if (q6 ? ((strides[i] & 1) || (reinterpret_cast<uintptr_t>(W[i]) & 1u)) : (!aligned16(W[i]) || (strides[i] & 15))) return PTM_E_ALIGN;
        if (!aligned16(ws) || (reinterpret_cast<uintptr_t>(Y[i]) & 15u)) return PTM_E_ALIGN;
        QfMat& m = a.m[o];
        m.W = static_cast<const uint8_t*>(W[i]);
        m.stride = strides[i];
        m.Xh = static_cast<const _Float16*>(ws);
        m.rowscale = reinterpret_cast<const float*>(m.Xh + (int64_t)mp * K);
        m.Y = Y[i];
        m.N = N[i];
        m.bps = (nblk + sp[i] - 1) / sp[i];
        const int splits = (nblk + m.bps - 1) / m.bps;  // no empty split
        m.ntiles = (N[i] + tn - 1) / tn;
        m.q6 = q6 ? 1 : 0;
        m.partials = splits > 1 ? part : nullptr;
        if (deferred_P) { deferred_P[i] = splits > 1 ? part : Y[i]; deferred_splits[i] = splits; }
        slots += m.ntiles * splits;
        m.slot_end = slots;
        if (splits > 1) {
            QfRedSeg& g = r.s[r.n++];
            g.P = part;
            g.Y = Y[i];
            g.total = (int64_t)M * N[i];
            g.splits = splits;
            red_blocks += (int)((g.total + 1023) / 1024);
            g.blk_end = red_blocks;
            part += (size_t)splits * M * N[i];
        }
    }
    static std::once_flag raised;
    std::call_once(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_rows_multi_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, QF_ROWS_LDS);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_multi_kernel<4, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, QF_ROWS_LDS);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_short_multi_kernel<4>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)qf_short_lds(QF_SHORT_BLOCKS));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_multi_kernel<2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  2 * 64 * QF_PITCH + 4 * 64);
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&qgemm_f16_multi_kernel<2, 4>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  2 * 64 * QF_PITCH + 4 * 64);
    });
    if (qf_short(M, most) && most <= 2)
        hipLaunchKernelGGL(qgemm_f16_short_multi_kernel<2>, dim3(slots), dim3(256), qf_short_lds(most), s, a, M, K);
    else if (qf_short(M, most))
        hipLaunchKernelGGL(qgemm_f16_short_multi_kernel<4>, dim3(slots), dim3(256), qf_short_lds(most), s, a, M, K);
    else if (M <= 32)
        hipLaunchKernelGGL((qgemm_f16_multi_kernel<1, 4>), dim3(slots, 1), dim3(256), 2 * (size_t)32 * QF_PITCH + 4 * 32, s, a, M, K);
    else if (narrow)
        hipLaunchKernelGGL((qgemm_f16_multi_kernel<2, 4>), dim3(slots, (M + 63) / 64), dim3(256), 2 * (size_t)64 * QF_PITCH + 4 * 64, s, a, M, K);
    else if (M <= 64)
        hipLaunchKernelGGL((qgemm_f16_multi_kernel<2, 8>), dim3(slots, 1), dim3(512), 2 * (size_t)64 * QF_PITCH + 4 * 64, s, a, M, K);
    else {
        bool q4 = true;
        for (int i = 0; i < n; ++i) q4 = q4 && types[i] == PTM_TYPE_Q4_K;
        int tall;
        qf_tall(slots, 1, M, q4, &tall);
        // without a tall tile, the kernel that has none: 44 and 88 workgroups of 1024 values 15.0 and 16.1 us with all of them in it, 14.8 and 15.8 so
        if (tall == 0) hipLaunchKernelGGL((qgemm_f16_multi_kernel<4, 8>), dim3(slots, (M + 127) / 128), dim3(512), QF_ROWS_LDS, s, a, M, K);
        else hipLaunchKernelGGL(qgemm_f16_rows_multi_kernel, dim3(qf_workgroups(slots, 1, M, tall)), dim3(512), QF_ROWS_LDS, s, a, M, K, slots, tall);
    }
    if (r.n > 0 && !deferred_P) hipLaunchKernelGGL(qgemm_split_reduce_multi_kernel, dim3(red_blocks), dim3(256), 0, s, r);
    return launch_status();
}

// Fills the row workspaces of qgemm_f16_impl (call it with reuse_rows afterwards): pre 1 = RMSNorm(X; gamma = X2), pre 2 =
// SiLU(X) * X2.  ws_round serves Q4_K matrices, ws_plain Q6_K ones; either may be NULL.
int qgemm_f16_prepare_fused(int pre, const float* X, const float* X2, float eps, int add_one, void* ws_round, void* ws_plain,
                            int M, int K, hipStream_t s) {
    if (!X || !X2 || (!ws_round && !ws_plain)) return PTM_E_NULL;
    if (M <= 0 || K <= 0 || (K % 256) != 0) return PTM_E_SHAPE;
    if (!aligned16(X) || !aligned16(X2) || !aligned16(ws_round) || !aligned16(ws_plain)) return PTM_E_ALIGN;
    const int mp = qf_mpad(M);
    _Float16* hr = static_cast<_Float16*>(ws_round);
    _Float16* hp = static_cast<_Float16*>(ws_plain);
    float* rr = hr ? reinterpret_cast<float*>(hr + (int64_t)mp * K) : nullptr;
    float* rp = hp ? reinterpret_cast<float*>(hp + (int64_t)mp * K) : nullptr;
    if (pre == 1) hipLaunchKernelGGL(qgemm_prepare_fused_kernel<1>, dim3(mp), dim3(256), 0, s, X, X2, eps, add_one, hr, rr, hp, rp, M, K);
    else if (pre == 2) hipLaunchKernelGGL(qgemm_prepare_fused_kernel<2>, dim3(mp), dim3(1024), 0, s, X, X2, eps, add_one, hr, rr, hp, rp, M, K);
    else return PTM_E_UNSUPPORTED;
    return launch_status();
}

// Fills a row workspace of K values with SiLU(gate) . up of M rows that are still G[sg] / U[su] slabs, a scale per row and K split of bps
// super-blocks (the workspace has room for QF_MAX_SPLITS scales a row).
bool qgemm_f16_act_rows_fit(int bps, int M, int K) { return M <= 65535 && bps * 256 <= ACT_CHUNK && (K / 256 + bps - 1) / bps <= QF_MAX_SPLITS; }
int qgemm_f16_act_rows(const float* G, const float* U, int sg, int su, bool gelu, bool rounded, void* ws, int bps, int M, int K, hipStream_t s) {
    if (!G || !U || !ws) return PTM_E_NULL;
    if (M <= 0 || K <= 0 || (K % 256) != 0 || sg < 1 || su < 1 || bps < 1) return PTM_E_SHAPE;
    if (!qgemm_f16_act_rows_fit(bps, M, K)) return PTM_E_UNSUPPORTED;
    if (!aligned16(G) || !aligned16(U) || !aligned16(ws)) return PTM_E_ALIGN;
    const int mp = qf_mpad(M), splits = (K / 256 + bps - 1) / bps;
    _Float16* rows = static_cast<_Float16*>(ws);
    hipLaunchKernelGGL(qgemm_act_rows_kernel, dim3(splits, M), dim3(256), 0, s, G, U, sg, su, gelu ? 1 : 0, rounded ? 1 : 0, rows,
                       reinterpret_cast<float*>(rows + (int64_t)mp * K), mp, bps * 256, M, K);
    return launch_status();
}

}  // namespace ptm

using namespace ptm;

extern "C" {

int64_t ptm_qgemm_workspace_bytes(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const int64_t mp = qg_mpad(M);
    return mp * K + 2 * (int64_t)(K / 32) * mp * 4;
}

int ptm_qgemm_q4k(const void* W, const void* X_bf16, float* Y, int M, int K, int N, int64_t stride, void* workspace,
                  ptm_stream_t stream) {
    int rc = qgemm_check(W, X_bf16, Y, M, K, N, stride, 144);
    if (rc != PTM_OK) return rc;
    if (!workspace) return PTM_E_NULL;
    if (!aligned16(W) || (stride & 15) || !aligned16(workspace)) return PTM_E_ALIGN;
    const int mp = qg_mpad(M);
    int8_t* qs = static_cast<int8_t*>(workspace);
    float* dT = reinterpret_cast<float*>(qs + (int64_t)mp * K);
    float* sT = dT + (int64_t)(K / 32) * mp;
    hipStream_t s = as_stream(stream);
    hipLaunchKernelGGL(qgemm_quantize_rows_kernel, dim3(mp), dim3(256), 0, s, static_cast<const uint16_t*>(X_bf16), qs, dT,
                       sT, M, mp, K);
    if ((rc = launch_status()) != PTM_OK) return rc;
    const dim3 grid((N + QG_NBLOCK - 1) / QG_NBLOCK, mp / QG_MCHUNK);
    hipLaunchKernelGGL(qgemm_q4k_kernel, grid, dim3(256), 0, s, static_cast<const uint8_t*>(W), stride, qs, dT, sT, Y, M, mp,
                       K, N);
    return launch_status();
}

int ptm_qgemm_q6k(const void* W, const void* X_bf16, float* Y, int M, int K, int N, int64_t stride, void* workspace,
                  ptm_stream_t stream) {
    (void)workspace;  // Q6_K consumes the bf16 activations directly
    const int rc = qgemm_check(W, X_bf16, Y, M, K, N, stride, 210);
    if (rc != PTM_OK) return rc;
    if ((stride & 1) || (reinterpret_cast<uintptr_t>(W) & 1u)) return PTM_E_ALIGN;
    const int mp = qg_mpad(M);
    const dim3 grid((N + QG_NBLOCK - 1) / QG_NBLOCK, mp / QG_MCHUNK);
    hipLaunchKernelGGL(qgemm_q6k_kernel, grid, dim3(256), 0, as_stream(stream), static_cast<const uint8_t*>(W), stride,
                       static_cast<const uint16_t*>(X_bf16), Y, M, K, N);
    return launch_status();
}

int64_t ptm_qgemm_f16_workspace_bytes(int M, int K) {
    if (M <= 0 || K <= 0) return 0;
    const int64_t mp = qf_mpad(M);
    return mp * K * 2 + mp * 4;
}

int ptm_qgemm_f16(uint32_t ggml_type, const void* W, const void* X_bf16, float* Y, int M, int K, int N, int64_t stride,
                  void* workspace, ptm_stream_t stream) {
    return qgemm_f16_impl(ggml_type, W, X_bf16, false, Y, M, K, N, stride, workspace, false, nullptr, 0, false, as_stream(stream),
                          nullptr, false);
}

int64_t ptm_qgemm_f16_f32_workspace_bytes(int M, int K, int N) {
    if (M <= 0 || K <= 0 || N <= 0) return 0;
    const int64_t base = (ptm_qgemm_f16_workspace_bytes(M, K) + 255) & ~(int64_t)255;
    const int splits = qgemm_f16_splits(N, K, M);
    return base + (splits > 1 ? (int64_t)splits * M * N * 4 : 0);
}

int ptm_qgemm_f16_f32(uint32_t ggml_type, const void* W, const float* X_f32, float* Y, int M, int K, int N, int64_t stride,
                      void* workspace, int accumulate, ptm_stream_t stream) {
    if (M <= 0 || K <= 0 || N <= 0) return PTM_E_SHAPE;
    if (!workspace) return PTM_E_NULL;
    const int64_t base = (ptm_qgemm_f16_workspace_bytes(M, K) + 255) & ~(int64_t)255;
    const int splits = qgemm_f16_splits(N, K, M);
    return qgemm_f16_impl(ggml_type, W, X_f32, true, Y, M, K, N, stride, workspace, accumulate != 0,
                          splits > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + base) : nullptr,
                          splits > 1 ? (size_t)splits * M * N * 4 : 0, false, as_stream(stream), nullptr, false);
}

}  // extern "C"
