// The GEMV dispatcher's other block formats: Q8_0 (34 B per 32 values), Q5_K (176 B per 256) and Q5_0 (22 B per 32),
// fp32 activations, as the reference's q8_0_gemv_avx2 / q5k_gemv_avx2 / q5_0_gemv_scalar compute them
// (torch/io/cpu_quant_gemv.h:784-826, :1091-1185, :1572-1630), and the dequantisers of the first two
// (torch/io/gguf_dequant.h:237-255, :348-388).
//
// slots_gemv_kernel: a lane takes 8 values of a row (16 of a Q5_K block: both nibbles of its bytes) at a time, so that neighbouring lanes read
// neighbouring pieces of x and of the row, and a wave several rows, so that x is loaded once for all of them; two passes over the row are
// requested together; split_gemv_kernel: a wave per pass.  Bound by requests in flight: Q8_0 with weights from HBM, in a graph, 9728 x 2560 7.9 us = 3.3 TB/s
// (two passes at a time 8.7), 30000 x 2560 19.5 us = 4.2 TB/s with two passes at a time, 500 x 1024 2.3 us (19.1, 50.1 and 2.6 with a lane per run of 32 values, as the exact Q4_K kernel below still has it: x and the
// row are then read in pieces 128 and 34 bytes apart, and every load instruction touches 64 cache lines); 9728 x 2560 called again and again on
// weights that the caches hold 6.1 us (6.6; 18.1).
#include "ptm_common.h"

#include <type_traits>

namespace ptm {

struct __attribute__((packed, aligned(2))) u32_a2 { uint32_t v; };

struct __attribute__((packed, aligned(2))) u64_a2 { uint32_t lo, hi; };

__device__ __forceinline__ void load8(const float* __restrict__ x, float (&v)[8]) {
    const float4 a = *reinterpret_cast<const float4*>(x), b = *reinterpret_cast<const float4*>(x + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}

// A format: VALUES of a row per slot; where waves share rows ROWS per wave of 2048 rows and more, FEW of 1024 to 2047; whether fewer than 2048 rows,
// too, have a wave for each pass (slots_launch); what a lane loads of the row for slot u, which values of x (two groups of 8 or 4), the slot's term.
struct FmtQ8_0 {
    static constexpr int BLOCK_BYTES = 34, VALUES = 8, ROWS = 4, FEW = 2;
    static constexpr bool SPLIT_FEW = false;
    struct Raw { u64_a2 q; uint32_t d; };
    struct X { float v[8]; };
    static __device__ __forceinline__ void load(const uint8_t* __restrict__ row, int u, Raw& r) {
        const uint8_t* p = row + (int64_t)(u >> 2) * 34;
        r.q = *reinterpret_cast<const u64_a2*>(p + 2 + 8 * (u & 3));
        r.d = reinterpret_cast<const u16_a2*>(p)->v;
    }
    static __device__ __forceinline__ void load_x(const float* __restrict__ x, int u, X& o) { load8(x + 8 * u, o.v); }
    static __device__ __forceinline__ float term(const Raw& r, const X& x, int) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = fmaf((float)(int8_t)((r.q.lo >> (8 * i)) & 0xffu), x.v[i], s);
            s = fmaf((float)(int8_t)((r.q.hi >> (8 * i)) & 0xffu), x.v[4 + i], s);
        }
        return h2f(r.d) * s;
    }
    static __device__ __forceinline__ float value(const uint8_t* __restrict__ blocks, int64_t e) {
        const uint8_t* p = blocks + (e >> 5) * 34;
        return h2f(reinterpret_cast<const u16_a2*>(p)->v) * (float)(int8_t)p[2 + (e & 31)];
    }
};

struct FmtQ5_0 {
    static constexpr int BLOCK_BYTES = 22, VALUES = 8, ROWS = 2, FEW = 1;  // four low nibbles and the four high ones of the same bytes, 16 values on
    static constexpr bool SPLIT_FEW = false;
    struct Raw { uint32_t q, h, d; };
    struct X { float v[8]; };
    static __device__ __forceinline__ void load(const uint8_t* __restrict__ row, int u, Raw& r) {
        const uint8_t* p = row + (int64_t)(u >> 2) * 22;
        r.q = reinterpret_cast<const u32_a2*>(p + 6 + 4 * (u & 3))->v;
        r.h = reinterpret_cast<const u32_a2*>(p + 2)->v;
        r.d = reinterpret_cast<const u16_a2*>(p)->v;
    }
    static __device__ __forceinline__ void load_x(const float* __restrict__ x, int u, X& o) {
        const float* p = x + 32 * (u >> 2) + 4 * (u & 3);
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 16);
        o.v[0] = a.x; o.v[1] = a.y; o.v[2] = a.z; o.v[3] = a.w;
        o.v[4] = b.x; o.v[5] = b.y; o.v[6] = b.z; o.v[7] = b.w;
    }
    static __device__ __forceinline__ float term(const Raw& r, const X& x, int u) {
        // four values at a time: the fifth bits spread to their bytes (times 1 + 2^7 + 2^14 + 2^21), 16 subtracted within each byte, which the conversion
        // then takes with its sign (9728 x 2560 7.5 -> 6.4 us; byte by byte a value was eight instructions, so it is four)
        const uint32_t h = r.h >> (4 * (u & 3));
        auto less16 = [](uint32_t nibbles, uint32_t high) {
            return (((nibbles & 0x0f0f0f0fu) | (((high & 0xfu) * 0x00204081u) & 0x01010101u) << 4 | 0x80808080u) - 0x10101010u) ^ 0x80808080u;
        };
        const uint32_t lo = less16(r.q, h), hi = less16(r.q >> 4, h >> 16);
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = fmaf((float)(int8_t)((lo >> (8 * i)) & 0xffu), x.v[i], s);
            s = fmaf((float)(int8_t)((hi >> (8 * i)) & 0xffu), x.v[4 + i], s);
        }
        return h2f(r.d) * s;
    }
};

struct FmtQ5_K {
    static constexpr int BLOCK_BYTES = 176, VALUES = 16, ROWS = 4, FEW = 2;  // eight low nibbles and the eight high ones of the same bytes, 32 values on
    static constexpr bool SPLIT_FEW = true;
    struct Raw { uint4 hdr; uint2 q, h; };
    struct X { float lo[8], hi[8]; };
    // scale and min of sub-block sb from the 12 packed bytes at p + 4 (get_scale_min_k4, gguf_dequant.h:289-297)
    static __device__ __forceinline__ void scale_min(const uint8_t* __restrict__ p, int sb, int& sc, int& mn) {
        const uint32_t* s = reinterpret_cast<const uint32_t*>(p + 4);
        q4k_scale_min(s[0], s[1], s[2], sb, sc, mn);
    }
    // slot u: bytes 8 (u % 4) .. of the pair of sub-blocks u / 4 % 4 of block u / 16.  Rows are aligned to 4 bytes.
    struct __attribute__((packed, aligned(4))) u128_a4 { uint32_t v[4]; };
    static __device__ __forceinline__ void load(const uint8_t* __restrict__ row, int u, Raw& r) {
        const uint8_t* p = row + (int64_t)(u >> 4) * 176;
        const int at = 8 * (u & 3), pair = (u >> 2) & 3;
        const u128_a4 h = *reinterpret_cast<const u128_a4*>(p);
        const uint32_t* q = reinterpret_cast<const uint32_t*>(p + 48 + 32 * pair + at);
        const uint32_t* b = reinterpret_cast<const uint32_t*>(p + 16 + at);
        r.hdr = make_uint4(h.v[0], h.v[1], h.v[2], h.v[3]);
        r.q = make_uint2(q[0], q[1]);
        r.h = make_uint2(b[0], b[1]);
    }
    static __device__ __forceinline__ void load_x(const float* __restrict__ x, int u, X& o) {
        const float* p = x + 256 * (u >> 4) + 64 * ((u >> 2) & 3) + 8 * (u & 3);
        load8(p, o.lo);
        load8(p + 32, o.hi);
    }
    static __device__ __forceinline__ float term(const Raw& r, const X& x, int u) {
        const int pair = (u >> 2) & 3;
        float out = 0.0f;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            int sc, mn;
            q4k_scale_min(r.hdr.y, r.hdr.z, r.hdr.w, 2 * pair + e, sc, mn);
            const uint32_t q0 = ((r.q.x >> (4 * e)) & 0x0f0f0f0fu) | (((r.h.x >> (2 * pair + e)) & 0x01010101u) << 4);
            const uint32_t q1 = ((r.q.y >> (4 * e)) & 0x0f0f0f0fu) | (((r.h.y >> (2 * pair + e)) & 0x01010101u) << 4);
            const float* v = e ? x.hi : x.lo;
            float sq = 0.0f, sx = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sq = fmaf((float)((q0 >> (8 * i)) & 0xffu), v[i], sq);
                sq = fmaf((float)((q1 >> (8 * i)) & 0xffu), v[4 + i], sq);
                sx += v[i] + v[4 + i];
            }
            out += fmaf(h2f(r.hdr.x) * (float)sc, sq, -((h2f(r.hdr.x >> 16) * (float)mn) * sx));
        }
        return out;
    }
    static __device__ __forceinline__ float value(const uint8_t* __restrict__ blocks, int64_t e) {
        const uint8_t* p = blocks + (e >> 8) * 176;
        const int r = (int)(e & 255), sb = r >> 5, pair = sb >> 1, hi = sb & 1, l = r & 31;
        const uint32_t dd = *reinterpret_cast<const uint32_t*>(p);
        int sc, mn;
        scale_min(p, sb, sc, mn);
        const float ds = h2f(dd) * (float)sc, ms = h2f(dd >> 16) * (float)mn;
        const uint32_t b = p[48 + 32 * pair + l];
        const int q = (int)((hi ? (b >> 4) : (b & 0xfu)) + (((p[16 + l] >> (2 * pair + hi)) & 1u) ? 16u : 0u));
        return ds * (float)q - ms;   // as the reference: d1 * q - m1, two roundings
    }
};

// Q4_K with fp32 activations, as the reference computes it where it has no AVX2 (q4k_gemv_scalar, cpu_quant_gemv.h:689-767):
// every weight is dequantised as fma(d * sc, q, -(dmin * m)) and multiplied with x, no Q8 rounding of the activations.
// The exact-math cross-check of the Q8-activation kernel, not a path of the decoder.  Run u is sub-block u & 7 of
// super-block u >> 3: 32 nibbles of one 32-byte group (low nibbles for even, high for odd sub-blocks).
struct FmtQ4_K_F32 {
    static constexpr int BLOCK_BYTES = 144;
    static __device__ __forceinline__ float term(const uint8_t* __restrict__ row, int u, const float* __restrict__ x) {
        const int sb = u & 7, hi = sb & 1;
        const uint8_t* p = row + (int64_t)(u >> 3) * 144;
        const uint4 hdr = *reinterpret_cast<const uint4*>(p);
        int sc, mn;
        q4k_scale_min(hdr.y, hdr.z, hdr.w, sb, sc, mn);
        const float d1 = h2f(hdr.x) * (float)sc, m1 = h2f(hdr.x >> 16) * (float)mn;
        const uint8_t* qs = p + 16 + 32 * (sb >> 1);
        const float* xb = x + 32 * u;
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) {
            const uint32_t q = (*reinterpret_cast<const uint32_t*>(qs + 4 * w) >> (4 * hi)) & 0x0f0f0f0fu;
            const float4 xv = *reinterpret_cast<const float4*>(xb + 4 * w);
            s = fmaf(fmaf(d1, (float)(q & 0xffu), -m1), xv.x, s);
            s = fmaf(fmaf(d1, (float)((q >> 8) & 0xffu), -m1), xv.y, s);
            s = fmaf(fmaf(d1, (float)((q >> 16) & 0xffu), -m1), xv.z, s);
            s = fmaf(fmaf(d1, (float)(q >> 24), -m1), xv.w, s);
        }
        return s;
    }
};

// y[r] (+)= sum over the row's runs of 32; one wave per row, four rows per workgroup
template <typename Fmt, bool ACC>
__global__ __launch_bounds__(256) void rowwave_gemv_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x,
                                                           float* __restrict__ y, int K, int N, int64_t stride) {
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= N) return;  // wave-uniform
    const uint8_t* row = W + (int64_t)r * stride;
    const int units = K / 32;
    float acc = 0.0f;
    for (int u = lane; u < units; u += 64) acc += Fmt::term(row, u, x);
    acc = sum64(acc);
    if (lane == 0) {
        if constexpr (ACC) y[r] += acc;
        else y[r] = acc;
    }
}

// y[r] (+)= the row's terms; R rows per wave, four waves per workgroup, C of them (1 or 4) at the same rows, U passes over a row requested together
template <typename Fmt, int R, int C, int U, bool ACC>
__global__ __launch_bounds__(256) void slots_gemv_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x, float* __restrict__ y,
                                                         int K, int N, int64_t stride) {
    __shared__ float part[4][R];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r0 = (blockIdx.x * (4 / C) + wave / C) * R;
    if (r0 >= N) return;  // a whole wave, and of C = 4 the whole workgroup
    const uint8_t* row[R];
    float acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        row[i] = W + (int64_t)min(r0 + i, N - 1) * stride;
        acc[i] = 0.0f;
    }
    const int slots = K / Fmt::VALUES;
    // a lane beyond the row repeats the last slot and does not count it
    for (int first = (wave % C) * 64 * U; first < slots; first += 64 * U * C) {
        typename Fmt::X xv[U];
        typename Fmt::Raw w[U][R];
#pragma unroll
        for (int p = 0; p < U; ++p) {
            const int u = min(first + 64 * p + lane, slots - 1);
            Fmt::load_x(x, u, xv[p]);
#pragma unroll
            for (int i = 0; i < R; ++i) Fmt::load(row[i], u, w[p][i]);
        }
#pragma unroll
        for (int p = 0; p < U; ++p) {
            const int at = first + 64 * p + lane, u = min(at, slots - 1);
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const float t = Fmt::term(w[p][i], xv[p], u);
                acc[i] += at < slots ? t : 0.0f;
            }
        }
    }
    float v = sum_rows<R>(acc);
    const int i = sum_row<R>(lane);
    if constexpr (C > 1) {
        if ((lane & (64 / R - 1)) == 0) part[wave][i] = v;
        __syncthreads();
        if (wave > 0) return;
        v = (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]);
    }
    if ((lane & (64 / R - 1)) == 0 && r0 + i < N) y[r0 + i] = ACC ? y[r0 + i] + v : v;
}

// The same for rows of up to SPLIT_PASSES passes: a wave for each pass, all of them at the same R rows, so that nothing is requested twice, no wave is without
// work (2560 values of Q8_0 are five passes: in twos for four waves, the last has none) and x, which goes out first, is read once for R rows.
constexpr int SPLIT_PASSES = 10;
template <typename Fmt, int R, bool ACC>
__global__ __launch_bounds__(64 * SPLIT_PASSES) void split_gemv_kernel(const uint8_t* __restrict__ W, const float* __restrict__ x, float* __restrict__ y,
                                                                       int K, int N, int64_t stride) {
    __shared__ float part[SPLIT_PASSES][R];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r0 = blockIdx.x * R, slots = K / Fmt::VALUES, at = 64 * wave + lane, u = min(at, slots - 1);
    typename Fmt::X xv;
    typename Fmt::Raw w[R];
    Fmt::load_x(x, u, xv);
    issue_order_fence();
#pragma unroll
    for (int i = 0; i < R; ++i) Fmt::load(W + (int64_t)min(r0 + i, N - 1) * stride, u, w[i]);
    float acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const float t = Fmt::term(w[i], xv, u);
        acc[i] = at < slots ? t : 0.0f;  // a lane beyond the row repeats the last slot and does not count it
    }
    const float v = sum_rows<R>(acc);
    if ((lane & (64 / R - 1)) == 0) part[wave][sum_row<R>(lane)] = v;
    __syncthreads();
    const int i = threadIdx.x;
    if (i >= R || r0 + i >= N) return;
    float s = part[0][i];
    for (int c = 1; c < (int)blockDim.x / 64; ++c) s += part[c][i];
    y[r0 + i] = ACC ? y[r0 + i] + s : s;
}

template <typename Fmt>
__global__ __launch_bounds__(256) void elementwise_dequant_kernel(const uint8_t* __restrict__ blocks, float* __restrict__ out,
                                                                  int64_t n) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e < n) out[e] = Fmt::value(blocks, e);
}

template <typename Fmt>
static int gemv_check(const void* W, const float* x, const float* y, int K, int N, int64_t stride, int per_block, int w_align) {
    if (!W || !x || !y) return PTM_E_NULL;
    if (K <= 0 || N <= 0 || (K % per_block) != 0) return PTM_E_SHAPE;
    if (stride < (int64_t)(K / per_block) * Fmt::BLOCK_BYTES) return PTM_E_SHAPE;
    if ((stride % w_align) != 0 || (reinterpret_cast<uintptr_t>(W) % w_align) != 0 || !aligned16(x) ||
        (reinterpret_cast<uintptr_t>(y) & 3u))
        return PTM_E_ALIGN;
    return PTM_OK;
}

template <typename Fmt>
static int slots_launch(const void* W, const float* x, float* y, int K, int N, int64_t stride, int per_block, int w_align,
                        bool accumulate, hipStream_t s) {
    const int rc = gemv_check<Fmt>(W, x, y, K, N, stride, per_block, w_align);
    if (rc != PTM_OK) return rc;
    const uint8_t* w = static_cast<const uint8_t*>(W);
    auto go = [&](auto rows, auto waves, auto passes) {
        constexpr int R = decltype(rows)::value, C = decltype(waves)::value, U = decltype(passes)::value;
        const dim3 grid((N + 4 / C * R - 1) / (4 / C * R)), block(256);
        if (accumulate) hipLaunchKernelGGL((slots_gemv_kernel<Fmt, R, C, U, true>), grid, block, 0, s, w, x, y, K, N, stride);
        else hipLaunchKernelGGL((slots_gemv_kernel<Fmt, R, C, U, false>), grid, block, 0, s, w, x, y, K, N, stride);
    };
    using std::integral_constant;
    constexpr integral_constant<int, 1> one;
    constexpr integral_constant<int, 2> two;
    constexpr integral_constant<int, 4> four;
    // Four waves at the same rows where a row has two requests or more for each of them, more rows to share x between the more rows there are.
    // us for one / two rows a wave, then for one / two / four with four waves at them, Q8_0: 9728 x 2560 12.4 10.4 | 11.2 9.5 9.0, 2560 x 9728
    // 12.6 15.4 | 11.9 10.9 10.5, 1024 x 2560 3.3 3.8 | 3.0 2.9 3.0, 700 x 14336 9.7 13.2 | 5.8 6.6 6.3, 9728 x 1024 5.3 5.0 | 7.2 6.2 5.0.
    // Q5_0 unpacks more per byte, and of 1024 to 2047 rows one a wave leaves fewer waves without work: 1024 x 2048 3.57 us with two, 3.07 with one (a
    // wave per row, 32 values a lane: 3.31), 1280 x 4096 4.75 4.36, 2047 x 2048 3.94 3.73, 2047 x 8192 7.97 8.14.
    // Rows of one pass: a second request would repeat it, Q5_K 2560 x 256 4.0 -> 3.2 us (a wave per row, 32 values a lane: 3.7), 9728 x 1024 7.2 ->
    // 4.8 (9.2), Q8_0 2560 x 512 3.0 -> 2.8 (3.8).
    const int slots = K / Fmt::VALUES, all = (slots + 63) / 64;
    // Three to ten passes, a wave for each.  us as below and so, on weights that the caches hold, Q8_0 9728 x 1536 5.5, 4.5, x 2560 6.6, 6.1, 2048 x 2560 2.8, 2.6,
    // 6000 x 5120 7.1, 6.9, 14336 x 4096 10.3, 10.4, 30000 x 3584 27.3, 24.9 (from HBM 9728 x 2560 8.7, 7.9, 14336 x 4096 15.1, 14.7); Q5_K 9728 x 2560 9.7, 7.2,
    // 2560 x 9728 10.2, 7.7, 30000 x 3584 22.4, 20.0; Q5_0 9728 x 2560 9.8, 6.4, 6000 x 5120 9.8, 7.3.  Of two passes, 9728 x 1024, they are within 2 % (Q5_K x 1536
    // 5.66, 5.71), of fourteen Q8_0 3000 x 7168 5.7, 5.6.  Fewer rows, two a workgroup, are faster for Q5_K alone: 1200 x 4096 3.6, 3.1 (Q8_0 2.9, 3.0),
    // 400 x 10240 3.4, 3.1, 300 x 2560 2.7, 2.3 (2.2, 2.2).
    auto split = [&](auto rows) {
        constexpr int R = decltype(rows)::value;
        const dim3 grid((N + R - 1) / R), block(64 * all);
        if (accumulate) hipLaunchKernelGGL((split_gemv_kernel<Fmt, R, true>), grid, block, 0, s, w, x, y, K, N, stride);
        else hipLaunchKernelGGL((split_gemv_kernel<Fmt, R, false>), grid, block, 0, s, w, x, y, K, N, stride);
    };
    if (all >= 3 && all <= SPLIT_PASSES && (N >= 2048 || Fmt::SPLIT_FEW)) {
        if (N >= 2048) split(four);
        else if constexpr (Fmt::SPLIT_FEW) split(two);
    } else if (slots >= 256) {
        if (N >= 2048) go(integral_constant<int, Fmt::ROWS>{}, four, two);
        else if (N >= 1024) go(integral_constant<int, Fmt::FEW>{}, four, two);
        else go(one, four, two);
    } else if (slots <= 64) {
        if (N >= 2048) go(two, one, one);
        else go(one, one, one);
    } else {
        if (N >= 2048) go(two, one, two);
        else go(one, one, two);
    }
    return launch_status();
}

template <typename Fmt>
static int dequant_launch(const void* blocks, float* out, int64_t n, int per_block, int align, hipStream_t s) {
    if (!blocks || !out) return PTM_E_NULL;
    if (n < 0 || (n % per_block) != 0) return PTM_E_SHAPE;
    if ((reinterpret_cast<uintptr_t>(blocks) % align) != 0 || (reinterpret_cast<uintptr_t>(out) & 3u)) return PTM_E_ALIGN;
    if (n == 0) return PTM_OK;
    if ((n + 255) / 256 > 0x7fffffff) return PTM_E_UNSUPPORTED;
    hipLaunchKernelGGL((elementwise_dequant_kernel<Fmt>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                       static_cast<const uint8_t*>(blocks), out, n);
    return launch_status();
}

}  // namespace ptm

using namespace ptm;

extern "C" {

int ptm_q8_0_gemv(const void* W, const float* x, float* y, int K, int N, int64_t row_stride_bytes, int accumulate,
                  ptm_stream_t stream) {
    return slots_launch<FmtQ8_0>(W, x, y, K, N, row_stride_bytes, 32, 2, accumulate != 0, as_stream(stream));
}

int ptm_q5_0_gemv(const void* W, const float* x, float* y, int K, int N, int64_t row_stride_bytes, int accumulate,
                  ptm_stream_t stream) {
    return slots_launch<FmtQ5_0>(W, x, y, K, N, row_stride_bytes, 32, 2, accumulate != 0, as_stream(stream));
}

int ptm_q5k_gemv(const void* W, const float* x, float* y, int K, int N, int64_t row_stride_bytes, int accumulate,
                 ptm_stream_t stream) {
    return slots_launch<FmtQ5_K>(W, x, y, K, N, row_stride_bytes, 256, 4, accumulate != 0, as_stream(stream));
}

int ptm_q4k_gemv_f32act(const void* W, const float* x, float* y, int K, int N, int64_t row_stride_bytes, int accumulate,
                        ptm_stream_t stream) {
    const int rc = gemv_check<FmtQ4_K_F32>(W, x, y, K, N, row_stride_bytes, 256, 16);
    if (rc != PTM_OK) return rc;
    const dim3 grid((N + 3) / 4), block(256);
    const uint8_t* w = static_cast<const uint8_t*>(W);
    if (accumulate) hipLaunchKernelGGL((rowwave_gemv_kernel<FmtQ4_K_F32, true>), grid, block, 0, as_stream(stream), w, x, y, K, N, row_stride_bytes);
    else hipLaunchKernelGGL((rowwave_gemv_kernel<FmtQ4_K_F32, false>), grid, block, 0, as_stream(stream), w, x, y, K, N, row_stride_bytes);
    return launch_status();
}

int ptm_dequant_q8_0(const void* blocks, float* out, int64_t n, ptm_stream_t stream) {
    return dequant_launch<FmtQ8_0>(blocks, out, n, 32, 2, as_stream(stream));
}

int ptm_dequant_q5k(const void* blocks, float* out, int64_t n, ptm_stream_t stream) {
    return dequant_launch<FmtQ5_K>(blocks, out, n, 256, 4, as_stream(stream));
}

}  // extern "C"
