// Device code of the Q4_K dequant-fused GEMV (see q4k_gemv.hip for the design notes); kept in a
// header so that a launch mixing Q4_K and Q6_K projections can call it per workgroup.
#pragma once
#include <climits>

#include "ptm_common.h"

namespace ptm {

struct Q4KArgs {
    const uint8_t* W[3];
    float* y[3];
    int row_end[3];  // cumulative row counts of the (up to 3) matrices
    int n_mat;
    int total_rows;  // MODE 1: 2*N interleaved (gate row r, up row r)
    int K;
    int log2S;       // lane groups per row = 1 << log2S
    int64_t stride;
    int tiles_per_wg;    // row tiles (of 32 >> log2S rows) a workgroup walks with ONE staging of x (0 or 1: one tile)
    const void* x;       // fp32 x[K] (XQ8 == false) or Q8 blocks (XQ8 == true)
    const float* gamma;  // RMSNorm weight (NORM)
    float eps;
    int add_one;
    int gelu;            // MODE 1: tanh-GELU(gate) * up (gemma) instead of SiLU(gate) * up
    // PRE (with NORM, K <= 4096): the branch output of the previous projection still waits for its post-norm and residual
    // add (gemma's post-attention / post-feed-forward norms, gguf_model.h:3656-3680, :3787-3807).  Every workgroup forms
    // x + RMSNorm(pre_h) * pre_w itself before its own RMSNorm; workgroup 0 also stores that sum to pre_out, which must not
    // be x (other workgroups still read x).
    const float* pre_h;
    const float* pre_w;
    float* pre_out;
};

enum { Q4K_THREADS = 256, Q4K_ONE_WAVES = 10 };

// ---- prologue: bring the Q8 activation into LDS; loads first (q4k_stage_issue), the arithmetic after the
// weight prefetch has been issued (q4k_stage_finish) --------------------------------------------------
// fp32 x of the workgroups that share it among many waves or tiles: thread t takes the 16 bytes at t, t + threads, ... - whole lines per instruction.  What bounds these kernels is how fast a CU's waves get
// their loads out, and an instruction takes a clock for every 64 bytes it touches: with 16 consecutive values a thread (64 bytes apart from lane
// to lane) the eight loads of x and the norm's weights took the time of 32, and the last of 1216 workgroups had its loads out 5.4 us behind the first.
template <int NX>
struct Q4KStage { float4 x[NX], g[NX], h[NX], w[NX]; float rs; u32x4 q8[NX]; };

template <int NX>
__device__ __forceinline__ void q4k_load(__amdgpu_buffer_rsrc_t r, int first, int threads, float4 (&v)[NX]) {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, (first + threads * u) * 16, 0, 0);  // zeros past the end
        v[u] = make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
    }
}
template <int NX>
__device__ __forceinline__ float q4k_sumsq(const float4 (&v)[NX], float ss) {
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        ss = fmaf(v[u].x, v[u].x, ss);
        ss = fmaf(v[u].y, v[u].y, ss);
        ss = fmaf(v[u].z, v[u].z, ss);
        ss = fmaf(v[u].w, v[u].w, ss);
    }
    return ss;
}
// values 4 * slot .. + 3 of x as Q8; the eight lanes of a block of 32 take part together (K is a multiple of 256).
// PLAIN: the norm's weights are taken as they are (add_one == 0)
template <bool NORM, bool PLAIN = false>
__device__ __forceinline__ void q4k_quantize4_store(float4 x, float4 g, float rs, float one, int slot, uint8_t* lds, int K) {
    if (4 * slot >= K) return;
    if constexpr (NORM && PLAIN) x = make_float4(x.x * rs * g.x, x.y * rs * g.y, x.z * rs * g.z, x.w * rs * g.w);
    else if constexpr (NORM) x = norm4(x, g, rs, one);
    float d, sum;
    reinterpret_cast<uint32_t*>(lds)[slot] = q8_quantize4(x, d, sum);
    if ((slot & 7) == 0) {
        float* xd = reinterpret_cast<float*>(lds + K);
        xd[slot >> 3] = d;
        xd[K / 32 + (slot >> 3)] = sum;
    }
}

// NX: 16-byte pieces of x a thread keeps in registers
// SHORT: add_one == 0 and no values beyond those that registers hold
template <bool XQ8, bool NORM, bool PRE, bool SHORT, int NX>
__device__ __forceinline__ Q4KStage<NX> q4k_stage_issue(const Q4KArgs a, uint8_t* lds, float* red, int threads) {
    static_assert(!PRE || (NORM && !XQ8), "the deferred post-norm comes with the RMSNorm prologue");
    Q4KStage<NX> st;
    const int tid = threadIdx.x;
    st.rs = 1.0f;
    if constexpr (XQ8) {
        const uint4* src = reinterpret_cast<const uint4*>(a.x);
        uint4* dst = reinterpret_cast<uint4*>(lds);
        const int n16 = (a.K + a.K / 4) / 16;
        // beyond the register window: copied first, while no other load is in flight
        if constexpr (!SHORT)
            for (int i = tid + NX * threads; i < n16; i += threads) dst[i] = src[i];
        issue_order_fence();  // keep the loads below from being hoisted above that loop
        const __amdgpu_buffer_rsrc_t r = make_rsrc(a.x, n16 * 16);
#pragma unroll
        for (int u = 0; u < NX; ++u) st.q8[u] = __builtin_amdgcn_raw_buffer_load_b128(r, (tid + threads * u) * 16, 0, 0);
    } else {
        const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.K * 4);
        const __amdgpu_buffer_rsrc_t rg = make_rsrc(NORM ? static_cast<const void*>(a.gamma) : a.x, a.K * 4);
        const float one = a.add_one ? 1.0f : 0.0f;
        // Slow path (beyond the values kept in registers) first, while no other load is in flight: the compiler cannot
        // count loads across these loops and waits for everything where the paths join.
        if (!SHORT && a.K > 4 * NX * threads) {
            if constexpr (NORM) {
                float ss = 0.0f;
                for (int base = 0; 4 * base < a.K; base += 4 * threads) {
                    float4 t[4];
                    q4k_load(rx, base + tid, threads, t);
                    ss = q4k_sumsq(t, ss);
                }
                ss = sum_of_waves(ss, red, threads >> 6);
                st.rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
            }
            for (int base = NX * threads; 4 * base < a.K; base += 4 * threads) {
                float4 t[4], g[4];
                q4k_load(rx, base + tid, threads, t);
                if constexpr (NORM) q4k_load(rg, base + tid, threads, g);
#pragma unroll
                for (int u = 0; u < 4; ++u) q4k_quantize4_store<NORM>(t[u], g[u], st.rs, one, base + tid + threads * u, lds, a.K);
            }
        }
        issue_order_fence();
        if constexpr (PRE) {  // the branch output first: its sum of squares is the first thing needed
            q4k_load(make_rsrc(a.pre_h, a.K * 4), tid, threads, st.h);
            q4k_load(make_rsrc(a.pre_w, a.K * 4), tid, threads, st.w);
        }
        q4k_load(rx, tid, threads, st.x);
        if constexpr (NORM) q4k_load(rg, tid, threads, st.g);
    }
    return st;
}

// x + RMSNorm(h) * w, h's sum of squares being ssh
template <int NX>
__device__ __forceinline__ void q4k_add_normed(const float4 (&x)[NX], const float4 (&h)[NX], const float4 (&w)[NX], float ssh, float one, const Q4KArgs& a,
                                               float4 (&xv)[NX]) {
    const float rsh = 1.0f / sqrtf(ssh / (float)a.K + a.eps);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
        xv[u].x = x[u].x + h[u].x * rsh * (w[u].x + one);
        xv[u].y = x[u].y + h[u].y * rsh * (w[u].y + one);
        xv[u].z = x[u].z + h[u].z * rsh * (w[u].z + one);
        xv[u].w = x[u].w + h[u].w * rsh * (w[u].w + one);
    }
}

template <bool XQ8, bool NORM, bool PRE, bool SHORT, int NX>
__device__ __forceinline__ void q4k_stage_finish(const Q4KStage<NX>& st, const Q4KArgs a, uint8_t* lds, float* red, int wg, int threads) {
    const int tid = threadIdx.x;
    const float one = a.add_one ? 1.0f : 0.0f;
    if constexpr (XQ8) {
        uint4* dst = reinterpret_cast<uint4*>(lds);
        const int n16 = (a.K + a.K / 4) / 16;
#pragma unroll
        for (int u = 0; u < NX; ++u) {
            const int i = tid + threads * u;
            if (i < n16) dst[i] = make_uint4(st.q8[u].x, st.q8[u].y, st.q8[u].z, st.q8[u].w);
        }
    } else if constexpr (PRE) {
        // the sum first (threads past the end hold zeros), then the kernel's own RMSNorm of it
        float4 xv[NX];
        q4k_add_normed(st.x, st.h, st.w, sum_of_waves(q4k_sumsq(st.h, 0.0f), red, threads >> 6), one, a, xv);
        if (wg == 0 && a.pre_out) {
#pragma unroll
            for (int u = 0; u < NX; ++u)
                if (4 * (tid + threads * u) < a.K) reinterpret_cast<float4*>(a.pre_out)[tid + threads * u] = xv[u];
        }
        const float ss = sum_of_waves(q4k_sumsq(xv, 0.0f), red, threads >> 6);
        const float rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
#pragma unroll
        for (int u = 0; u < NX; ++u) q4k_quantize4_store<true>(xv[u], st.g[u], rs, one, tid + threads * u, lds, a.K);
    } else {
        float rs = st.rs;
        if constexpr (NORM) {
            if (SHORT || a.K <= 4 * NX * threads) {
                const float ss = sum_of_waves(q4k_sumsq(st.x, 0.0f), red, threads >> 6);
                rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
            }
        }
#pragma unroll
        for (int u = 0; u < NX; ++u) q4k_quantize4_store<NORM, SHORT>(st.x[u], st.g[u], rs, one, tid + threads * u, lds, a.K);
    }
    __syncthreads();
}

// Workgroups of four waves that stage x for one tile take half a Q8 block a thread: the 16 consecutive values [16t, 16t + 16) (lanes t, t ^ 1 share a
// block), so that the quotients of the Q8 rule and what crosses lanes are paid once per 16 values; there each wave's instructions in front of its
// tile count for more than the lines its loads touch.  q / k / v behind a launch that writes x, in pieces as above and so: 6144 x 4096 8.76, 8.10 us, 3072 x 3584
// 7.40, 6.87, gate / up 2 x 1536 x 4096 7.46, 6.88, a product of 1024 x 9728 8.28, 6.97, 512 x 18944 10.72, 8.36; the other way round, 0.16, for 2560 to 4096 x 1024
// and 5120 to 8192 x 512.  (Several tiles a workgroup, pieces: 2 x 14336 x 2560 13.4 us, halves 14.2; 2 x 11008 x 2048 10.2, 9.9.)
struct Q4KHalves { float4 x[4], g[4], h[4], w[4]; float rs; };

__device__ __forceinline__ void q4k_load16(__amdgpu_buffer_rsrc_t r, int first, float4 (&v)[4]) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(r, (first + 4 * u) * 4, 0, 0);  // zeros past the end
        v[u] = make_float4(__uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w));
    }
}
// Q8 rule of quantize_x_q8 (reference: torch/io/cpu_quant_gemv.h:147-198) on the half block `unit` (16 values).
template <bool NORM>
__device__ __forceinline__ void q4k_quantize16_store(const float4 (&xv)[4], const float4 (&gv)[4], float rs, float one,
                                                     int unit, uint8_t* lds, int K) {
    float v[16];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        float4 t = xv[u];
        if constexpr (NORM) t = norm4(t, gv[u], rs, one);
        v[4 * u] = t.x; v[4 * u + 1] = t.y; v[4 * u + 2] = t.z; v[4 * u + 3] = t.w;
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, dpp_f<0xB1>(amax));
    float d, id;
    q8_scales(amax, d, id);
    int isum = 0;
    uint32_t w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        uint32_t q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) q[i] = (uint32_t)max(-127, min(127, (int)rintf(v[4 * u + i] * id)));
        w[u] = pack_bytes(q[0], q[1], q[2], q[3]);
        isum = __builtin_amdgcn_sdot4((int)w[u], 0x01010101, isum, false);
    }
    isum += dpp_i<0xB1>(isum);
    *reinterpret_cast<uint4*>(lds + 16 * unit) = make_uint4(w[0], w[1], w[2], w[3]);
    if ((unit & 1) == 0) {
        float* xd = reinterpret_cast<float*>(lds + K);
        xd[unit >> 1] = d;
        xd[K / 32 + (unit >> 1)] = d * (float)isum;
    }
}

template <bool NORM, bool PRE>
__device__ __forceinline__ Q4KHalves q4k_halves_issue(const Q4KArgs a, uint8_t* lds, float* red) {
    static_assert(!PRE || NORM, "the deferred post-norm comes with the RMSNorm prologue");
    Q4KHalves st;
    const int tid = threadIdx.x;
    st.rs = 1.0f;
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(a.x, a.K * 4);
    const __amdgpu_buffer_rsrc_t rg = make_rsrc(NORM ? static_cast<const void*>(a.gamma) : a.x, a.K * 4);
    if (a.K > 16 * Q4K_THREADS) {  // first, as above
        if constexpr (NORM) {
            float ss = 0.0f;
            for (int base = 0; base < a.K; base += 16 * Q4K_THREADS) {
                float4 t[4];
                q4k_load16(rx, base + 16 * tid, t);
                ss = q4k_sumsq(t, ss);
            }
            ss = block_sum256(ss, red);
            st.rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
        }
        for (int base = 16 * Q4K_THREADS; base < a.K; base += 16 * Q4K_THREADS) {
            float4 t[4], g[4];
            q4k_load16(rx, base + 16 * tid, t);
            if constexpr (NORM) q4k_load16(rg, base + 16 * tid, g);
            if (base + 16 * tid < a.K) q4k_quantize16_store<NORM>(t, g, st.rs, a.add_one ? 1.0f : 0.0f, base / 16 + tid, lds, a.K);
        }
    }
    issue_order_fence();
    if constexpr (PRE) {
        q4k_load16(make_rsrc(a.pre_h, a.K * 4), 16 * tid, st.h);
        q4k_load16(make_rsrc(a.pre_w, a.K * 4), 16 * tid, st.w);
    }
    q4k_load16(rx, 16 * tid, st.x);
    if constexpr (NORM) q4k_load16(rg, 16 * tid, st.g);
    return st;
}

template <bool NORM, bool PRE>
__device__ __forceinline__ void q4k_halves_finish(const Q4KHalves& st, const Q4KArgs a, uint8_t* lds, float* red, int wg) {
    const int tid = threadIdx.x;
    const float one = a.add_one ? 1.0f : 0.0f;
    if constexpr (PRE) {
        float4 xv[4];
        q4k_add_normed(st.x, st.h, st.w, block_sum256(q4k_sumsq(st.h, 0.0f), red), one, a, xv);
        if (wg == 0 && a.pre_out && 16 * tid < a.K) {
#pragma unroll
            for (int u = 0; u < 4; ++u) reinterpret_cast<float4*>(a.pre_out)[4 * tid + u] = xv[u];
        }
        const float ss = block_sum256(q4k_sumsq(xv, 0.0f), red);
        const float rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
        if (16 * tid < a.K) q4k_quantize16_store<true>(xv, st.g, rs, one, tid, lds, a.K);
    } else {
        float rs = st.rs;
        if constexpr (NORM) {
            if (a.K <= 16 * Q4K_THREADS) {
                const float ss = block_sum256(q4k_sumsq(st.x, 0.0f), red);
                rs = 1.0f / sqrtf(ss / (float)a.K + a.eps);
            }
        }
        if (16 * tid < a.K) q4k_quantize16_store<NORM>(st.x, st.g, rs, one, tid, lds, a.K);
    }
    __syncthreads();
}

// What lane j of a block's eight keeps: where in the header the scale and the min of sub-block j lie, and where its activations do.
// The mapping is that of q4k_scale_min; a byte select puts a value's low bits into byte 0 and, of the last four sub-blocks, its two high
// bits on top of byte 1, and byte-to-float conversions join them: a fifth of the instructions of a block less than with shifts.
struct Q4KLane {
    uint32_t select, mask_sc, mask_mn;
    float low_mn;
    const uint8_t* xq;  // low-nibble activations of the lane in block 0, the high-nibble ones 32 on
    const float* xd;    // scale of its sub-block's activations in block 0
    int sums;           // from there to their sum
    bool odd;
};
__device__ __forceinline__ Q4KLane q4k_lane(const uint8_t* lds, int K, int j) {
    Q4KLane l;
    l.select = 0x0c0c0000u | (uint32_t)(j < 4 ? 0x0c : j - 4) << 8 | (uint32_t)j;
    l.mask_sc = j < 4 ? 0x003fu : 0xc00fu;
    l.mask_mn = j < 4 ? 0x003fu : 0xc0f0u;
    l.low_mn = j < 4 ? 1.0f : 0.0625f;
    l.xq = lds + (j >> 1) * 64 + (j & 1) * 16;
    l.xd = reinterpret_cast<const float*>(lds + K) + j;
    l.sums = K / 32;
    l.odd = j & 1;
    return l;
}

// contribution of super-block b to lane j's chain (sub-block j of the block)
__device__ __forceinline__ float q4k_block_term(const uint4 hdr, const uint4 qv, const Q4KLane& l, int b) {
    const int4 xl = *reinterpret_cast<const int4*>(l.xq + b * 256);
    const int4 xh = *reinterpret_cast<const int4*>(l.xq + b * 256 + 32);
    int lo = 0, hi = 0;
    lo = __builtin_amdgcn_sdot4((int)(qv.x & 0x0f0f0f0fu), xl.x, lo, false);
    lo = __builtin_amdgcn_sdot4((int)(qv.y & 0x0f0f0f0fu), xl.y, lo, false);
    lo = __builtin_amdgcn_sdot4((int)(qv.z & 0x0f0f0f0fu), xl.z, lo, false);
    lo = __builtin_amdgcn_sdot4((int)(qv.w & 0x0f0f0f0fu), xl.w, lo, false);
    hi = __builtin_amdgcn_sdot4((int)((qv.x >> 4) & 0x0f0f0f0fu), xh.x, hi, false);
    hi = __builtin_amdgcn_sdot4((int)((qv.y >> 4) & 0x0f0f0f0fu), xh.y, hi, false);
    hi = __builtin_amdgcn_sdot4((int)((qv.z >> 4) & 0x0f0f0f0fu), xh.z, hi, false);
    hi = __builtin_amdgcn_sdot4((int)((qv.w >> 4) & 0x0f0f0f0fu), xh.w, hi, false);
    // even lane keeps the low-nibble half-dot and receives its partner's; odd lane the high one
    const int keep = l.odd ? hi : lo;
    const int give = l.odd ? lo : hi;
    const int isum = keep + dpp_i<0xB1>(give);
    const uint32_t s = __builtin_amdgcn_perm(hdr.w, hdr.y, l.select) & l.mask_sc;
    const uint32_t m = __builtin_amdgcn_perm(hdr.w, hdr.z, l.select) & l.mask_mn;
    const float sc = fmaf((float)((s >> 8) & 0xffu), 0.25f, (float)(s & 0xffu));
    const float mn = fmaf((float)((m >> 8) & 0xffu), 0.25f, (float)(m & 0xffu) * l.low_mn);
    const float d = h2f(hdr.x), dmin = h2f(hdr.x >> 16);
    const float w = d * sc * l.xd[b * 8];
    const float c = dmin * mn * l.xd[b * 8 + l.sums];
    return fmaf(w, (float)isum, -c);
}

__device__ __forceinline__ float gelu_mul_ref(float g, float u) {
    // reference: gguf_model.h:3730-3738
    const float x3 = g * g * g;
    const float t = tanhf(0.7978845608028654f * (g + 0.044715f * x3));
    return 0.5f * g * (1.0f + t) * u;
}

__device__ __forceinline__ float silu_mul_ref(float g, float u) {
    // reference: gguf_model.h:3741-3755 (clamp, libm exp, 1/(1+e), g*sig, *u)
    float ng = 0.0f - g;
    ng = fminf(fmaxf(ng, -88.0f), 88.0f);
    const float sig = 1.0f / (1.0f + expf(ng));
    return (g * sig) * u;
}

// MODE 0: y = or += W.x for up to three matrices over a flattened row space
// MODE 1: gate/up pair with SiLU over interleaved virtual rows (2r = gate row r, 2r+1 = up row r):
//         y[0][r] = silu(Wg[r].x) * (Wu[r].x)
// NB: super-blocks per lane group and pass; every pass issues exactly NB block loads, unconditionally (indices
//     past the row's end are clamped, their terms dropped), so the count of loads in flight is static and a
//     block is consumed as soon as it has arrived instead of after the whole prefetch.
// ROLLT (very tall matrices: a workgroup walks several row tiles, each a single pass of NB blocks per lane group): the
//     passes roll ACROSS tiles - a consumed block's registers are refilled with the same slot of the NEXT tile's row, so a
//     wave never stands with nothing in flight between two tiles (behind the last tile the refills repeat that tile: their
//     number stays static, the lines are in cache, nothing consumes them).
// LS >= 0 (the host's choice, q4k_one): blockDim.x / 64 waves, 1 << LS lane groups per row whose blocks are a single pass, all but the last of the NB a group
//     requests being there for every group; one tile, add_one == 0, x in PIECES 16-byte pieces a thread, EARLY blocks requested in front of its
//     staging.  Addresses are then one base and constants: 70 -> 56 instructions a block, and a launch's setup a third.
template <bool XQ8, bool NORM, bool ACC, int MODE, int NB, bool ROLLT = false, bool PRE = false, int LS = -1, int PIECES = 4, int EARLY = NB, int DEPTH = NB>
__device__ __forceinline__ void q4k_gemv_body(const Q4KArgs a, uint8_t* lds, int wg) {
    constexpr bool ONE = LS >= 0, HALVES = !ONE && !XQ8 && !ROLLT;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane & 7, grp = lane >> 3;
    const int log2S = ONE ? LS : a.log2S;
    const int S = 1 << log2S;
    const int sub = grp & (S - 1);
    const int rows_per_wave = 8 >> log2S;
    const int nblk = a.K / 256;
    const int nb_max = (nblk + S - 1) >> log2S;  // passes are sized for the group with the most blocks
    const int tpw = a.tiles_per_wg > 1 ? a.tiles_per_wg : 1;
    const int waves = ONE ? (int)(blockDim.x >> 6) : 4;
    const int n_tiles = (a.total_rows + waves * rows_per_wave - 1) / (waves * rows_per_wave);
    const Q4KLane ln = q4k_lane(lds, a.K, j);

    // One row tile: first pass of weight loads, `between` (the activation prologue on the first tile, nothing on the
    // others), block terms, reduction, store.
    auto run_tile = [&](int tile, auto&& between) {
        // opaque: a select over the argument struct's arrays (or over what the lambda holds by reference) would push all of it to scratch
        const GlobalBytes W0 = in_global(a.W[0]), W1 = in_global(a.W[1]);
        const int r = (tile * waves + wave) * rows_per_wave + (grp >> log2S);
        const bool live = r < a.total_rows;
        const int rr = live ? r : a.total_rows - 1;
        int mat = 0, local = rr;
        GlobalBytes row;
        GlobalFloats y = nullptr;
        if constexpr (MODE == 1) {
            mat = rr & 1;
            local = rr >> 1;
            row = mat == 0 ? W0 : W1;
        } else {
            const GlobalBytes W2 = in_global(a.W[2]);
            const int end0 = in_registers(a.n_mat > 1 ? a.row_end[0] : INT_MAX), end1 = in_registers(a.n_mat > 2 ? a.row_end[1] : INT_MAX);
            mat = rr >= end1 ? 2 : rr >= end0 ? 1 : 0;
            local = rr - (mat == 2 ? end1 : mat == 1 ? end0 : 0);
            row = mat == 0 ? W0 : (mat == 1 ? W1 : W2);
            const GlobalFloats y0 = in_global(a.y[0]), y1 = in_global(a.y[1]), y2 = in_global(a.y[2]);
            y = (mat == 0 ? y0 : (mat == 1 ? y1 : y2)) + local;
        }
        float y_old = 0.0f;
        if constexpr (ACC) y_old = *y;  // in front of the weights: behind the sums it would be one more trip to memory
        row += ONE ? (int64_t)((uint64_t)(uint32_t)local * (uint32_t)a.stride) : (int64_t)local * a.stride;
        uint4 hdr[NB], qv[NB];
        const int last = ONE ? min(sub + ((NB - 1) << log2S), nblk - 1) : 0;
        auto request = [&](int u) {
            const GlobalBytes p = ONE ? (u < NB - 1 ? row + sub * 144 + (u << log2S) * 144 : row + last * 144)
                                      : row + (int64_t)min(sub + (u << log2S), nblk - 1) * 144;
            hdr[u] = load16(p);
            qv[u] = load16(p + 16 + 16 * j);
        };
        if constexpr (ONE) __builtin_amdgcn_s_setprio(0);
        issue_order_fence();
#pragma unroll
        for (int u = 0; u < (ONE ? EARLY : NB); ++u) request(u);
        issue_order_fence();
        between();
        if constexpr (ONE) {
#pragma unroll
            for (int u = EARLY; u < DEPTH; ++u) request(u);
            issue_order_fence();
        }

        // passes roll: a consumed block's registers are refilled from the next pass at once, so a lane group keeps
        // NB - 1 .. NB blocks in flight while it computes; the last pass only consumes
        float acc = 0.0f;
        int i0 = 0;
        for (; !ONE && i0 + NB < nb_max; i0 += NB) {
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int b = sub + ((i0 + u) << log2S);
                const float t = q4k_block_term(hdr[u], qv[u], ln, min(b, nblk - 1));
                acc += b < nblk ? t : 0.0f;
                const GlobalBytes p = row + (int64_t)min(sub + ((i0 + NB + u) << log2S), nblk - 1) * 144;
                hdr[u] = load16(p);
                qv[u] = load16(p + 16 + 16 * j);
            }
        }
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            if constexpr (ONE) {
                if (u < NB - 1) {
                    Q4KLane at = ln;  // one base, constant offsets
                    at.xq += sub * 256;
                    at.xd += sub * 8;
                    acc += q4k_block_term(hdr[u], qv[u], at, u << LS);
                } else {
                    const float t = q4k_block_term(hdr[u], qv[u], ln, last);
                    acc += sub + (u << LS) < nblk ? t : 0.0f;
                }
                if (u + DEPTH < NB) {
                    request(u + DEPTH);
                    issue_order_fence();
                }
                continue;
            }
            const int b = sub + ((i0 + u) << log2S);
            const float t = q4k_block_term(hdr[u], qv[u], ln, min(b, nblk - 1));
            acc += b < nblk ? t : 0.0f;
        }
        // reduce: 8 lanes of the group, then the S groups of the row
        float p = sum8(acc);
        if (S >= 2) p += dpp_f<0x128>(p);  // row_ror:8 = the other 8-lane half of the 16-lane row
        if (S >= 4) p = add16(p);
        if (S >= 8) p = add32(p);

        if constexpr (MODE == 1) {
            // gate and up of one row sit S groups apart, the gate in the lower lanes
            float other;
            if (S == 1) other = dpp_f<0x128>(p);
            else if (S == 2) other = pair16(p).b;
            else other = pair32(p).b;
            if (live && mat == 0 && sub == 0 && j == 0) a.y[0][local] = a.gelu ? gelu_mul_ref(p, other) : silu_mul_ref(p, other);
        } else {
            if (live && sub == 0 && j == 0) *y = ACC ? y_old + p : p;
        }
    };

    // ---- activation loads first, then the first tile's weight loads, then the activation prologue ----
    __shared__ float red[16];
    static_assert(!(PRE && ROLLT), "the deferred post-norm is built into the one-tile-at-a-time form only");
    if constexpr (ONE) {
        const int threads = blockDim.x;
        __builtin_amdgcn_s_setprio(3);
        const auto stg = q4k_stage_issue<XQ8, NORM, PRE, true, PIECES>(a, lds, red, threads);
        run_tile(wg, [&] {
            __builtin_amdgcn_s_setprio(2);
            q4k_stage_finish<XQ8, NORM, PRE, true, PIECES>(stg, a, lds, red, wg, threads);
            __builtin_amdgcn_s_setprio(0);
        });
        return;
    }
    const auto stg = [&] {
        if constexpr (HALVES) return q4k_halves_issue<NORM, PRE>(a, lds, red);
        else return q4k_stage_issue<XQ8, NORM, PRE, false, XQ8 ? 2 : PIECES>(a, lds, red, Q4K_THREADS);
    }();
    auto finish = [&] {
        if constexpr (HALVES) q4k_halves_finish<NORM, PRE>(stg, a, lds, red, wg);
        else q4k_stage_finish<XQ8, NORM, PRE, false>(stg, a, lds, red, wg, Q4K_THREADS);
    };
    if constexpr (ROLLT) {
        // MODE 0: one matrix (a.W[0], a.y[0]); MODE 1: virtual row 2 r = gate row r (a.W[0]), 2 r + 1 = up row r (a.W[1]).
        // The pointers are taken out of the argument struct once: a select over its arrays per tile would push it to scratch.
        const uint8_t* const W0 = a.W[0];
        const uint8_t* const W1 = MODE == 1 ? a.W[1] : a.W[0];
        float* const y0 = a.y[0];
        auto row_ptr = [&](int rv) {   // virtual row (clamped) -> first byte of its weights
            const int rc = min(rv, a.total_rows - 1);
            if constexpr (MODE == 1) return ((rc & 1) ? W1 : W0) + (int64_t)(rc >> 1) * a.stride;
            else return W0 + (int64_t)rc * a.stride;
        };
        const int total_rows = a.total_rows;
        const int boff = sub * 144, bstep = 144 << log2S;
        int tile = wg * tpw;
        const int tile_end = min(tile + tpw, n_tiles);  // workgroup-uniform; the grid holds no workgroup without a tile
        int r = (tile * 4 + wave) * rows_per_wave + (grp >> log2S);
        const uint8_t* row = row_ptr(r);
        uint4 hdr[NB], qv[NB];
        issue_order_fence();
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const uint8_t* p = row + min(boff + u * bstep, (nblk - 1) * 144);
            hdr[u] = *reinterpret_cast<const uint4*>(p);
            qv[u] = *reinterpret_cast<const uint4*>(p + 16 + 16 * j);
        }
        issue_order_fence();
        finish();
        for (; tile < tile_end; ++tile) {
            const int r_next = tile + 1 < tile_end ? r + 4 * rows_per_wave : r;
            const uint8_t* row_next = row_ptr(r_next);
            float acc = 0.0f;
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int b = sub + (u << log2S);
                const float t = q4k_block_term(hdr[u], qv[u], ln, min(b, nblk - 1));
                acc += b < nblk ? t : 0.0f;
                const uint8_t* p = row_next + min(boff + u * bstep, (nblk - 1) * 144);
                hdr[u] = *reinterpret_cast<const uint4*>(p);
                qv[u] = *reinterpret_cast<const uint4*>(p + 16 + 16 * j);
            }
            float p = sum8(acc);
            if (S >= 2) p += dpp_f<0x128>(p);
            if (S >= 4) p = add16(p);
            if (S >= 8) p = add32(p);
            if constexpr (MODE == 1) {
                // gate and up of one row sit S groups apart, the gate in the lower lanes
                float other;
                if (S == 1) other = dpp_f<0x128>(p);
                else if (S == 2) other = pair16(p).b;
                else other = pair32(p).b;
                if (r < total_rows && (r & 1) == 0 && sub == 0 && j == 0)
                    y0[r >> 1] = a.gelu ? gelu_mul_ref(p, other) : silu_mul_ref(p, other);
            } else {
                if (r < total_rows && sub == 0 && j == 0) {
                    if constexpr (ACC) y0[r] += p;
                    else y0[r] = p;
                }
            }
            r = r_next;
        }
        return;
    }
    run_tile(wg * tpw, finish);
    // further tiles reuse the staged activations: the quantisation of x is paid once per workgroup
    for (int k = 1; k < tpw; ++k) {
        const int tile = wg * tpw + k;
        if (tile >= n_tiles) break;
        run_tile(tile, [] {});
    }
}

// lane groups per row: enough workgroups to cover the chip, and all of a group's blocks in one pass
inline int q4k_pick_log2S(int total_rows, int nblk, int max_log2S) {
    int l = 0;
    while (l < max_log2S) {
        const int S = 1 << l;
        const int wgs = (total_rows * S + 31) / 32;
        const int nb = (nblk + S - 1) / S;
        if (nb <= 5 && wgs >= 600) break;  // 5 blocks in flight per group: measured better than 10 (registers -> occupancy)
        if (nb <= 1) break;
        ++l;
    }
    return l;
}
inline int q4k_workgroups(int total_rows, int log2S) {
    const int rows_per_wg = 32 >> log2S;
    return (total_rows + rows_per_wg - 1) / rows_per_wg;
}
// Row tiles per workgroup: beyond ~1200 tiles a workgroup walks several, so that the activation prologue (every
// workgroup quantises the whole vector) is amortised.
inline int q4k_tiles_per_wg(int n_tiles) {
    const int max_wgs = 1280;
    int t = 1;
    while (t < 8 && (n_tiles + t - 1) / t > max_wgs) ++t;
    return t;
}
// The same for the kernel whose loads roll across a workgroup's tiles (q4k_gemv_tall_kernel): at most 768 workgroups, all
// resident at once (151936 x 2560: 9496 tiles; 2048 / 1024 / 768 / 512 workgroups measured 42.2 / 41.7 / 41.5 / 41.0 us).
inline int q4k_tiles_per_wg_rolling(int n_tiles) {
    const int t = (n_tiles + 767) / 768;
    return t > 16 ? 16 : t;
}
inline int q4k_blocks_per_pass(int nblk, int log2S) {
    static const int cand[] = {2, 3, 4, 5, 10};
    return pick_blocks_per_pass((nblk + (1 << log2S) - 1) >> log2S, cand, 5);
}

}  // namespace ptm
