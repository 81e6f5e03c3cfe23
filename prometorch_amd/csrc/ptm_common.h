// Shared device helpers for the gfx950 kernels (wave64, DPP cross-lane ops, block decode).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include <initializer_list>

#include "../../include/ptm.h"

#define PTM_WAVE 64

namespace ptm {

// ---- error plumbing -------------------------------------------------------------------
extern thread_local int g_last_hip_error;
inline int hip_status(hipError_t e) {
    if (e == hipSuccess) return PTM_OK;
    g_last_hip_error = (int)e;
    return PTM_E_HIP;
}
inline int launch_status() { return hip_status(hipGetLastError()); }
inline hipStream_t as_stream(ptm_stream_t s) { return reinterpret_cast<hipStream_t>(s); }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Kernel arguments are read here, at the start, together: each 64-byte line of them is a trip to memory for the launch's first reader, and
// the compiler reads a line where its first use is, one trip after the other (eight decode steps of Qwen3-4B shapes at 2048 positions 10764 -> 10593
// us, 24 Nadozen steps behind 30 prompt tokens 8438 -> 8303).
template <typename... T>
__device__ __forceinline__ void read_now(const T&... v) {
    (void)std::initializer_list<int>{(([](auto x) { asm volatile("" ::"s"(x)); })(v), 0)...};
}

// A uniform value that the compiler takes as it is, not as the load it comes from.  A pointer is then one it knows nothing of: in_global
// says where it points (a load through a pointer to anywhere is waited for with LDS accesses, too).
template <typename T>
__device__ __forceinline__ T in_registers(T v) {
    asm("" : "+s"(v));
    return v;
}
typedef const __attribute__((address_space(1))) uint8_t* GlobalBytes;
typedef __attribute__((address_space(1))) float* GlobalFloats;
__device__ __forceinline__ GlobalBytes in_global(const uint8_t* p) { return (GlobalBytes)in_registers(p); }
__device__ __forceinline__ GlobalFloats in_global(float* p) { return (GlobalFloats)in_registers(p); }
__device__ __forceinline__ uint4 load16(GlobalBytes p) {
    typedef uint32_t vec __attribute__((ext_vector_type(4)));
    const vec v = *(const __attribute__((address_space(1))) vec*)p;
    return make_uint4(v.x, v.y, v.z, v.w);
}

// Bookkeeping of a decode step done by the thread that finishes the argmax (all NULL: plain argmax):
// publish the token, feed it back as the next input, advance the position.
struct ArgmaxAdvance {
    int* d_token;
    int64_t* d_past;
    int* d_step;
    int64_t* tokens_out;
    int cap;
};

// ---- DPP lane exchanges (row = 16 lanes) ------------------------------------------------
// quad_perm encodings: [1,0,3,2] = 0xB1 (xor 1), [2,3,0,1] = 0x4E (xor 2);
// 0x141 = row_half_mirror (lane i <-> 7-i inside each 8), 0x140 = row_mirror (i <-> 15-i).
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, true));
}
// all-reduce (sum / max) over aligned groups of 8 lanes
__device__ __forceinline__ float sum8(float v) {
    v += dpp_f<0xB1>(v);
    v += dpp_f<0x4E>(v);
    v += dpp_f<0x141>(v);
    return v;
}
__device__ __forceinline__ int sum8i(int v) {
    v += dpp_i<0xB1>(v);
    v += dpp_i<0x4E>(v);
    v += dpp_i<0x141>(v);
    return v;
}
__device__ __forceinline__ float max8(float v) {
    v = fmaxf(v, dpp_f<0xB1>(v));
    v = fmaxf(v, dpp_f<0x4E>(v));
    v = fmaxf(v, dpp_f<0x141>(v));
    return v;
}
__device__ __forceinline__ float sum16(float v) {
    v = sum8(v);
    v += dpp_f<0x140>(v);
    return v;
}
// The two values of a lane pair 16 / 32 lanes apart, in every lane of the pair the same way round: a lane swap, which is a vector
// instruction where a shuffle is a trip through LDS.
struct LanePair { float a, b; };
__device__ __forceinline__ LanePair pair16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ LanePair pair32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ float add16(float v) {
    const LanePair p = pair16(v);
    return p.a + p.b;
}
__device__ __forceinline__ float add32(float v) {
    const LanePair p = pair32(v);
    return p.a + p.b;
}
// all-reduce over each half of the wave (lanes 0..31, 32..63)
__device__ __forceinline__ float sum32(float v) { return add16(sum16(v)); }
// sum over groups of LPP = 8, 16 or 32 consecutive lanes
template <int LPP>
__device__ __forceinline__ float sum_lanes(float v) {
    static_assert(LPP == 8 || LPP == 16 || LPP == 32, "lane group of 8, 16 or 32");
    if constexpr (LPP == 8) return sum8(v);
    else if constexpr (LPP == 16) return sum16(v);
    else return sum32(v);
}
// all-reduce over the whole wave64
__device__ __forceinline__ float sum64(float v) {
    return add32(sum32(v));
}
// The sums over the wave of R = 1, 2 or 4 values in one go: a swap of two registers halves them both.  Lane l has that of value sum_row<R>(l).
template <int R>
__device__ __forceinline__ float sum_rows(const float (&v)[R]) {
    static_assert(R == 1 || R == 2 || R == 4, "registers that halve evenly");
    auto fold32 = [](float a, float b) {  // lanes 0..31: a, 32..63: b
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(r[0]) + __uint_as_float(r[1]);
    };
    if constexpr (R == 1) {
        return sum64(v[0]);
    } else if constexpr (R == 2) {
        return sum32(fold32(v[0], v[1]));
    } else {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(fold32(v[0], v[1])), __float_as_uint(fold32(v[2], v[3])), false, false);
        return sum16(__uint_as_float(r[0]) + __uint_as_float(r[1]));
    }
}
template <int R>
__device__ __forceinline__ int sum_row(int lane) {
    return R == 1 ? 0 : R == 2 ? lane >> 5 : (lane >> 5) + 2 * ((lane >> 4) & 1);
}
__device__ __forceinline__ float max64(float v) {
    v = max8(v);
    v = fmaxf(v, dpp_f<0x140>(v));
    LanePair p = pair16(v);
    p = pair32(fmaxf(p.a, p.b));
    return fmaxf(p.a, p.b);
}

// ---- fp16 ---------------------------------------------------------------------------
__device__ __forceinline__ float h2f(uint32_t bits16) {
    return __half2float(__ushort_as_half((unsigned short)(bits16 & 0xffffu)));
}
__device__ __forceinline__ unsigned short f2h_bits(float f) { return __half_as_ushort(__float2half_rn(f)); }

// ---- Q4_K header decode: 12 packed bytes (3 dwords) -> (scale, min) of sub-block j ------
// Same mapping as get_scale_min_k4 (reference: torch/io/gguf_dequant.h:289-297).
__device__ __forceinline__ void q4k_scale_min(uint32_t s0, uint32_t s1, uint32_t s2, int j, int& sc, int& mn) {
    const int sh = 8 * (j & 3);
    const uint32_t b0 = (s0 >> sh) & 0xffu, b1 = (s1 >> sh) & 0xffu, b2 = (s2 >> sh) & 0xffu;
    const int sc_lo = b0 & 63u, mn_lo = b1 & 63u;
    const int sc_hi = (b2 & 0x0fu) | ((b0 >> 6) << 4);
    const int mn_hi = (b2 >> 4) | ((b1 >> 6) << 4);
    sc = j < 4 ? sc_lo : sc_hi;
    mn = j < 4 ? mn_lo : mn_hi;
}

// 16-byte load from an address that is only 2-byte aligned (Q6_K blocks are 210 B).
struct __attribute__((packed, aligned(2))) u128_a2 { uint32_t v[4]; };
__device__ __forceinline__ uint4 ld16_a2(const uint8_t* p) {
    const u128_a2 t = *reinterpret_cast<const u128_a2*>(p);
    return make_uint4(t.v[0], t.v[1], t.v[2], t.v[3]);
}
struct __attribute__((packed, aligned(2))) u16_a2 { uint16_t v; };

// Q8 activation layout in memory: int8 qs[K] | float d[K/32] | float sum[K/32]
__host__ __device__ inline int64_t q8_bytes(int K) { return (int64_t)K + K / 4; }

// the low bytes of four values, the first lowest
__device__ __forceinline__ uint32_t pack_bytes(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_amdgcn_perm(b, a, 0x0c0c0400u) | __builtin_amdgcn_perm(d, c, 0x04000c0cu);
}

// d = amax / 127 and id = 1 / d, 0 where d is, both correctly rounded: a quotient from a correctly rounded reciprocal (of 127 a constant, of d the
// hardware's with one Newton step) is put right by one exact remainder (Markstein, IBM J. Res. Dev. 34, 1990).  6 instructions where the IEEE
// sequences take 24.  One step does not round every reciprocal of every hardware correctly; here it does, for each of the 2^23 amax of a binade and so,
// by their scaling, of all from 2^-90 to 2^90 (test_quantize_q8_scales_are_ieee_quotients).  Other amax, 0 and NaN among them: the IEEE sequences.
__device__ __forceinline__ void q8_scales(float amax, float& d, float& id) {
    const float r127 = 1.0f / 127.0f, q = amax * r127;
    d = fmaf(fmaf(-127.0f, q, amax), r127, q);
    const float r = __builtin_amdgcn_rcpf(d);
    id = fmaf(fmaf(-d, r, 1.0f), r, r);
    if (!(amax >= 0x1p-90f && amax <= 0x1p90f)) {
        d = amax / 127.0f;
        id = d > 0.0f ? 1.0f / d : 0.0f;
    }
}

// Quantise the 32 floats held as float4 by the 8 lanes of an aligned lane group.
// Returns the packed 4 int8 of this lane; d and sum (d * sum q) are group-uniform.
// Same rule as quantize_x_q8 (reference: torch/io/cpu_quant_gemv.h:147-198).
__device__ __forceinline__ uint32_t q8_quantize4(float4 v, float& d, float& sum) {
    float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
    amax = max8(amax);
    float id;
    q8_scales(amax, d, id);
    int q0 = (int)rintf(v.x * id), q1 = (int)rintf(v.y * id), q2 = (int)rintf(v.z * id), q3 = (int)rintf(v.w * id);
    q0 = max(-127, min(127, q0));
    q1 = max(-127, min(127, q1));
    q2 = max(-127, min(127, q2));
    q3 = max(-127, min(127, q3));
    const uint32_t q = pack_bytes((uint32_t)q0, (uint32_t)q1, (uint32_t)q2, (uint32_t)q3);
    sum = d * (float)sum8i(__builtin_amdgcn_sdot4((int)q, 0x01010101, 0, false));
    return q;
}

// Block-wide sum over `waves` <= 16 waves; red is 16 floats of LDS.
__device__ __forceinline__ float sum_of_waves(float v, float* red, int waves) {
    v = sum64(v);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    const int i = threadIdx.x & 15;
    return sum16(i < waves ? red[i] : 0.0f);
}
// for blockDim.x = 256 (4 waves)
__device__ __forceinline__ float block_sum256(float v, float* red) {
    v = sum64(v);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// ---- activation staging --------------------------------------------------------------------------
// A 256-thread workgroup walks x[K] as float4 slots i = tid + 256*u.  Loads are issued four slots
// at a time BEFORE any of them is consumed, so a staging pass costs one memory round trip per 4096
// values instead of one per 1024.  For K <= 4096 the slots stay in registers between the
// sum-of-squares pass and the normalise pass.
struct XChunk { float4 v[4]; };

// Activations are fetched with buffer loads: the hardware range check returns zeros for slots past the end of
// the vector, so the load needs no predicate.  (A predicated global load is compiled to a branch around the
// load; the compiler can then no longer count the loads in flight and waits for ALL of them, the weight
// prefetch included, before the first use of x.)
// Compiler-only fence: memory operations are neither moved nor scheduled across it.  Used to pin the ISSUE
// order of loads (activations, then weights), which decides the order in which their data can be consumed.
__device__ __forceinline__ void issue_order_fence() { asm volatile("" ::: "memory"); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ XChunk load_chunk(__amdgpu_buffer_rsrc_t rs, int base) {
    XChunk c;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = base + (int)threadIdx.x + 256 * u;
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, i * 16, 0, 0);
        c.v[u] = make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
    }
    return c;
}

__device__ __forceinline__ float chunk_sumsq(const XChunk& c, float ss) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        ss = fmaf(c.v[u].x, c.v[u].x, ss);
        ss = fmaf(c.v[u].y, c.v[u].y, ss);
        ss = fmaf(c.v[u].z, c.v[u].z, ss);
        ss = fmaf(c.v[u].w, c.v[u].w, ss);
    }
    return ss;
}

// x * rs * (gamma [+1]) in the reference's order (cpu_quant_gemv.h:2599)
__device__ __forceinline__ float4 norm4(float4 v, float4 g, float rs, float one) {
    v.x = v.x * rs * (g.x + one);
    v.y = v.y * rs * (g.y + one);
    v.z = v.z * rs * (g.z + one);
    v.w = v.w * rs * (g.w + one);
    return v;
}

// Staging is split in two so that a kernel can put its (few) activation loads in front of its (many)
// weight loads: vector loads complete in issue order, so activation loads issued behind the weight
// prefetch could only be consumed after every weight had arrived.
//   XStage<NCH> st = stage_issue<NORM, NCH>(x, gamma, K, eps, add_one, red, emit);   // loads of the first NCH*4096 values
//   ... issue weight loads ...
//   stage_finish<NORM, NCH>(st, K, eps, add_one, red, emit);
// emit(i, value) is called for every float4 slot i of x (RMS-normalised with gamma when NORM), all 256
// threads taking part; emit may use cross-lane ops (slots are handed out wave-uniformly: K % 256 == 0).
// Between the two calls only unconditional loads may be issued, and stage_finish issues none: the compiler
// can then count the loads in flight and wait for exactly the activation loads.  Vectors longer than
// NCH*4096 values take a slow path that stages the part beyond the register window first, inside stage_issue.
template <int NCH = 1>
struct XStage { XChunk x[NCH], g[NCH]; float rs; };

template <bool NORM, typename Emit>
__device__ __forceinline__ void emit_chunk(const XChunk& c, const XChunk& g, int base, int n4, float rs, float one,
                                           Emit& emit) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = base + (int)threadIdx.x + 256 * u;
        if (i < n4) {
            float4 v = c.v[u];
            if constexpr (NORM) v = norm4(v, g.v[u], rs, one);
            emit(i, v);
        }
    }
}

template <bool NORM, int NCH = 1, typename Emit>
__device__ __forceinline__ XStage<NCH> stage_issue(const float* __restrict__ x, const float* __restrict__ gamma, int K,
                                                   float eps, int add_one, float* red4, Emit emit) {
    const __amdgpu_buffer_rsrc_t x4 = make_rsrc(x, K * 4);
    const __amdgpu_buffer_rsrc_t g4 = make_rsrc(NORM ? gamma : x, K * 4);
    const int n4 = K / 4;
    XStage<NCH> st;
    st.rs = 1.0f;
    // Slow path first, while no other load is in flight: the compiler cannot count loads across this loop and
    // waits for everything outstanding where the paths join, which costs nothing here.
    if (n4 > 1024 * NCH) {
        if constexpr (NORM) {
            float ss = 0.0f;
            for (int base = 0; base < n4; base += 1024) ss = chunk_sumsq(load_chunk(x4, base), ss);
            ss = block_sum256(ss, red4);
            st.rs = 1.0f / sqrtf(ss / (float)K + eps);
        }
        for (int base = 1024 * NCH; base < n4; base += 1024) {
            const XChunk c = load_chunk(x4, base);
            XChunk g = c;
            if constexpr (NORM) g = load_chunk(g4, base);
            emit_chunk<NORM>(c, g, base, n4, st.rs, add_one ? 1.0f : 0.0f, emit);
        }
    }
    issue_order_fence();  // keep the loads below from being hoisted above the slow path
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        st.x[c] = load_chunk(x4, 1024 * c);
        if constexpr (NORM) st.g[c] = load_chunk(g4, 1024 * c);
    }
    return st;
}

template <bool NORM, int NCH = 1, typename Emit>
__device__ __forceinline__ void stage_finish(const XStage<NCH>& st, int K, float eps, int add_one, float* red4,
                                             Emit emit) {
    const int n4 = K / 4;
    float rs = st.rs;
    if constexpr (NORM) {
        if (n4 <= 1024 * NCH) {
            float ss = 0.0f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) ss = chunk_sumsq(st.x[c], ss);
            ss = block_sum256(ss, red4);
            rs = 1.0f / sqrtf(ss / (float)K + eps);
        }
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c)
        if (1024 * c < n4) emit_chunk<NORM>(st.x[c], st.g[c], 1024 * c, n4, rs, add_one ? 1.0f : 0.0f, emit);
}

// The same staging with a deferred post-norm in front (K <= 4096, one chunk): the vector that is normalised is
// x + RMSNorm(h) * w, formed by every workgroup from x, the branch output h and the post-norm weight w; pre_out (NULL in all
// but one workgroup) receives that sum.  Slots past the end of the vectors load as zeros and stay zero.
struct XStagePre { XChunk x, g, h, w; };

__device__ __forceinline__ XStagePre stage_issue_pre(const float* x, const float* gamma, const float* h, const float* w, int K) {
    XStagePre st;
    st.h = load_chunk(make_rsrc(h, K * 4), 0);  // the branch output first: its sum of squares is the first thing needed
    st.w = load_chunk(make_rsrc(w, K * 4), 0);
    st.x = load_chunk(make_rsrc(x, K * 4), 0);
    st.g = load_chunk(make_rsrc(gamma, K * 4), 0);
    return st;
}

template <typename Emit>
__device__ __forceinline__ void stage_finish_pre(const XStagePre& st, int K, float eps, int add_one, float* red4,
                                                 float* pre_out, Emit emit) {
    const int n4 = K / 4;
    const float one = add_one ? 1.0f : 0.0f;
    const float ssh = block_sum256(chunk_sumsq(st.h, 0.0f), red4);
    const float rsh = 1.0f / sqrtf(ssh / (float)K + eps);
    XChunk xe;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        xe.v[u].x = st.x.v[u].x + st.h.v[u].x * rsh * (st.w.v[u].x + one);
        xe.v[u].y = st.x.v[u].y + st.h.v[u].y * rsh * (st.w.v[u].y + one);
        xe.v[u].z = st.x.v[u].z + st.h.v[u].z * rsh * (st.w.v[u].z + one);
        xe.v[u].w = st.x.v[u].w + st.h.v[u].w * rsh * (st.w.v[u].w + one);
        const int i = (int)threadIdx.x + 256 * u;
        if (pre_out && i < n4) reinterpret_cast<float4*>(pre_out)[i] = xe.v[u];
    }
    const float ss = block_sum256(chunk_sumsq(xe, 0.0f), red4);
    const float rs = 1.0f / sqrtf(ss / (float)K + eps);
    emit_chunk<true>(xe, st.g, 0, n4, rs, one, emit);
}

// Blocks per pass for a lane group that owns nb_max blocks: the candidate (from a small set, so that the
// number of kernel instances stays small) that wastes the fewest padded block slots; ties go to the larger.
inline int pick_blocks_per_pass(int nb_max, const int* cand, int n_cand) {
    int best = cand[0], best_waste = 1 << 30;
    for (int i = 0; i < n_cand; ++i) {
        const int waste = (nb_max + cand[i] - 1) / cand[i] * cand[i] - nb_max;
        if (waste < best_waste || (waste == best_waste && cand[i] > best)) { best = cand[i]; best_waste = waste; }
    }
    return best;
}

}  // namespace ptm
