// Prompt attention of the block decoders on the matrix cores, bfloat16: a workgroup owns one kv head and 128 query vectors, walks the visible keys in
// tiles of 64 through LDS; S^T = K . Q^T, online softmax in the accumulator layout, O^T += V^T . P^T with P as two bfloat16 terms (16 bits of the
// fp32 weights).  In a file, and so a code object, of its own: where a decode step's kernels lie in memory is then not moved by its size (a step of
// 52 launches took 1 % longer with them in one).
#include "attention.h"

#include <type_traits>

namespace ptm {

// v_mfma_f32_32x32x16_bf16: A: lane l holds row l % 32, summation indices 8 (l / 32) + 0..7; B: column l % 32, the same
// indices; C: column l % 32, rows 8 (r / 4) + 4 (l / 32) + r % 4.  The 16 keys of a P.V step are the ones the lane already
// holds in its S^T accumulator, in that order.
// A tile's vector arithmetic takes longer than its 48 MFMAs, so it is kept short: the cap in three instructions beside 2^x and 1 / x (ten as
// written: 1030 rows of 32 heads of 128, capped, 54.5 -> 46.4 us) in a kernel of its own, conversions in pairs, scale and reference of an exponent in one
// multiply-add, no branch around a piece that is padding (it is read from zeros).  With the pairing of long row blocks and short ones, launches in a row:
// 2048 rows of 32 heads of 128, gated, 88 -> 79 us, 1500 rows 66 -> 59, 1030 rows of 192 and 128 46.6 -> 45.1, capped 42.6 -> 40.2.  A reference that moves
// only when it is passed by 2^8 takes 1 to 7 us less, but then the largest weight is no longer 1, and a tenth to a third more of the results were not the
// bfloat16 number nearest to the exact one.  Two groups of waves on alternate tiles, and the scores of the next 32 keys formed between the parts of a softmax (K
// a tile ahead in LDS), were no faster: 47.3 and 47.8 us, capped.
__device__ const uint4 zero_piece = {0, 0, 0, 0};

// Workgroups of a class that share a CU.  (Of 256 and 256 the registers leave room for one.)
constexpr int mfma_resident(int DQ, int DV) { return DQ <= 192 && DV <= 128 ? 2 : 1; }
// Row blocks go longest first.  Where two workgroups share a CU and all are there at once, the second 256 come shortest first, so that the longest row block
// has the shortest beside it: heads of 128, 512 workgroups 85 -> 79 us, 328 43 -> 41; where only a few share (heads of 64, 264) 23.9 -> 24.5.  With one a CU
// it would put long ones last: heads of 256, 512 workgroups 165 us, and 134 so.
__host__ __device__ constexpr int mfma_order(int id, int grid, int resident) {
    return resident == 2 && grid > 256 && grid <= 512 && id >= 256 ? grid - 1 - (id - 256) : id;
}

template <int DQ, int DV, bool CAP>
__global__ __launch_bounds__(256, mfma_resident(DQ, DV)) void attention_mfma_kernel(const ptm_attention_args a) {
    constexpr int KS = DQ / 16, DT = DV / 32, KP = DQ * 2 + 16, VP = DV * 2 + 64;
    __shared__ __align__(16) uint8_t s_k[64 * KP];
    __shared__ __align__(16) uint8_t s_v[64 * VP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 31, kh = lane >> 5;
    const int per = a.heads / a.kv_heads, dq = a.dim1 + a.dim2;
    int sh = 0;  // a row takes 1 << sh slots (heads) of a wave's 32 query vectors
    while ((1 << sh) < per && sh < 5) ++sh;
    const int htiles = (per + 31) / 32, rpw = 32 >> sh, bm = 4 * rpw;
    // all kv heads of a row block together
    const int id = mfma_order(blockIdx.x, gridDim.x, mfma_resident(DQ, DV));
    const int gh = id % (a.kv_heads * htiles), g = gh / htiles, ht = gh % htiles;
    const int m_base = ((a.rows + bm - 1) / bm - 1 - id / (a.kv_heads * htiles)) * bm;
    const int slot = (j & ((1 << sh) - 1)) + 32 * ht, row = m_base + wave * rpw + (j >> sh);
    const bool live = slot < per && row < a.rows;
    const int row_c = row < a.rows ? row : a.rows - 1, head = g * per + (slot < per ? slot : per - 1);
    const int64_t pos = a.pos0 + row_c;

    at_b8 qf[KS];
    {
        const uint16_t* src = static_cast<const uint16_t*>(a.Q) + (int64_t)row_c * a.q_row + (int64_t)head * dq + 8 * kh;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            u32x4 v = {0, 0, 0, 0};
            if (16 * ks + 8 * kh < dq && a.scale != 0.0f) v = *reinterpret_cast<const u32x4*>(src + 16 * ks);
            if (a.scale < 0.0f) v ^= 0x80008000u;  // the loop's scale is positive
            qf[ks] = __builtin_bit_cast(at_b8, v);
        }
    }
    at_f16 acc[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = 0.0f;
    // the two lane halves of a query add their sums at the end: one of them holds the sink
    float m_run = a.sink ? a.sink[head] * LOG2E : -INFINITY, l_run = a.sink && kh == 0 ? 1.0f : 0.0f;

    const int64_t p_min = a.pos0 + m_base, p_max = a.pos0 + (m_base + bm < a.rows ? m_base + bm : a.rows) - 1;
    const int wt0 = a.window > 0 && p_min - a.window + 1 > 0 ? (int)((p_min - a.window + 1) / 64) : 0;
    const int kt = (a.keep_first + 63) / 64, nk = a.window > 0 ? (kt < wt0 ? kt : wt0) : 0;
    const int ntiles = nk + (int)(p_max / 64) - wt0 + 1;
    auto tile_at = [&](int i) { return i < nk ? i : wt0 + i - nk; };

    // A thread stages 16-byte pieces of rows tid / 8 and tid / 8 + 32, columns 8 (tid % 8) + 64 g; past the key or value size it reads zeros.
    constexpr int GK = DQ / 64, GV = DV / 64;
    const int r0 = tid >> 3, c0 = (tid & 7) * 8;
    const uint16_t* kp[GK];
    const uint16_t* vp[GV];
    uint32_t kstr[GK], vstr[GV];
#pragma unroll
    for (int i = 0; i < GK; ++i) {
        const int c = c0 + 64 * i;
        kp[i] = c < a.dim1 ? static_cast<const uint16_t*>(a.K1) + (int64_t)g * a.k1_head + c
                : c < dq   ? static_cast<const uint16_t*>(a.K2) + (c - a.dim1)
                           : reinterpret_cast<const uint16_t*>(&zero_piece);
        kstr[i] = c < a.dim1 ? (uint32_t)a.k1_row : c < dq ? (uint32_t)a.k2_row : 0u;
    }
#pragma unroll
    for (int i = 0; i < GV; ++i) {
        const int c = c0 + 64 * i;
        vp[i] = c < a.vdim ? static_cast<const uint16_t*>(a.V) + (int64_t)g * a.v_head + c : reinterpret_cast<const uint16_t*>(&zero_piece);
        vstr[i] = c < a.vdim ? (uint32_t)a.v_row : 0u;
    }
    u32x4 kreg[2 * GK], vreg[2 * GV];
    const int key_last = (int)(p_max - a.kv_pos0);
    // keys past the last visible one repeat it, keys before the array its first; both are masked
    auto key_of = [&](int tile, int r) {
        const int key = (int)((int64_t)tile * 64 - a.kv_pos0) + r;
        return (uint32_t)max(min(key, key_last), 0);
    };
    auto fetch_k = [&](int tile) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t key = key_of(tile, r0 + 32 * u);
#pragma unroll
            for (int i = 0; i < GK; ++i) kreg[GK * u + i] = *reinterpret_cast<const u32x4*>(kp[i] + (uint64_t)key * kstr[i]);
        }
    };
    auto fetch_v = [&](int tile) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t key = key_of(tile, r0 + 32 * u);
#pragma unroll
            for (int i = 0; i < GV; ++i) vreg[GV * u + i] = *reinterpret_cast<const u32x4*>(vp[i] + (uint64_t)key * vstr[i]);
        }
    };
    // scores in base 2, capped: cap tanh(s / cap) = cap - 2 cap / (2^(s turn) + 1), which ends at +-cap for large arguments
    const float sc2 = a.scale != 0.0f ? fabsf(a.scale) * LOG2E : 1.0f, cap2 = a.softcap * LOG2E, turn = CAP ? 2.0f * sc2 / a.softcap : 0.0f;
    const float mul = CAP ? 1.0f : sc2;  // of a score in its exponent
    fetch_k(tile_at(0));
    fetch_v(tile_at(0));
    for (int it = 0; it < ntiles; ++it) {
        const int64_t k0 = (int64_t)tile_at(it) * 64;
        __syncthreads();  // every wave has finished reading the previous tile
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int i = 0; i < GK; ++i) *reinterpret_cast<u32x4*>(s_k + (r0 + 32 * u) * KP + (c0 + 64 * i) * 2) = kreg[GK * u + i];
#pragma unroll
            for (int i = 0; i < GV; ++i) *reinterpret_cast<u32x4*>(s_v + (r0 + 32 * u) * VP + (c0 + 64 * i) * 2) = vreg[GV * u + i];
        }
        __syncthreads();
        const int next = tile_at(it + 1 < ntiles ? it + 1 : it);
        fetch_k(next);
        issue_order_fence();
        at_f16 sc[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[u][r] = 0.0f;
        }
        // a few fragments are read at a time, of the two halves in turn: the MFMAs wait for a batch, not each for its own read
        constexpr int KB = 4;
#pragma unroll
        for (int k4 = 0; k4 < KS; k4 += KB)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                at_b8 ka[KB];
#pragma unroll
                for (int w = 0; w < KB; ++w) ka[w] = *reinterpret_cast<const at_b8*>(s_k + (32 * u + j) * KP + (16 * (k4 + w) + 8 * kh) * 2);
#pragma unroll
                for (int w = 0; w < KB; ++w) asm volatile("" : "+v"(ka[w]));
#pragma unroll
                for (int w = 0; w < KB; ++w) sc[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[w], qf[k4 + w], sc[u], 0, 0, 0);
            }
        issue_order_fence();
        fetch_v(next);
        issue_order_fence();
        if constexpr (CAP) {
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[u][r] = fmaf(-2.0f * cap2, __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(sc[u][r] * turn) + 1.0f), cap2);
        }
        // a tile some query of the workgroup does not see whole (workgroup-uniform)
        const bool whole = k0 + 63 <= p_min && (a.window <= 0 || p_max - k0 < a.window || k0 + 63 < a.keep_first);
        if (!whole) {
            issue_order_fence();  // keeps this a branch
            const int last = (int)(pos - k0 < 64 ? pos - k0 : 64);                                        // keys up to here
            const int64_t f64 = a.window > 0 ? pos - a.window + 1 - k0 : 0;
            const int first = (int)(f64 < 0 ? 0 : f64 < 64 ? f64 : 64);                                   // window from here
            const int kept = (int)(a.keep_first - k0 < 0 ? 0 : a.keep_first - k0 < 64 ? a.keep_first - k0 : 64);  // kept below here
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int o = 32 * u + 8 * (r >> 2) + 4 * kh + (r & 3);
                    sc[u][r] = o <= last && (o >= first || o < kept) ? sc[u][r] : -INFINITY;
                }
        }
        float mx = sc[0][0];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[u][r]);
        const LanePair p = pair32(mx);
        mx = fmaxf(p.a, p.b);
        // The reference of a query's weights is its largest exponent so far: the largest weight is 1, which two bfloat16 terms hold exactly.
        mx *= mul;
        const float m_new = fmaxf(m_run, mx), ms = m_new == -INFINITY ? 0.0f : m_new;  // nothing visible yet
        const float corr = __builtin_amdgcn_exp2f(m_run - ms);
        float psum = 0.0f;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                sc[u][r] = __builtin_amdgcn_exp2f(fmaf(sc[u][r], mul, -ms));
                psum += sc[u][r];
            }
        l_run = fmaf(l_run, corr, psum);
        if (__builtin_amdgcn_ballot_w64(m_new != m_run) != 0) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[dt][r] *= corr;
        }
        m_run = m_new;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                at_b8 hi, lo;
#pragma unroll
                for (int i = 0; i < 8; i += 2) {  // two conversions an instruction
                    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
                    typedef float f2 __attribute__((ext_vector_type(2)));
                    const f2 p = {sc[u][8 * ks + i], sc[u][8 * ks + i + 1]};
                    const b2 h = __builtin_convertvector(p, b2);
                    const f2 rest = {p[0] - (float)h[0], p[1] - (float)h[1]};
                    const b2 l = __builtin_convertvector(rest, b2);
                    hi[i] = h[0];
                    hi[i + 1] = h[1];
                    lo[i] = l[0];
                    lo[i + 1] = l[1];
                }
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const uint8_t* vrow = s_v + (32 * u + 16 * ks + 4 * kh + ((lane & 15) >> 2)) * VP + (32 * dt + (j & 16) + 4 * (lane & 3)) * 2;
                    const at_s4 v0 = lds_tr16(vrow), v1 = lds_tr16(vrow + 8 * VP);
                    typedef short s8 __attribute__((ext_vector_type(8)));
                    const at_b8 va = __builtin_bit_cast(at_b8, (s8){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]});
                    acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, hi, acc[dt], 0, 0, 0);
                    acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, lo, acc[dt], 0, 0, 0);
                }
            }
    }
    const float inv = 1.0f / (add32(l_run));
    if (!live) return;
    uint16_t* dst = static_cast<uint16_t*>(a.O) + (int64_t)row * a.o_row + (int64_t)head * a.vdim + 4 * kh;
    const float scale = a.out_scale != 0.0f ? a.out_scale : 1.0f;
    const float* gate = a.gate ? a.gate + (int64_t)row * a.gate_row + (int64_t)head * a.gate_head : nullptr;
    const int gates = gate ? a.gate_head : 0;
    const bool fours = !((a.gate_row | (int64_t)gates) & 3) && !(reinterpret_cast<uintptr_t>(a.gate) & 15);
    float4 z[4 * DT];
    if (gate) {  // requested together, four at a time where they lie so (2048 rows of 32 heads of 128: one after the other 7 us more)
#pragma unroll
        for (int i = 0; i < 4 * DT; ++i) {
            const int v = 8 * i + 4 * kh;
            if (fours) z[i] = *reinterpret_cast<const float4*>(gate + min(v, max(gates - 4, 0)));
            else z[i] = make_float4(gate[min(v, gates - 1)], gate[min(v + 1, gates - 1)], gate[min(v + 2, gates - 1)], gate[min(v + 3, gates - 1)]);
        }
    }
    auto factor = [&](int v, float z) { return v < gates ? scale * sigmoid_f(z) : scale; };  // out_factor
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (32 * dt + 8 * q < a.vdim) {
                float v0 = acc[dt][4 * q] * inv, v1 = acc[dt][4 * q + 1] * inv, v2 = acc[dt][4 * q + 2] * inv, v3 = acc[dt][4 * q + 3] * inv;
                if (gate) {
                    const int v = 32 * dt + 8 * q + 4 * kh;
                    const float4 x = z[4 * dt + q];
                    v0 *= factor(v, x.x);
                    v1 *= factor(v + 1, x.y);
                    v2 *= factor(v + 2, x.z);
                    v3 *= factor(v + 3, x.w);
                } else if (a.out_scale != 0.0f) {
                    v0 *= scale;
                    v1 *= scale;
                    v2 *= scale;
                    v3 *= scale;
                }
                *reinterpret_cast<uint2*>(dst + 32 * dt + 8 * q) =
                    make_uint2((uint32_t)f_bf16(v0) | ((uint32_t)f_bf16(v1) << 16), (uint32_t)f_bf16(v2) | ((uint32_t)f_bf16(v3) << 16));
            }
}

template <int DQ, int DV>
static int mfma_launch(const ptm_attention_args& a, hipStream_t s) {
    const int per = a.heads / a.kv_heads;
    int sh = 0;
    while ((1 << sh) < per && sh < 5) ++sh;
    const int bm = 4 * (32 >> sh), htiles = (per + 31) / 32;
    const dim3 grid((unsigned)((a.rows + bm - 1) / bm * a.kv_heads * htiles));
    if (a.softcap > 0.0f) hipLaunchKernelGGL((attention_mfma_kernel<DQ, DV, true>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((attention_mfma_kernel<DQ, DV, false>), grid, dim3(256), 0, s, a);
    return launch_status();
}

// f(key size, value size) of the class that has such heads
template <typename F>
static int mfma_class(int dq, int dv, F f) {
    using std::integral_constant;
    if (dq <= 64 && dv <= 64) return f(integral_constant<int, 64>{}, integral_constant<int, 64>{});
    if (dq <= 128 && dv <= 64) return f(integral_constant<int, 128>{}, integral_constant<int, 64>{});
    if (dq <= 128 && dv <= 128) return f(integral_constant<int, 128>{}, integral_constant<int, 128>{});
    if (dq <= 192 && dv <= 128) return f(integral_constant<int, 192>{}, integral_constant<int, 128>{});
    return f(integral_constant<int, 256>{}, integral_constant<int, 256>{});
}

int attention_mfma(const ptm_attention_args& a, hipStream_t s) {
    return mfma_class(a.dim1 + a.dim2, a.vdim, [&](auto dq, auto dv) { return mfma_launch<decltype(dq)::value, decltype(dv)::value>(a, s); });
}
// which row block's turn a workgroup's is, counted from the longest
int attention_mfma_order(int dq, int dv, int id, int grid) {
    return mfma_class(dq, dv, [&](auto q, auto v) { return mfma_order(id, grid, mfma_resident(decltype(q)::value, decltype(v)::value)); });
}

}  // namespace ptm
