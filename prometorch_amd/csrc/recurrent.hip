// Recurrent mixers: a matrix state per head, kept in fp32 and carried from token to token.
//
//   wkv   o_t = (S + diag(u) k v^T)^T r,  S <- diag(w) S + k v^T          (decay w per key channel and token)
//   ssm   S <- a S + dt B x^T,  y_t = S^T C + D x                         (decay a per head and token; B, C per group of heads)
//
// A state is stored per value column, its key values consecutive and padded: [heads][columns][16 * KPL].
// One token: 16 lanes share a column, KPL key values each, so a wave holds four columns and a read of the state is consecutive.
// Prompt rows: 16 tokens at a time on the fp32 matrix cores (scan_columns); a launch in front leaves what the 16 take from each other.
// A sequence's first position starts from zeros instead of the stored state, so nothing has to be cleared between sequences.
// What a token needs from earlier ones besides the state (the token shift's vector, the convolution's inputs) lies in rings
// indexed by position; a slot is never read and written by the same launch.
#include "dense.h"
#include "gemm_tile.h"

#include <mutex>
#include <type_traits>

namespace ptm {

typedef float rc_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float softplus_f(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

template <int KPL>
__device__ __forceinline__ void load_keys(float (&s)[KPL], const float* p) {
#pragma unroll
    for (int i = 0; i < KPL; i += 4) {
        const float4 v = *reinterpret_cast<const float4*>(p + i);
        s[i] = v.x; s[i + 1] = v.y; s[i + 2] = v.z; s[i + 3] = v.w;
    }
}
template <int KPL>
__device__ __forceinline__ void store_keys(float* p, const float (&s)[KPL]) {
#pragma unroll
    for (int i = 0; i < KPL; i += 4) *reinterpret_cast<float4*>(p + i) = make_float4(s[i], s[i + 1], s[i + 2], s[i + 3]);
}

// f(integral constants 0 .. N - 1)
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// key values per lane for a state of n key channels (0: too many)
static int keys_per_lane(int n) { return n <= 64 ? 4 : n <= 128 ? 8 : n <= 256 ? 16 : n <= 512 ? 32 : 0; }
int64_t recurrent_state_floats(int heads, int keys, int columns) { return (int64_t)heads * columns * 16 * keys_per_lane(keys); }
bool recurrent_supported(int keys) { return keys > 0 && keys_per_lane(keys) > 0; }

// ---- one token ---------------------------------------------------------------------------------
// grid heads, 1024 threads.  64 columns at a time; the low-rank decay product of the head's channels first, the first columns'
// state requested before it.  Output: o over its root mean square, times norm and silu(gate).
template <int KPL>
__global__ __launch_bounds__(1024) void wkv_step_kernel(const WkvStep a) {
    constexpr int KP = 16 * KPL;
    extern __shared__ __align__(16) float s_low[];  // tanh of the low-rank vector, padded to 64
    __shared__ __align__(16) float s_r[KP], s_k[KP], s_u[KP], s_w[KP];
    __shared__ float s_o[KP], s_v[KP], red[16];
    const int tid = threadIdx.x, sub = tid & 15, grp = tid >> 4, h = blockIdx.x, d = a.dim, hd = a.heads * d;
    float* state = a.state + (int64_t)h * d * KP;
    float S[KPL];
    load_keys<KPL>(S, state + (int64_t)min(grp, d - 1) * KP + sub * KPL);
    const int64_t pos = *a.d_past;
    const int rp = (a.rank + 63) & ~63;
    for (int i = tid; i < rp; i += 1024) s_low[i] = i < a.rank ? tanhf(a.proj[4 * (int64_t)hd + i]) : 0.0f;
    for (int i = tid; i < KP; i += 1024) {
        const bool in = i < d;
        const int64_t c = (int64_t)h * d + i;
        s_r[i] = in ? a.proj[c] : 0.0f;
        s_k[i] = in ? a.proj[hd + c] : 0.0f;
        s_v[i] = in ? a.proj[2 * (int64_t)hd + c] : 0.0f;
        s_u[i] = in ? a.u[c] : 0.0f;
        if (!in) s_w[i] = 0.0f;
    }
    __syncthreads();
    for (int c = grp; c < d; c += 64) {
        const uint16_t* row = a.w2 + ((int64_t)h * d + c) * a.w2_ld;
        float t = 0.0f;
        for (int i = sub * 8; i < rp; i += 128) {
            const u32x4 w = *reinterpret_cast<const u32x4*>(row + i);
            const float4 x0 = *reinterpret_cast<const float4*>(s_low + i), x1 = *reinterpret_cast<const float4*>(s_low + i + 4);
            t = fmaf(bf16_lo(w.x), x0.x, t); t = fmaf(bf16_hi(w.x), x0.y, t); t = fmaf(bf16_lo(w.y), x0.z, t); t = fmaf(bf16_hi(w.y), x0.w, t);
            t = fmaf(bf16_lo(w.z), x1.x, t); t = fmaf(bf16_hi(w.z), x1.y, t); t = fmaf(bf16_lo(w.w), x1.z, t); t = fmaf(bf16_hi(w.w), x1.w, t);
        }
        t = sum16(t);
        if (sub == 0) s_w[c] = expf(-expf(t + a.w0[(int64_t)h * d + c]));
    }
    __syncthreads();
    float r[KPL], k[KPL], u[KPL], w[KPL];
    load_keys<KPL>(r, s_r + sub * KPL);
    load_keys<KPL>(k, s_k + sub * KPL);
    load_keys<KPL>(u, s_u + sub * KPL);
    load_keys<KPL>(w, s_w + sub * KPL);
    for (int c0 = 0; c0 < d; c0 += 64) {
        const int c = c0 + grp;
        float* at = state + (int64_t)min(c, d - 1) * KP + sub * KPL;
        if (c0 > 0) load_keys<KPL>(S, at);
        const float v = s_v[min(c, d - 1)];
        float o = 0.0f;
#pragma unroll
        for (int i = 0; i < KPL; ++i) {
            if (pos == 0) S[i] = 0.0f;
            const float kv = k[i] * v;
            o = fmaf(r[i], fmaf(u[i], kv, S[i]), o);
            S[i] = fmaf(w[i], S[i], kv);
        }
        o = sum16(o);
        if (c < d) {
            store_keys<KPL>(at, S);
            if (sub == 0) s_o[c] = o;
        }
    }
    __syncthreads();
    float ss = 0.0f;
    for (int i = tid; i < d; i += 1024) ss = fmaf(s_o[i], s_o[i], ss);
    const float rn = 1.0f / sqrtf(block_sum<16>(ss, red) / (float)d + a.eps);
    for (int i = tid; i < d; i += 1024) {
        const int64_t c = (int64_t)h * d + i;
        a.out[c] = s_o[i] * rn * a.norm[c] * silu_f(a.proj[3 * (int64_t)hd + c]);
    }
}

// the convolution's output for one channel of a token whose own input is x
__device__ __forceinline__ float conv_step(const SsmShape& m, const float* ring, int channels, int ch, int pos, float x) {
    const float* w = m.conv + (int64_t)ch * m.taps;
    float acc = fmaf(w[m.taps - 1], x, m.conv_b[ch]);
    for (int j0 = 1; j0 < m.taps; j0 += 3) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {  // requested together
            const int j = min(j0 + q, m.taps - 1), p = pos - j;
            const float in = ring[(int64_t)(max(p, 0) % m.taps) * channels + ch], t = w[m.taps - 1 - j];
            acc = fmaf(t, j0 + q < m.taps && p >= 0 ? in : 0.0f, acc);
        }
    }
    return silu_f(acc);
}

// grid (heads, ceil(vdim / 16)), 256 threads: convolution, state update, y * silu(z)
template <int KPL>
__global__ __launch_bounds__(256) void ssm_step_kernel(const SsmStep a) {
    constexpr int KP = 16 * KPL;
    __shared__ __align__(16) float s_b[KP], s_c[KP];
    __shared__ float s_x[16];
    const SsmShape& m = a.m;
    const int tid = threadIdx.x, sub = tid & 15, grp = tid >> 4, h = blockIdx.x, N = m.state, g = h / (m.heads / m.groups);
    const int inner = m.heads * m.vdim, channels = inner + 2 * m.groups * N, c = blockIdx.y * 16 + grp;
    float* state = a.state + ((int64_t)h * m.vdim + min(c, m.vdim - 1)) * KP + sub * KPL;
    float S[KPL];
    load_keys<KPL>(S, state);
    const int pos = (int)*a.d_past;
    float* slot = a.ring + (int64_t)(pos % m.taps) * channels;
    const float *z = a.proj, *x = a.proj + inner;  // x, B and C: the convolution's channels
    const bool writer = h % (m.heads / m.groups) == 0 && blockIdx.y == 0;
    for (int i = tid; i < 2 * KP; i += 256) {
        const int n = i % KP;
        float v = 0.0f;
        if (n < N) {
            const int ch = inner + (i < KP ? 0 : m.groups * N) + g * N + n;
            const float in = x[ch];
            v = conv_step(m, a.ring, channels, ch, pos, in);
            if (writer) slot[ch] = in;
        }
        (i < KP ? s_b : s_c)[n] = v;
    }
    if (tid < 16 && (int)blockIdx.y * 16 + tid < m.vdim) {
        const int ch = h * m.vdim + blockIdx.y * 16 + tid;
        const float in = x[ch];
        s_x[tid] = conv_step(m, a.ring, channels, ch, pos, in);
        slot[ch] = in;
    }
    const float dt = softplus_f(a.proj[inner + channels + h] + m.dt_bias[h]), decay = expf(m.neg_a[h] * dt);
    __syncthreads();
    if (c >= m.vdim) return;
    float B[KPL], C[KPL];
    load_keys<KPL>(B, s_b + sub * KPL);
    load_keys<KPL>(C, s_c + sub * KPL);
    const float xv = s_x[grp], dx = dt * xv;
    float y = 0.0f;
#pragma unroll
    for (int i = 0; i < KPL; ++i) {
        if (pos == 0) S[i] = 0.0f;
        S[i] = fmaf(decay, S[i], B[i] * dx);
        y = fmaf(S[i], C[i], y);
    }
    store_keys<KPL>(state, S);
    y = sum16(y);
    const int64_t at = (int64_t)h * m.vdim + c;
    if (sub == 0) a.out[at] = fmaf(m.D[h], xv, y) * silu_f(z[at]);
}

// ---- prompt rows ---------------------------------------------------------------------------------
// value of lane N of each row of 16 lanes, as an operand of the next instruction
template <int N>
__device__ __forceinline__ float row_lane(float v) { return dpp_f<0x150 + N>(v); }

static int padded_keys(int n) { return 16 * keys_per_lane(n); }

// The scan's o of each row and head over its root mean square, times norm and silu(gate).  It moves memory: four values a lane and G lanes a head where the
// addresses allow, 256 / G heads a workgroup (2048 rows of 40 heads of 64: a wave per head 22.2 us, this 12.9; from 64 values on a wave per head has every
// lane at work, too, and heads of more than 128 have no form here).  grid ceil(rows * heads / (256 / G))
template <bool F32, int G>
__global__ __launch_bounds__(256) void wkv_out_fours_kernel(const WkvRows a) {
    const int at = blockIdx.x * (256 / G) + threadIdx.x / G, row = at / a.heads, h = at % a.heads, d = a.dim, e = 4 * (threadIdx.x % G);
    if (row >= a.M) return;
    const bool in = e < d;
    const int c = h * d + (in ? e : 0);
    const rc_f4 o = *reinterpret_cast<const rc_f4*>(a.o + row * a.o_ld + c), g = *reinterpret_cast<const rc_f4*>(a.proj + row * a.ld + 3 * a.section + c),
                n = *reinterpret_cast<const rc_f4*>(a.norm + c);
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) ss = fmaf(o[i], o[i], ss);
    const float r = 1.0f / sqrtf(sum_lanes<G>(in ? ss : 0.0f) / (float)d + a.eps);
    rc_f4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = o[i] * r * n[i] * silu_f(g[i]);
    if (!in) return;
    if constexpr (F32) *reinterpret_cast<rc_f4*>(static_cast<float*>(a.out) + row * a.out_ld + c) = v;
    else *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + row * a.out_ld + c) =
             make_uint2((uint32_t)f_bf16(v[0]) | ((uint32_t)f_bf16(v[1]) << 16), (uint32_t)f_bf16(v[2]) | ((uint32_t)f_bf16(v[3]) << 16));
}
// the same for any head and alignment, grid (rows, ceil(heads / 4)), a wave per head, NV values a lane
template <bool F32, int NV>
__global__ __launch_bounds__(256) void wkv_out_rows_kernel(const WkvRows a) {
    const int lane = threadIdx.x & 63, h = blockIdx.y * 4 + (threadIdx.x >> 6), d = a.dim;
    if (h >= a.heads) return;
    const float *p = a.proj + blockIdx.x * a.ld + h * d, *o = a.o + blockIdx.x * a.o_ld + h * d;
    float v[NV], g[NV], n[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int e = min(lane + 64 * i, d - 1);
        v[i] = o[e];
        g[i] = p[3 * a.section + e];
        n[i] = a.norm[h * d + e];
    }
    float ss = 0.0f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        v[i] = lane + 64 * i < d ? v[i] : 0.0f;
        ss = fmaf(v[i], v[i], ss);
    }
    const float r = 1.0f / sqrtf(sum64(ss) / (float)d + a.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (lane + 64 * i < d) put_elem<F32>(a.out, blockIdx.x * a.out_ld + h * d + lane + 64 * i, v[i] * r * n[i] * silu_f(g[i]));
}

// grid (rows, ceil(wp / 1024)): the five inputs h + (h' - h) * mu, [5][rows][wp]
template <bool F32>
__global__ __launch_bounds__(256) void token_shift_rows_kernel(const float* __restrict__ h, const float* __restrict__ shift, const float* __restrict__ mu,
                                                               int n, int64_t pos0, int wp, void* __restrict__ out) {
    const int i = (blockIdx.y * 256 + threadIdx.x) * 4;
    if (i >= wp) return;
    const int64_t row = blockIdx.x;
    const float4 x = *reinterpret_cast<const float4*>(h + row * wp + i);
    float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row > 0) p = *reinterpret_cast<const float4*>(h + (row - 1) * wp + i);
    else if (pos0 > 0) p = *reinterpret_cast<const float4*>(shift + (pos0 - 1) % 2 * wp + i);
    const float4 d = make_float4(p.x - x.x, p.y - x.y, p.z - x.z, p.w - x.w);
    for (int s = 0; s < n; ++s) {
        const float4 m = *reinterpret_cast<const float4*>(mu + (int64_t)s * wp + i);
        const float4 v = make_float4(fmaf(d.x, m.x, x.x), fmaf(d.y, m.y, x.y), fmaf(d.z, m.z, x.z), fmaf(d.w, m.w, x.w));
        const int64_t at = ((int64_t)s * gridDim.x + row) * wp + i;
        if constexpr (F32) *reinterpret_cast<float4*>(static_cast<float*>(out) + at) = v;
        else *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + at) =
                 make_uint2((uint32_t)f_bf16(v.x) | ((uint32_t)f_bf16(v.y) << 16), (uint32_t)f_bf16(v.z) | ((uint32_t)f_bf16(v.w) << 16));
    }
}

// grid rows: tanh of the sum of `slabs` partial products, padded with zeros to ld
template <bool F32>
__global__ __launch_bounds__(64) void tanh_rows_kernel(const float* __restrict__ g, int slabs, int64_t slab, int n, int ld, void* __restrict__ out) {
    for (int i = threadIdx.x; i < ld; i += 64) {
        float v = 0.0f;
        if (i < n)
#pragma unroll 4
            for (int z = 0; z < slabs; ++z) v += g[z * slab + (int64_t)blockIdx.x * ld + i];
        put_elem<F32>(out, (int64_t)blockIdx.x * ld + i, tanhf(v));
    }
}

// Where x, B and C of a convolved row lie: x, then B and C of every group, each padded to 4, then sixteen zeros, which stand for the keys that the matrix
// products have beyond these (and end the 16 columns of the last head).  All padding is zeros.  Padded to the keys of the products instead, up to 64 for one,
// a row of thousands of small groups is megabytes, and 2048 of them pass the 32 bits of an offset.
__host__ __device__ inline int conv_x(const SsmShape& m) { return (m.heads * m.vdim + 3) & ~3; }
__host__ __device__ inline int conv_keys(const SsmShape& m) { return (m.state + 3) & ~3; }
int64_t ssm_conv_row(const SsmShape& m) { return conv_x(m) + 2 * (int64_t)m.groups * conv_keys(m) + 16; }
// per 16 tokens and head: what the tokens take from each other [16 from][16 to], the state's decay up to each, each one's share of the new state
constexpr int SSM_TILE = 288;
int64_t ssm_tile_floats(int heads, int rows) { return (int64_t)((rows + 15) / 16) * heads * SSM_TILE; }

// grid (ceil(rows / 8), ceil(row / 256) + 1): convolution and silu of x, B and C, eight rows per thread; the last column of workgroups leaves
// decay and dt, [rows][2][heads]
constexpr int CONV_ROWS = 8;
__global__ __launch_bounds__(256) void ssm_conv_rows_kernel(const SsmRows a) {
    const SsmShape& m = a.m;
    const int inner = m.heads * m.vdim, channels = inner + 2 * m.groups * m.state, r0 = blockIdx.x * CONV_ROWS, rows = min(CONV_ROWS, a.M - r0);
    if (blockIdx.y == gridDim.y - 1) {
        for (int i = threadIdx.x; i < rows * m.heads; i += 256) {
            const int64_t row = r0 + i / m.heads;
            const int h = i % m.heads;
            const float dt = softplus_f(a.proj[row * a.ld + inner + channels + h] + m.dt_bias[h]);
            a.decay[row * 2 * m.heads + h] = expf(m.neg_a[h] * dt);
            a.decay[(row * 2 + 1) * m.heads + h] = dt;
        }
        return;
    }
    const int at = blockIdx.y * 256 + threadIdx.x;
    if (at >= a.conv_ld) return;
    int ch = at;
    if (at >= conv_x(m)) {
        const int keys = conv_keys(m), q = at - conv_x(m), n = q % keys;
        ch = n < m.state && q / keys < 2 * m.groups ? inner + q / keys * m.state + n : channels;
    } else if (at >= inner) ch = channels;
    if (ch == channels) {
        for (int r = 0; r < rows; ++r) a.conv[(int64_t)(r0 + r) * a.conv_ld + at] = 0.0f;
        return;
    }
    const float *x = a.proj + inner + ch, *w = m.conv + (int64_t)ch * m.taps, bias = m.conv_b[ch];
    auto input = [&](int row) {  // of row r0 + row, also of rows and positions before
        const int64_t p = a.pos0 + r0 + row;
        return r0 + row >= 0 ? x[(int64_t)min(r0 + row, a.M - 1) * a.ld] : p >= 0 ? a.ring[p % m.taps * channels + ch] : 0.0f;
    };
    float* out = a.conv + (int64_t)r0 * a.conv_ld + at;
    if (m.taps <= 4) {
        float in[CONV_ROWS + 3], t[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) t[j] = j < m.taps ? w[m.taps - 1 - j] : 0.0f;
#pragma unroll
        for (int i = 0; i < CONV_ROWS + 3; ++i) in[i] = 3 - i < m.taps ? input(i - 3) : 0.0f;
#pragma unroll
        for (int r = 0; r < CONV_ROWS; ++r)
            if (r < rows) out[(int64_t)r * a.conv_ld] = silu_f(fmaf(t[3], in[r], fmaf(t[2], in[r + 1], fmaf(t[1], in[r + 2], fmaf(t[0], in[r + 3], bias)))));
    } else {
        for (int r = 0; r < rows; ++r) {
            float acc = bias;
            for (int j = 0; j < m.taps; ++j) acc = fmaf(w[m.taps - 1 - j], input(r - j), acc);
            out[(int64_t)r * a.conv_ld] = silu_f(acc);
        }
    }
}

// What 16 tokens of a head take from each other: M[s][t] = (C_t . B_s) dt_s prod(s < q <= t) decay_q, with the skip D on the diagonal, the products P_t =
// prod(q <= t) and Q_s = dt_s prod(q > s) beside it.  Products of decays, never quotients.  grid (ceil(rows / 16), ceil(heads of a group / 4 each),
// groups), `each` heads a wave (ssm_rows); tokens past the last
// leave everything as it is.
__global__ __launch_bounds__(256) void ssm_tiles_kernel(const SsmRows a, int each) {
    const SsmShape& m = a.m;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, j = lane & 15, g4 = lane >> 4, t0 = blockIdx.x * 16, per = m.heads / m.groups;
    const int first = (blockIdx.y * 4 + wave) * each, end = min(first + each, per);
    if (first >= per) return;
    const int64_t row = (int64_t)min(t0 + j, a.M - 1);
    const bool here = t0 + j < a.M;
    float next_decay, next_Q, next_dt[4], next_skip;
    auto fetch = [&](int in_group) {
        const int h = blockIdx.z * per + in_group;
        const float* step = a.decay + h;
        next_decay = step[row * 2 * m.heads];
        next_Q = step[(row * 2 + 1) * m.heads];
#pragma unroll
        for (int i = 0; i < 4; ++i) next_dt[i] = step[((int64_t)min(t0 + 4 * g4 + i, a.M - 1) * 2 + 1) * m.heads];
        next_skip = m.D[h];
    };
    fetch(first);
    const float* conv = a.conv + row * a.conv_ld;
    const int keys = conv_keys(m), b_at = conv_x(m) + blockIdx.z * keys, c_at = b_at + m.groups * keys, zeros = (int)a.conv_ld - 4;
    rc_f4 dot = {0.f, 0.f, 0.f, 0.f}, odd = dot;  // rows s = 4 g4 + i, column t = j
    for (int k = 0; k < a.keys; k += 64) {
        rc_f4 B[4], C[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int key = k + 16 * i + 4 * g4;
            B[i] = *reinterpret_cast<const rc_f4*>(conv + (key < keys ? b_at + key : zeros));
            C[i] = *reinterpret_cast<const rc_f4*>(conv + (key < keys ? c_at + key : zeros));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                dot = __builtin_amdgcn_mfma_f32_16x16x4f32(B[i][e], C[i][e], dot, 0, 0, 0);
                odd = __builtin_amdgcn_mfma_f32_16x16x4f32(B[i][e + 1], C[i][e + 1], odd, 0, 0, 0);
            }
    }
    dot += odd;
    for (int n = first; n < end; ++n) {
        const int h = blockIdx.z * per + n;
        const float decay = here ? next_decay : 1.0f, skip = next_skip, dt[4] = {next_dt[0], next_dt[1], next_dt[2], next_dt[3]};
        float p[4] = {1.f, 1.f, 1.f, 1.f}, P = 1.0f, Q = here ? next_Q : 0.0f;
        if (n + 1 < end) fetch(n + 1);
        static_for<16>([&](auto T) {
            constexpr int q = decltype(T)::value;
            const float d = row_lane<q>(decay), to = q <= j ? d : 1.0f;
            P *= to;
            Q *= q > j ? d : 1.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) p[i] *= q > 4 * g4 + i ? to : 1.0f;
        });
        float* out = a.tiles + ((int64_t)h * gridDim.x + blockIdx.x) * SSM_TILE;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int from = 4 * g4 + i;
            const float v = dot[i] * (dt[i] * p[i]);
            out[16 * from + j] = from > j || t0 + from >= a.M ? 0.0f : from == j ? v + skip : v;
        }
        if (g4 == 0) {
            out[256 + j] = P;
            out[272 + j] = Q;
        }
    }
}

constexpr int scan_tile_lds(int keys) { return 128 * keys + 4096 + 1024; }
constexpr int scan_stages(int keys) { return keys <= 128 ? 4 : keys <= 256 ? 3 : 2; }
static int scan_lds(int waves, int keys) { return 2048 * waves + scan_stages(keys) * scan_tile_lds(keys); }

// What a scan over the tokens reads and leaves for one head and 16 columns from c0 on.
struct Scan {
    int M, tiles, columns, c0;
    bool from_zero;
    const float* bc;            // SSM: rows of B and C, `bc_step` bytes a token (all tokens in 32 bits), at bytes b_at and c_at.  WKV: the tiles
    uint32_t bc_step, b_at, c_at, zeros_at;
    int pieces;                 // SSM: 16-byte pieces of B; the others are at zeros_at
    const float* pairs;         // SSM: M, P and Q of each tile.  WKV: M and the keys' decays, behind the rows of the tiles
    uint32_t tile_bytes;        // from one tile's to the next's
    const float* x;
    uint32_t x_step, x_at;
    float* state;               // of the head's first column
    float* y;                   // of the head's first column
    int64_t y_ld;
};
constexpr int wkv_tile(int keys) { return 33 * keys + 256; }  // floats: [16][k | r] with the decays to the tile's edges, M, the decays of the whole tile

// The state goes from 16 tokens to the next 16 on v_mfma_f32_16x16x4_f32:
//   ssm  y_t = P_t (C_t S) + sum(s <= t) M[s][t] x_s,  S <- P_15 S + sum(s) B_s Q_s x_s
//   wkv  the same with the decays inside r and k (C and B) and per key in front of S, and the bonus on M's diagonal
// A wave has 16 columns and KT tiles of 16 keys of the state, as sums (row r of tile q is key KT r + q of the wave's), which are, register by
// register, also the operand of C S.  The waves' sums meet in LDS.
// A tile of tokens comes through LDS, STAGES of them in flight, with full instructions (B and C: 16-byte pieces, piece ^ row).
// What bounds it: a turn (0.65 us) has 544 clocks of MFMAs on a SIMD and as many of LDS traffic on the CU, behind a barrier for the waves' sums; 40 heads are
// 160 workgroups.  SSM, 2048 tokens of 40 heads of 64, 128 keys: 89 us, 11 for the tiles in front; token by token on the vector units 217.  Four waves of
// twice the keys 98, operands from memory straight to registers 104 (without loads 63, without the barrier 75).
// WKV, 2048 tokens of 40 heads of 64: 64 us, 31 for the tiles in front; token by token, with a slab of sums per 16 keys, 157 and 9 more to add the slabs.
template <int W, int KT, bool WKV>
__device__ __forceinline__ void scan_columns(const Scan& a, uint8_t* ss_lds) {
    constexpr int KP = 16 * W * KT, ROW = KP / 2, STAGES = scan_stages(KP), TILE = scan_tile_lds(KP), BC = 128 * KP;  // ROW: pieces of a row's B and C
    constexpr int BCI = 2 * KT, PER = W == 8 ? BCI + 1 : BCI + 2;  // a wave's instructions for B and C of a tile, for all of it
    constexpr int PIECES = WKV ? 16 + KP / 16 : 18;               // a wave's share of M and what lies behind it
    // LDS: s_y, then the tiles: B and C, M and what lies behind it, x
    float (*s_y)[W][256] = reinterpret_cast<float (*)[W][256]>(ss_lds);
    constexpr int TILES = 2 * W * 1024;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), w4 = wave & 3, j = lane & 15, g4 = lane >> 4;
    const int c0 = a.c0, c = min(c0 + j, a.columns - 1), tiles = a.tiles;
    float* state = a.state + (int64_t)c * KP + 16 * KT * wave + 4 * KT * g4;
    rc_f4 S[KT];
    {
        float keys[4 * KT];
        load_keys<4 * KT>(keys, state);
#pragma unroll
        for (int q = 0; q < KT; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) S[q][i] = a.from_zero ? 0.0f : keys[KT * i + q];
    }
    // memory -> LDS; rows past the last repeat it and are taken out again in registers, columns of x past the last are what lies there and are not stored
    const uint32_t last = (uint32_t)(a.M - 1) * a.bc_step, x_last = (uint32_t)(a.M - 1) * a.x_step;
    const gt_i4 rows = gt_buffer(a.bc), pairs = gt_buffer(a.pairs), xs = gt_buffer(a.x);
    const uint32_t lds0 = (uint32_t)(uintptr_t)ss_lds + TILES;
    uint32_t row_of[BCI], col_of[BCI];
#pragma unroll
    for (int i = 0; i < BCI; ++i) {
        const int p = (BCI * wave + i) * 64 + lane, q = (p % ROW) ^ (p / ROW & 15), of = q % (ROW / 2);
        row_of[i] = p / ROW * (WKV ? 16 * ROW : a.bc_step);
        col_of[i] = WKV ? 16 * q : of < a.pieces ? (q < ROW / 2 ? a.b_at : a.c_at) + 16 * of : a.zeros_at;
    }
    const uint32_t x_row = (4 * g4 + w4) * a.x_step, x_col = a.x_at + 4 * (c0 + j), pair_at = 16 * (PIECES * w4 + min(lane, PIECES - 1));
    auto fetch = [&](int n, int i) {
        const uint32_t at = __builtin_amdgcn_readfirstlane(lds0 + n % STAGES * TILE);
        if (i < BCI) {
            if constexpr (WKV) gt_to_lds(at + (BCI * wave + i) * 1024, (int)(row_of[i] + col_of[i]), rows, n * a.tile_bytes);
            else gt_to_lds(at + (BCI * wave + i) * 1024, (int)(min(16 * n * a.bc_step + row_of[i], last) + col_of[i]), rows, 0);
        } else if (W == 8 ? wave < 4 : i == BCI) gt_to_lds(at + BC + w4 * 1024, (int)pair_at, pairs, n * a.tile_bytes);
        else gt_word_to_lds(at + BC + 4096 + w4 * 256, (int)(min(16 * n * a.x_step + x_row, x_last) + x_col), xs, 0);
    };
    // LDS -> registers
    struct Tile {
        rc_f4 P, Q;
        float C[4 * KT], B[4][KT], x[4], xw, from, end, decay[4 * KT];  // P, Q and end: SSM; decay: WKV
    } T0, T1;
    auto pair = [&](int f) { return BC + f / (4 * PIECES) * 1024 + f % (4 * PIECES) * 4; };  // where float f of M and what lies behind it is in a tile
    const int from_at = pair(16 * (4 * g4 + w4) + j), p_at = pair(256 + 4 * g4), q_at = pair(272 + 4 * g4), end_at = pair(271);
    int decay_at[KT];
#pragma unroll
    for (int q = 0; q < KT; ++q) decay_at[q] = pair(256 + 16 * KT * wave + 4 * KT * g4 + 4 * q);
    const int x_at = BC + 4096 + 64 * g4 + 4 * j;                        // of row 4 g4: row 4 g4 + i 256 i further on
    constexpr int READS = KT + 6;
    auto read = [&](Tile& v, int n, int part) {
        const uint8_t* t = ss_lds + TILES + n % STAGES * TILE;
        if (part < KT) {
            const int q = part;
            const float4 x = *reinterpret_cast<const float4*>(t + (j * ROW + ((ROW / 2 + (4 * wave + g4) * KT + q) ^ j)) * 16);
            v.C[4 * q] = x.x; v.C[4 * q + 1] = x.y; v.C[4 * q + 2] = x.z; v.C[4 * q + 3] = x.w;
        } else if (part < KT + 4) {
            const int i = part - KT, r = 4 * g4 + i, k = (16 * wave + j) * KT;
            const uint8_t* b = t + (r * ROW + ((k >> 2) ^ r)) * 16 + (k & 3) * 4;
            if constexpr (KT == 1) v.B[i][0] = *reinterpret_cast<const float*>(b);
            else if constexpr (KT == 2) {
                const float2 x = *reinterpret_cast<const float2*>(b);
                v.B[i][0] = x.x; v.B[i][1] = x.y;
            } else {
                const float4 x = *reinterpret_cast<const float4*>(b);
                v.B[i][0] = x.x; v.B[i][1] = x.y; v.B[i][2] = x.z; v.B[i][3] = x.w;
            }
            v.x[i] = *reinterpret_cast<const float*>(t + x_at + 256 * i);
        } else if (part == KT + 4) {
            v.xw = *reinterpret_cast<const float*>(t + x_at + 256 * w4);
            v.from = *reinterpret_cast<const float*>(t + from_at);
            if constexpr (!WKV) v.end = *reinterpret_cast<const float*>(t + end_at);
        } else if constexpr (WKV) {
#pragma unroll
            for (int q = 0; q < KT; ++q) {
                const float4 x = *reinterpret_cast<const float4*>(t + decay_at[q]);
                v.decay[4 * q] = x.x; v.decay[4 * q + 1] = x.y; v.decay[4 * q + 2] = x.z; v.decay[4 * q + 3] = x.w;
            }
        } else {
            v.P = *reinterpret_cast<const rc_f4*>(t + p_at);
            v.Q = *reinterpret_cast<const rc_f4*>(t + q_at);
        }
    };
    // the waves' sums of a tile (waves 0 .. 3), on their way from LDS while the next tile is used
    float sums[W];
    auto read_sums = [&](int n) {
        if (wave < 4)
#pragma unroll
            for (int w = 0; w < W; ++w) sums[w] = s_y[n & 1][w][tid & 255];
    };
    const bool stored = tid < 256 && c0 + j < a.columns;
    float* y = a.y + (int64_t)(tid >> 4 & 15) * a.y_ld + c0 + j;
    auto put = [&](int n) {
        if (!stored || 16 * n + (tid >> 4) >= a.M) return;
        float v = (sums[0] + sums[1]) + (sums[2] + sums[3]);
        if constexpr (W == 8) v += (sums[4] + sums[5]) + (sums[6] + sums[7]);
        y[(int64_t)16 * n * a.y_ld] = v;
    };
    auto run = [&](Tile& v, Tile& next, int n) {
        // the next tile has arrived in every wave's part; the one used now lies in registers, and its LDS takes one more
        if (n + STAGES - 1 < tiles) gt_arrived<(STAGES - 2) * PER>();
        else gt_arrived<0>();
        if (16 * n + 16 > a.M)  // what repeats the last row may be infinite, and a factor of zero does not take it out of the state
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (16 * n + 4 * g4 + i >= a.M) {
                    v.x[i] = 0.0f;
                    if constexpr (!WKV)  // (their k are zeros in the tiles)
#pragma unroll
                        for (int q = 0; q < KT; ++q) v.B[i][q] = 0.0f;
                }
        rc_f4 old[KT], here = {0.f, 0.f, 0.f, 0.f}, next_S[KT];
        float dx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) dx[i] = WKV ? v.x[i] : v.x[i] * v.Q[i];
#pragma unroll
        for (int q = 0; q < KT; ++q) {
            old[q] = rc_f4{0.f, 0.f, 0.f, 0.f};
            if constexpr (WKV) {
#pragma unroll
                for (int i = 0; i < 4; ++i) next_S[q][i] = S[q][i] * v.decay[KT * i + q];
            } else next_S[q] = S[q] * v.end;
        }
        // sums that do not depend on each other take turns, and what is read and requested for later tiles goes out between them
        constexpr int OPS = 1 + READS + PER, SLOTS = 4 * KT;
        const bool more = n + STAGES < tiles;
        auto between = [&](int slot) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int o = 0; o < OPS; ++o)
                if (o * SLOTS / OPS == slot) {
                    if (o == 0) read_sums(n + 1);  // n - 1
                    else if (o <= READS) read(next, n + 1, o - 1);
                    else if (more) fetch(n + STAGES, o - 1 - READS);
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        if (wave < 4) here = __builtin_amdgcn_mfma_f32_16x16x4f32(v.from, v.xw, here, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < KT; ++q) {
                old[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.C[KT * i + q], S[q][i], old[q], 0, 0, 0);
                next_S[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.B[i][q], dx[i], next_S[q], 0, 0, 0);
                between(KT * i + q);
            }
        if (n > 0) put(n - 1);
#pragma unroll
        for (int q = 0; q < KT; ++q) S[q] = next_S[q];
#pragma unroll
        for (int q = 1; q < KT; ++q) old[0] += old[q];
        if (__builtin_expect(wave < 4 && __builtin_amdgcn_ballot_w64(!(fabsf(v.xw) < INFINITY)) != 0, 0)) {  // 0 times infinity: no token takes from a later one
            here = rc_f4{0.f, 0.f, 0.f, 0.f};
            const float* t = a.pairs + (int64_t)n * (a.tile_bytes / 4);
            for (int b = 0; b < 4; ++b) {
                const float xs = __shfl(v.xw, 16 * b + j, 64);
                const int from = 4 * b + wave;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (from <= 4 * g4 + i) here[i] = fmaf(t[16 * from + 4 * g4 + i], xs, here[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) s_y[n & 1][wave][16 * (4 * g4 + i) + j] = WKV ? old[0][i] + here[i] : fmaf(v.P[i], old[0][i], here[i]);
    };
#pragma unroll
    for (int n = 0; n < STAGES; ++n)
        if (n < tiles)
#pragma unroll
            for (int i = 0; i < PER; ++i) fetch(n, i);
    if (tiles >= STAGES) gt_arrived<(STAGES - 1) * PER>();
    else gt_arrived<0>();
#pragma unroll
    for (int i = 0; i < READS; ++i) read(T0, 0, i);
    for (int n = 0; n < tiles; n += 2) {
        run(T0, T1, n);
        if (n + 1 < tiles) run(T1, T0, n + 1);
    }
    __syncthreads();
    read_sums(tiles - 1);
    put(tiles - 1);
    if (c0 + j < a.columns) {
        float keys[4 * KT];
#pragma unroll
        for (int q = 0; q < KT; ++q)
#pragma unroll
            for (int i = 0; i < 4; ++i) keys[KT * i + q] = S[q][i];
        store_keys<4 * KT>(state, keys);
    }
}


// grid (heads, ceil(vdim / 16)), W waves
template <int W, int KT>
__global__ __launch_bounds__(64 * W, 1) void ssm_scan_kernel(const SsmRows a) {
    extern __shared__ __align__(16) uint8_t scan_mem[];
    const SsmShape& m = a.m;
    const int tid = threadIdx.x, h = blockIdx.x, N = m.state, per = m.heads / m.groups, g = h / per, inner = m.heads * m.vdim, channels = inner + 2 * m.groups * N;
    const int c0 = blockIdx.y * 16;
    // the ring takes the inputs of the last positions
    for (int q = 0; q < m.taps && q < a.M; ++q) {
        const float* row = a.proj + (int64_t)(a.M - 1 - q) * a.ld + inner;
        float* slot = a.ring + (a.pos0 + a.M - 1 - q) % m.taps * channels;
        if (tid < 16 && c0 + tid < m.vdim) slot[h * m.vdim + c0 + tid] = row[h * m.vdim + c0 + tid];
        if (h % per == 0 && blockIdx.y == 0)
            for (int i = tid; i < 2 * N; i += 64 * W) {
                const int ch = inner + (i < N ? 0 : m.groups * N) + g * N + i % N;
                slot[ch] = row[ch];
            }
    }
    Scan s;
    s.M = a.M;
    s.tiles = (a.M + 15) / 16;
    s.columns = m.vdim;
    s.c0 = c0;
    s.from_zero = a.pos0 == 0;
    s.bc = s.x = a.conv;
    s.bc_step = s.x_step = (uint32_t)a.conv_ld * 4;
    s.b_at = 4 * (conv_x(m) + g * conv_keys(m));
    s.c_at = 4 * (conv_x(m) + (m.groups + g) * conv_keys(m));
    s.zeros_at = s.bc_step - 16;
    s.pieces = conv_keys(m) / 4;
    s.pairs = a.tiles + (int64_t)h * s.tiles * SSM_TILE;
    s.tile_bytes = SSM_TILE * 4;
    s.x_at = 4 * h * m.vdim;
    s.state = a.state + (int64_t)h * m.vdim * a.keys;
    s.y = a.y + h * m.vdim;
    s.y_ld = inner;
    scan_columns<W, KT, false>(s, scan_mem);
}

// What 16 tokens of a head take from each other, and their r and k with the decays to the edges of the tile.  M[s][t] = sum over keys of
// r_t k_s prod(s < q < t) w_q, the bonus r_t u k_s on its diagonal.  A pair of tokens meets at one size B of 1, 2, 4 and 8: the highest bit in which
// their places differ.  There the product is that of the decays behind s in its block of B times those in front of t in the next: products of
// decays, never quotients, and one matrix product a size.  It moves memory (2048 rows of 40 heads of 64: 63 MB in, 47 out, 31 us).
// grid (ceil(rows / 16), heads), four waves that share the keys; tokens past the last leave everything as it is.
__global__ __launch_bounds__(256) void wkv_tiles_kernel(const WkvRows a) {
    __shared__ float s_m[4][256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 15, g4 = lane >> 4, t0 = blockIdx.x * 16, h = blockIdx.y, d = a.dim, kp = a.keys;
    const bool here = t0 + j < a.M, fours = !((d | a.ld | a.section) & 3) && !(reinterpret_cast<uintptr_t>(a.u) & 15);
    const float *p = a.proj + (int64_t)min(t0 + j, a.M - 1) * a.ld + h * d, *u = a.u + h * d;
    float* out = a.tiles + ((int64_t)h * gridDim.x + blockIdx.x) * wkv_tile(kp);
    float m[4] = {0.f, 0.f, 0.f, 0.f};  // from 4 g4 + i to j
    for (int k0 = 16 * wave; k0 < kp; k0 += 64) {
        const int key = k0 + 4 * g4;
        rc_f4 r, k, w, b;
        if (fours) {
            const int at = min(key, d - 4);
            r = *reinterpret_cast<const rc_f4*>(p + at);
            k = *reinterpret_cast<const rc_f4*>(p + a.section + at);
            w = *reinterpret_cast<const rc_f4*>(p + 4 * a.section + at);
            b = *reinterpret_cast<const rc_f4*>(u + at);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int at = min(key + i, d - 1);
                r[i] = p[at];
                k[i] = p[a.section + at];
                w[i] = p[4 * a.section + at];
                b[i] = u[at];
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const bool in = here && key + i < d;
            r[i] = in ? r[i] : 0.0f;
            k[i] = in ? k[i] : 0.0f;
            w[i] = in ? w[i] : 1.0f;
            b[i] = key + i < d ? b[i] : 0.0f;
        }
        rc_f4 dot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) dot = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i] * b[i], r[i], dot, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) m[i] += 4 * g4 + i == j ? dot[i] : 0.0f;
        static_for<4>([&](auto L) {  // r and k: with the decays in front of and behind the token in its block of B, w: those of the whole block
            constexpr int B = 1 << decltype(L)::value, other = B == 1 ? 0xB1 : B == 2 ? 0x4E : B == 4 ? 0x141 : 0x140;
            rc_f4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i], r[i], sum, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int from = 4 * g4 + i;
                m[i] += ((from ^ j) & ~(2 * B - 1)) == 0 && !(from & B) && (j & B) ? sum[i] : 0.0f;
                const float next = dpp_f<other>(w[i]);
                r[i] *= j & B ? next : 1.0f;
                k[i] *= j & B ? 1.0f : next;
                w[i] *= next;
            }
        });
        *reinterpret_cast<rc_f4*>(out + j * 2 * kp + key) = k;
        *reinterpret_cast<rc_f4*>(out + j * 2 * kp + kp + key) = r;
        if (j == 0) *reinterpret_cast<rc_f4*>(out + 32 * kp + 256 + key) = w;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s_m[wave][16 * (4 * g4 + i) + j] = m[i];
    __syncthreads();
    out[32 * kp + tid] = (s_m[0][tid] + s_m[1][tid]) + (s_m[2][tid] + s_m[3][tid]);
}

// grid (heads, ceil(dim / 16)), W waves
template <int W, int KT>
__global__ __launch_bounds__(64 * W, 1) void wkv_scan_kernel(const WkvRows a) {
    extern __shared__ __align__(16) uint8_t scan_mem[];
    const int h = blockIdx.x;
    if (h == 0 && blockIdx.y == 0)  // the next token's shift reads the last row
        for (int i = threadIdx.x; i < a.wp; i += 64 * W) a.shift[(a.pos0 + a.M - 1) % 2 * a.wp + i] = a.h_last[i];
    Scan s;
    s.M = a.M;
    s.tiles = (a.M + 15) / 16;
    s.columns = a.dim;
    s.c0 = blockIdx.y * 16;
    s.from_zero = a.pos0 == 0;
    s.tile_bytes = wkv_tile(a.keys) * 4;
    s.bc = a.tiles + (int64_t)h * s.tiles * wkv_tile(a.keys);
    s.bc_step = s.b_at = s.c_at = s.zeros_at = 0;
    s.pieces = 0;
    s.pairs = s.bc + 32 * a.keys;
    s.x = a.proj;
    s.x_step = (uint32_t)a.ld * 4;
    s.x_at = (uint32_t)(2 * a.section + h * a.dim) * 4;
    s.state = a.state + (int64_t)h * a.dim * a.keys;
    s.y = a.o + h * a.dim;
    s.y_ld = a.o_ld;
    scan_columns<W, KT, true>(s, scan_mem);
}

// grid rows: the scan's y * silu(z), normed in equal parts, times norm and the branch's scale.  All that a row reads goes out together (2560 values, each
// piece's loads behind the use of the one before: 16 rows 10.3 us, 2048 24).
template <bool F32>
__global__ __launch_bounds__(256) void ssm_out_rows_kernel(const SsmRows a) {
    __shared__ float red[4];
    const SsmShape& m = a.m;
    const int tid = threadIdx.x, inner = m.heads * m.vdim, part = inner / m.norm_groups;
    const float *y = a.y + (int64_t)blockIdx.x * inner, *z = a.proj + blockIdx.x * a.ld;
    constexpr int NS = 16;  // values kept in registers: parts of up to 4096
    const int pieces = min((part + 255) / 256, NS);
    for (int p = 0; p < m.norm_groups; ++p) {
        const int c0 = p * part;
        float v[NS], g[NS], n[NS], ss = 0.0f;
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (i < pieces) {
                const int c = c0 + min(tid + 256 * i, part - 1);
                v[i] = y[c];
                g[i] = z[c];
                n[i] = m.norm[c];
            }
        issue_order_fence();
#pragma unroll
        for (int i = 0; i < NS; ++i)
            if (i < pieces) {
                v[i] = tid + 256 * i < part ? v[i] * silu_f(g[i]) : 0.0f;
                ss = fmaf(v[i], v[i], ss);
            }
        for (int c = tid + 256 * NS; c < part; c += 256) {
            const float t = y[c0 + c] * silu_f(z[c0 + c]);
            ss = fmaf(t, t, ss);
        }
        const float r = 1.0f / sqrtf(block_sum<4>(ss, red) / (float)part + a.eps) * m.scale;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int c = tid + 256 * i;
            if (c < part) put_elem<F32>(a.out, blockIdx.x * a.out_ld + c0 + c, v[i] * r * n[i]);
        }
        for (int c = tid + 256 * NS; c < part; c += 256) put_elem<F32>(a.out, blockIdx.x * a.out_ld + c0 + c, y[c0 + c] * silu_f(z[c0 + c]) * r * m.norm[c0 + c]);
    }
}

// ---- launches ------------------------------------------------------------------------------------
#define PTM_KPL(n, LAUNCH)                                 \
    switch (keys_per_lane(n)) {                            \
        case 4: LAUNCH(4); break;                          \
        case 8: LAUNCH(8); break;                          \
        case 16: LAUNCH(16); break;                        \
        case 32: LAUNCH(32); break;                        \
        default: return PTM_E_UNSUPPORTED;                 \
    }

int wkv_step(const WkvStep& a, hipStream_t s) {
    const size_t lds = (size_t)up64(a.rank) * 4;
    if (a.rank > 8192) return PTM_E_UNSUPPORTED;
#define PTM_RUN(KPL) hipLaunchKernelGGL(wkv_step_kernel<KPL>, dim3(a.heads), dim3(1024), lds, s, a)
    PTM_KPL(a.dim, PTM_RUN)
#undef PTM_RUN
    return launch_status();
}

int ssm_step(const SsmStep& a, hipStream_t s) {
    const dim3 grid(a.m.heads, (a.m.vdim + 15) / 16);
#define PTM_RUN(KPL) hipLaunchKernelGGL(ssm_step_kernel<KPL>, grid, dim3(256), 0, s, a)
    PTM_KPL(a.m.state, PTM_RUN)
#undef PTM_RUN
    return launch_status();
}

int token_shift_rows(const float* h, const float* shift, const float* mu, int n, int rows, int64_t pos0, int wp, bool fp32, void* out, hipStream_t s) {
    const dim3 grid(rows, (wp + 1023) / 1024);
    if (fp32) hipLaunchKernelGGL(token_shift_rows_kernel<true>, grid, dim3(256), 0, s, h, shift, mu, n, pos0, wp, out);
    else hipLaunchKernelGGL(token_shift_rows_kernel<false>, grid, dim3(256), 0, s, h, shift, mu, n, pos0, wp, out);
    return launch_status();
}

int tanh_rows(const float* g, int slabs, int64_t slab, int rows, int n, bool fp32, void* out, hipStream_t s) {
    if (fp32) hipLaunchKernelGGL(tanh_rows_kernel<true>, dim3(rows), dim3(64), 0, s, g, slabs, slab, n, up64(n), out);
    else hipLaunchKernelGGL(tanh_rows_kernel<false>, dim3(rows), dim3(64), 0, s, g, slabs, slab, n, up64(n), out);
    return launch_status();
}

int64_t wkv_tile_floats(int heads, int dim, int rows) { return (int64_t)((rows + 15) / 16) * heads * wkv_tile(padded_keys(dim)); }

int wkv_rows(WkvRows a, bool fp32, hipStream_t s) {
    if (!recurrent_supported(a.dim)) return PTM_E_UNSUPPORTED;
    if (a.M * a.ld >= (int64_t)1 << 30) return PTM_E_UNSUPPORTED;  // 32-bit offsets of the scan; not reached by 2048 rows of what a decoder accepts
    a.keys = padded_keys(a.dim);
    hipLaunchKernelGGL(wkv_tiles_kernel, dim3((a.M + 15) / 16, a.heads), dim3(256), 0, s, a);
    static std::once_flag raised;
    std::call_once(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&wkv_scan_kernel<8, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 128));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&wkv_scan_kernel<8, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 256));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&wkv_scan_kernel<8, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 512));
    });
    const dim3 grid(a.heads, (a.dim + 15) / 16);
#define PTM_RUN(W, KT) hipLaunchKernelGGL((wkv_scan_kernel<W, KT>), grid, dim3(64 * W), scan_lds(W, a.keys), s, a)
    switch (a.keys) {
        case 64: PTM_RUN(4, 1); break;
        case 128: PTM_RUN(8, 1); break;
        case 256: PTM_RUN(8, 2); break;
        default: PTM_RUN(8, 4);
    }
#undef PTM_RUN
    const bool fours = !((a.dim | a.ld | a.section | a.o_ld | a.out_ld) & 3) &&
                       !((reinterpret_cast<uintptr_t>(a.o) | reinterpret_cast<uintptr_t>(a.proj) | reinterpret_cast<uintptr_t>(a.norm) | reinterpret_cast<uintptr_t>(a.out)) & 15);
    const dim3 out_grid(a.M, (a.heads + 3) / 4);
#define PTM_FOURS(G)                                                                                                                                         \
    if (fp32) hipLaunchKernelGGL((wkv_out_fours_kernel<true, G>), dim3((unsigned)(((int64_t)a.M * a.heads * G + 255) / 256)), dim3(256), 0, s, a);           \
    else hipLaunchKernelGGL((wkv_out_fours_kernel<false, G>), dim3((unsigned)(((int64_t)a.M * a.heads * G + 255) / 256)), dim3(256), 0, s, a)
#define PTM_RUN(NV)                                                                                                  \
    if (fp32) hipLaunchKernelGGL((wkv_out_rows_kernel<true, NV>), out_grid, dim3(256), 0, s, a);                     \
    else hipLaunchKernelGGL((wkv_out_rows_kernel<false, NV>), out_grid, dim3(256), 0, s, a)
    if (fours && a.dim <= 64) { PTM_FOURS(16); }
    else if (fours && a.dim <= 128) { PTM_FOURS(32); }
    else if (a.dim <= 64) { PTM_RUN(1); }
    else if (a.dim <= 128) { PTM_RUN(2); }
    else { PTM_RUN(8); }
#undef PTM_FOURS
#undef PTM_RUN
    return launch_status();
}

int ssm_rows(SsmRows a, bool fp32, hipStream_t s) {
    const SsmShape& m = a.m;
    if (!recurrent_supported(m.state)) return PTM_E_UNSUPPORTED;
    a.keys = padded_keys(m.state);
    a.conv_ld = ssm_conv_row(m);
    if (a.M * a.conv_ld >= (int64_t)1 << 30) return PTM_E_UNSUPPORTED;  // 32-bit offsets of the scan; not reached by 2048 rows of what a decoder accepts
    hipLaunchKernelGGL(ssm_conv_rows_kernel, dim3((a.M + CONV_ROWS - 1) / CONV_ROWS, (unsigned)((a.conv_ld + 255) / 256 + 1)), dim3(256), 0, s, a);
    // One head a wave, or two, which read B and C once: 128 keys, 16 to 1600 heads of tiles 6.3 and 7.0 us, 2600 8.7 and 8.3, 4120 11.6 and 9.8, 12288 23.8 and 16.9.
    const int per = m.heads / m.groups, each = (int64_t)(a.M + 15) / 16 * m.heads > 4096 ? 2 : 1;
    hipLaunchKernelGGL(ssm_tiles_kernel, dim3((a.M + 15) / 16, (per + 4 * each - 1) / (4 * each), m.groups), dim3(256), 0, s, a, each);
    const dim3 grid(m.heads, (m.vdim + 15) / 16);
    static std::once_flag raised;
    std::call_once(raised, [] {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&ssm_scan_kernel<8, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 128));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&ssm_scan_kernel<8, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 256));
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&ssm_scan_kernel<8, 4>), hipFuncAttributeMaxDynamicSharedMemorySize, scan_lds(8, 512));
    });
#define PTM_RUN(W, KT) hipLaunchKernelGGL((ssm_scan_kernel<W, KT>), grid, dim3(64 * W), scan_lds(W, a.keys), s, a)
    switch (a.keys) {
        case 64: PTM_RUN(4, 1); break;
        case 128: PTM_RUN(8, 1); break;
        case 256: PTM_RUN(8, 2); break;
        default: PTM_RUN(8, 4);
    }
#undef PTM_RUN
    if (fp32) hipLaunchKernelGGL(ssm_out_rows_kernel<true>, dim3(a.M), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(ssm_out_rows_kernel<false>, dim3(a.M), dim3(256), 0, s, a);
    return launch_status();
}
#undef PTM_KPL

}  // namespace ptm
