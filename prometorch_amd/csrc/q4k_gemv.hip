// Q4_K dequant-fused GEMV for gfx950 (wave64).
//
// Arithmetic follows the reference CPU kernel (torch/io/cpu_quant_gemv.h:505-685): the
// activation vector is quantised to Q8 blocks of 32 (cpu_quant_gemv.h:147-198), each 32-wide
// sub-block contributes  fma(d*sc*dx, (float)isum, -(dmin*m*sx))  with isum the exact int32
// dot of 4-bit weights and int8 activations; only the order in which the per-sub-block terms
// are added differs (per-lane chains + a cross-lane tree instead of two scalar chains).
//
// Data movement: a super-block (144 B) is fetched by an aligned group of 8 lanes: lane j takes
// the 16-byte header {d, dmin, scales[12]} and the j-th 16-byte slice of qs[128] with 128-bit
// loads, so every fetched byte is used.  A slice holds 16 low nibbles (sub-block 2*(j/2)) and
// 16 high nibbles (sub-block 2*(j/2)+1); lane pairs swap halves through one DPP move so that
// lane j ends up owning the complete integer dot of sub-block j.
// A row is shared by S lane groups (S = 1, 2, 4 or 8 - a whole wave), group s taking blocks
// s, s+S, ...; S is chosen on the host so that a launch has several hundred workgroups even for
// short-and-wide matrices (o-proj: 2560 rows) and so that each group's blocks are all in flight
// at once (five per group measured best: fewer registers, more waves per SIMD).  The first pass of
// weight loads is issued BEFORE the activation vector is staged (RMSNorm, Q8 quantisation, LDS), so HBM
// latency overlaps the prologue; every pass issues a fixed number of loads (template NB) and activations
// come through range-checked buffer loads, so no load sits under a branch and the compiler can wait for
// exactly the block it is about to use.  Very tall matrices let a workgroup walk several row tiles with
// one staging of x; where a tile is a single pass, the block loads roll across the tiles (q4k_gemv_tall_kernel: a consumed
// block's registers are refilled from the next tile's row, 151936 x 2560: 44.5 -> 41.6 us).
#include "q4k_body.h"

namespace ptm {

template <bool XQ8, bool NORM, bool ACC, int MODE, int NB>
__global__ __launch_bounds__(Q4K_THREADS) void q4k_gemv_kernel(const Q4KArgs a) {
    read_now(a.W[0], a.K, a.gamma);
    extern __shared__ __align__(16) uint8_t lds[];
    q4k_gemv_body<XQ8, NORM, ACC, MODE, NB>(a, lds, blockIdx.x);
}

// The same where a row's blocks are one pass of 1 << LS lane groups, in workgroups of up to ten waves (q4k_one).  What bounds a launch of 14 to 40
// MB is the order in which a CU's waves get their requests out: a wave that asks for all its blocks at once stands in the queue of the memory path for
// up to 5 us, x behind the weights of others, and only then starts to stage x.  Here x goes out first (wave priority 3), then EARLY blocks, then
// the staging (priority 2, in front of other waves' products), then the other blocks; 2.5 blocks of 20 waves, 40 KB a CU, keep HBM busy.  Weights
// from HBM, in a graph behind a launch that writes x, that launch (2.1 us) included: gate / up 9728 x 2560 12.0 -> 9.6 us, q / k / v 6144 x 2560 7.1 -> 6.3,
// o 2560 x 4096 5.7 -> 5.3.  More than two pieces of x a thread are no gain (q / k / v 6144 x 4096 8.2 -> 8.1, gate / up 11.2 either way) and stay with
// q4k_gemv_kernel.
template <bool XQ8, bool NORM, bool ACC, int MODE, int NB, int LS, int PIECES>
__global__ __launch_bounds__(64 * Q4K_ONE_WAVES) void q4k_gemv_one_kernel(const Q4KArgs a) {
    read_now(a.W[0], a.K, a.gamma);
    extern __shared__ __align__(16) uint8_t lds[];
    q4k_gemv_body<XQ8, NORM, ACC, MODE, NB, false, false, LS, PIECES, MODE == 1 ? 1 : (NB + 1) / 2>(a, lds, blockIdx.x);
}

// a workgroup walks several row tiles, every tile one pass of NB blocks per lane group: the passes roll across the tiles
template <bool XQ8, bool NORM, bool ACC, int MODE, int NB>
__global__ __launch_bounds__(Q4K_THREADS) void q4k_gemv_tall_kernel(const Q4KArgs a) {
    read_now(a.W[0], a.K, a.gamma);
    extern __shared__ __align__(16) uint8_t lds[];
    q4k_gemv_body<XQ8, NORM, ACC, MODE, NB, true>(a, lds, blockIdx.x);
}

// Few rows, long rows (a Q4_K down projection: 2560 x 9728, as in the layers of a Q4_K_M file whose ffn_down is Q4_K): with
// four rows per workgroup, 640 workgroups would each quantise the whole 9728-value activation vector for four rows' worth
// of weights.  Here a workgroup is blockDim.x / 64 waves of one row each (the row's super-blocks strided over the wave's 8 lane
// groups), sized so that the launch is one workgroup per CU (two for 17 to 32 rows per CU): x is quantised once per workgroup, up to eight
// 16-byte pieces per thread.  Of a group's blocks two are requested in front of the staging, three are in flight.  Block-to-lane assignment and
// reduction order are those of q4k_gemv_body with 8 lane groups per row, so the result is bit-identical to that kernel's.  Against passes
// of three blocks in a loop, weights from HBM, in a graph with two small launches in front (3.7 us, included): 2560 x 9728 10.6 -> 9.7 us, 4096 x
// 14336 13.8 -> 12.7, 3584 x 11008 12.0 -> 11.2; two workgroups of eight waves instead of one of 16, 4096 x 14336: 13.4.
template <bool ACC, int NB, int PIECES>
__global__ __launch_bounds__(1024) void q4k_gemv_rows_kernel(const Q4KArgs a) {
    read_now(a.W[0], a.K);
    extern __shared__ __align__(16) uint8_t lds[];
    q4k_gemv_body<false, false, ACC, 0, NB, false, false, 3, PIECES, NB < 2 ? NB : 2, NB < 3 ? NB : 3>(a, lds, blockIdx.x);
}

// The same for rows of more than ten blocks a lane group, x of more than eight pieces a thread and where it is faster (q4k_rows_in_order): passes of NB blocks, rolling as in q4k_gemv_body, x staged by half
// blocks (q4k_halves_issue says why), XL of them a thread.  In pieces 4096 x 25600 took 18.0 us, so 17.4, 2048 x 25600 18.1 and 15.0.
enum { Q4K_LONGROW_MAX_WAVES = 16 };
template <bool ACC, int NB, int XL>
__global__ __launch_bounds__(64 * Q4K_LONGROW_MAX_WAVES) void q4k_gemv_longrow_kernel(const uint8_t* __restrict__ W, int64_t stride,
                                                                                       const float* __restrict__ x, float* y, int N, int K) {
    extern __shared__ __align__(16) uint8_t lds[];
    const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6, j = lane & 7, sub = lane >> 3;
    const int nblk = K / 256;
    const int r = blockIdx.x * (nthr >> 6) + wave;
    const bool live = r < N;
    const uint8_t* row = W + (int64_t)(live ? r : N - 1) * stride;
    // activation loads first (range-checked: zeros past the end), then the weights, then the Q8 arithmetic
    const __amdgpu_buffer_rsrc_t rx = make_rsrc(x, K * 4);
    float4 xv[XL][4];
#pragma unroll
    for (int u = 0; u < XL; ++u) q4k_load16(rx, 16 * (tid + nthr * u), xv[u]);
    issue_order_fence();
    uint4 hdr[NB], qv[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const uint8_t* p = row + (int64_t)min(sub + 8 * u, nblk - 1) * 144;
        hdr[u] = *reinterpret_cast<const uint4*>(p);
        qv[u] = *reinterpret_cast<const uint4*>(p + 16 + 16 * j);
    }
    issue_order_fence();
#pragma unroll
    for (int u = 0; u < XL; ++u) {  // lanes t, t ^ 1 share a block: both inside or both outside (nthr is a multiple of 64)
        const int unit = tid + nthr * u;
        if (16 * unit < K) q4k_quantize16_store<false>(xv[u], xv[u], 1.0f, 0.0f, unit, lds, K);
    }
    __syncthreads();
    const Q4KLane ln = q4k_lane(lds, K, j);
    // passes roll as in q4k_gemv_body: a consumed block's registers are refilled from the next pass at once
    const int nb_max = (nblk + 7) >> 3;
    float acc = 0.0f;
    int i0 = 0;
    for (; i0 + NB < nb_max; i0 += NB) {
#pragma unroll
        for (int u = 0; u < NB; ++u) {
            const int b = sub + 8 * (i0 + u);
            const float t = q4k_block_term(hdr[u], qv[u], ln, min(b, nblk - 1));
            acc += b < nblk ? t : 0.0f;
            const uint8_t* p = row + (int64_t)min(sub + 8 * (i0 + NB + u), nblk - 1) * 144;
            hdr[u] = *reinterpret_cast<const uint4*>(p);
            qv[u] = *reinterpret_cast<const uint4*>(p + 16 + 16 * j);
        }
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
        const int b = sub + 8 * (i0 + u);
        const float t = q4k_block_term(hdr[u], qv[u], ln, min(b, nblk - 1));
        acc += b < nblk ? t : 0.0f;
    }
    float p = sum8(acc);
    p += dpp_f<0x128>(p);
    p = add16(p);
    p = add32(p);
    if (live && lane == 0) {
        if constexpr (ACC) y[r] += p;
        else y[r] = p;
    }
}

// waves per workgroup and half blocks of x per thread of that launch, or waves = 0 when the shape is not one for it.  Up to
// 16 rows per CU make one workgroup per CU, up to 32 two (each quantises x for itself).
struct Q4KLongrow { int waves, xl; };
static Q4KLongrow q4k_longrow_shape(int N, int K) {
    if (K < 4096) return {0, 0};                                  // long rows
    const int rows_per_cu = (N + 255) / 256;
    const int per_cu = (rows_per_cu + Q4K_LONGROW_MAX_WAVES - 1) / Q4K_LONGROW_MAX_WAVES;
    if (per_cu > 2) return {0, 0};
    const int waves = (rows_per_cu + per_cu - 1) / per_cu;
    if (waves < 2) return {0, 0};
    const int xl = (K / 16 + 64 * waves - 1) / (64 * waves);
    if (xl > 3) return {0, 0};
    return {waves, xl};
}

template <bool ACC, int PIECES>
static void (*q4k_rows_kernel(int nb))(const Q4KArgs) {
    switch (nb) {
        case 2: return q4k_gemv_rows_kernel<ACC, 2, PIECES>;
        case 3: return q4k_gemv_rows_kernel<ACC, 3, PIECES>;
        case 4: return q4k_gemv_rows_kernel<ACC, 4, PIECES>;
        case 5: return q4k_gemv_rows_kernel<ACC, 5, PIECES>;
        case 6: return q4k_gemv_rows_kernel<ACC, 6, PIECES>;
        case 7: return q4k_gemv_rows_kernel<ACC, 7, PIECES>;
        case 8: return q4k_gemv_rows_kernel<ACC, 8, PIECES>;
        case 9: return q4k_gemv_rows_kernel<ACC, 9, PIECES>;
        default: return q4k_gemv_rows_kernel<ACC, 10, PIECES>;
    }
}
// Whether x in pieces and blocks in an order (q4k_gemv_rows_kernel) is faster than the passes of the other, for rows of up to ten blocks a lane group.  us behind a launch
// that writes x, so and in passes: two and three waves are too few to share the staging, 512 x 4096 6.09, 5.20, 768 x 6144 6.21, 5.65.  Of two
// blocks a group (4096 values) nothing is left to request in order, and it is the staging of 12 waves and more that counts: 2816 x 4096 5.89, 6.07, 3584 6.51,
// 6.32, 4096 6.69, 6.28; two workgroups a CU, 5120 x 4096 7.44, 7.21, 6144 7.66, 7.27, but 7168 8.49, 8.74, 8192 8.41, 8.43.  Others 0.1 to 1.3 less so.
bool q4k_rows_in_order(int N, int K, int waves) {
    return waves >= 4 && (K > 4096 || (N <= 256 * Q4K_LONGROW_MAX_WAVES ? waves <= 11 : waves > 12));
}

template <bool ACC>
static int q4k_launch_longrow(const Q4KArgs& a, Q4KLongrow sh, hipStream_t s) {
    const dim3 grid((a.total_rows + sh.waves - 1) / sh.waves), block(64 * sh.waves);
    const size_t lds = (size_t)q8_bytes(a.K);
    const int nb = (a.K / 256 + 7) / 8, pieces = (a.K / 4 + 64 * sh.waves - 1) / (64 * sh.waves);
    if (q4k_rows_in_order(a.total_rows, a.K, sh.waves) && nb <= 10 && pieces <= 8 && a.stride < 1ll << 31) {
        const auto kernel = pieces <= 4 ? q4k_rows_kernel<ACC, 4>(nb) : q4k_rows_kernel<ACC, 8>(nb);
        hipLaunchKernelGGL(kernel, grid, block, lds, s, a);
        return launch_status();
    }
    const float* x = static_cast<const float*>(a.x);
#define PTM_LR(NB, XL) hipLaunchKernelGGL((q4k_gemv_longrow_kernel<ACC, NB, XL>), grid, block, lds, s, a.W[0], a.stride, x, a.y[0], a.total_rows, a.K)
    // blocks in flight per lane group: two; three for workgroups of up to ten waves (2560 x 9728, 10 waves, five blocks per
    // group: 1 / 2 / 3 / 5 in flight 7.5 / 7.0 / 6.9 / 7.0 us; 3584 x 18944, 14 waves: 1 / 2 / 3 in flight 12.8 / 11.3 / 12.2).  One half block
    // of x a thread is there for 4096 values only: of more, eight pieces are.
    if (nb > 2 && sh.waves <= 10) {
        if (sh.xl <= 2) PTM_LR(3, 2);
        else PTM_LR(3, 3);
    } else {
        if (sh.xl == 1) PTM_LR(2, 1);
        else if (sh.xl == 2) PTM_LR(2, 2);
        else PTM_LR(2, 3);
    }
#undef PTM_LR
    return launch_status();
}

// How a launch is laid out for q4k_gemv_one_kernel (waves 0: not at all): a row's blocks in one pass of up to five a lane group, the waves of a CU
// in workgroups of at most ten, which share the staging of x (one of 15 or 16 waves instead of two: 7376 x 1024 6.15 -> 6.45 us, 8192 x 2048 7.9 -> 8.3; of
// four instead of ten, 9728 x 2560: 9.45 -> 9.9), at most two 16-byte pieces of x a thread.
struct Q4KOne { int waves, nb, ls, pieces; };
template <bool XQ8, bool NORM, int MODE>
static Q4KOne q4k_one(const Q4KArgs& a) {
    const int nblk = a.K / 256;
    int ls = a.log2S;
    // q / k / v: six waves a CU with more blocks each are better than twelve (6144 x 2560: 6.5 -> 6.3 us), from 6144 rows of four lane groups and 3072 of eight on: with twice the
    // blocks and with the lane groups as they are 6144 x 2560 6.57, 7.03, 3072 x 2560 5.48, 5.93, but 5120 x 2560 6.33, 6.13, 2048 x 2560 5.81, 5.42 (5376 to
    // 5888 rows, which stay with the latter, 0.2 to 0.4 less with the former).
    if (NORM && MODE == 0 && ls > 1 && (nblk + (1 << (ls - 1)) - 1) >> (ls - 1) <= 5 && (int64_t)a.total_rows << (ls - 1) >= 12288) --ls;
    const int nb = (nblk + (1 << ls) - 1) >> ls;
    if (ls < 1 || nb > 5 || a.add_one || a.stride >= 1ll << 31) return {0, 0, 0, 0};
    const int rows_per_wave = 8 >> ls, total = (a.total_rows + rows_per_wave - 1) / rows_per_wave, per_cu = (total + 255) / 256;
    const int wgs = (per_cu + Q4K_ONE_WAVES - 1) / Q4K_ONE_WAVES;
    const int waves = per_cu < 4 ? 4 : (per_cu + wgs - 1) / wgs;
    const int pieces = ((XQ8 ? (a.K + a.K / 4) / 16 : a.K / 4) + 64 * waves - 1) / (64 * waves);
    return {pieces <= 2 ? waves : 0, nb, ls, pieces};
}
template <bool XQ8, bool NORM, bool ACC, int MODE, int LS, int PIECES>
static void (*q4k_one_kernel(int nb))(const Q4KArgs) {
    switch (nb) {
        case 1: return q4k_gemv_one_kernel<XQ8, NORM, ACC, MODE, 1, LS, PIECES>;
        case 2: return q4k_gemv_one_kernel<XQ8, NORM, ACC, MODE, 2, LS, PIECES>;
        case 3: return q4k_gemv_one_kernel<XQ8, NORM, ACC, MODE, 3, LS, PIECES>;
        case 4: return q4k_gemv_one_kernel<XQ8, NORM, ACC, MODE, 4, LS, PIECES>;
        default: return q4k_gemv_one_kernel<XQ8, NORM, ACC, MODE, 5, LS, PIECES>;
    }
}
template <bool XQ8, bool NORM, bool ACC, int MODE, int PIECES>
static void (*q4k_one_kernel(const Q4KOne& o))(const Q4KArgs) {
    if (o.ls == 1) return q4k_one_kernel<XQ8, NORM, ACC, MODE, 1, PIECES>(o.nb);
    if (MODE == 1 || o.ls == 2) return q4k_one_kernel<XQ8, NORM, ACC, MODE, 2, PIECES>(o.nb);
    return q4k_one_kernel<XQ8, NORM, ACC, MODE, MODE == 1 ? 2 : 3, PIECES>(o.nb);
}

template <bool XQ8, bool NORM, bool ACC, int MODE>
static int q4k_launch(Q4KArgs& a, hipStream_t s) {
    a.log2S = q4k_pick_log2S(a.total_rows, a.K / 256, MODE == 1 ? 2 : 3);
    const int n_tiles = q4k_workgroups(a.total_rows, a.log2S);
    a.tiles_per_wg = q4k_tiles_per_wg(n_tiles);
    const dim3 block(Q4K_THREADS);
    const size_t lds = (size_t)q8_bytes(a.K);
    const int nb = q4k_blocks_per_pass(a.K / 256, a.log2S);
    {
        // a very tall matrix (or gate / up pair) whose lane groups hold a row's blocks in a single pass: the loads roll
        // across the tiles
        const int nb_max = (a.K / 256 + (1 << a.log2S) - 1) >> a.log2S;
                // (only beyond 1280 tiles: the Qwen3-4B gate / up pair, 1216 tiles, as 608 workgroups of two rolling tiles measured
        // 9.88 us against 9.45 with one tile per workgroup)
        if ((MODE == 1 || a.n_mat == 1) && a.tiles_per_wg > 1 && nb_max <= nb && nb <= 5) {
            a.tiles_per_wg = q4k_tiles_per_wg_rolling(n_tiles);
            const dim3 grid((n_tiles + a.tiles_per_wg - 1) / a.tiles_per_wg);
            switch (nb) {
                case 2: hipLaunchKernelGGL((q4k_gemv_tall_kernel<XQ8, NORM, ACC, MODE, 2>), grid, block, lds, s, a); break;
                case 3: hipLaunchKernelGGL((q4k_gemv_tall_kernel<XQ8, NORM, ACC, MODE, 3>), grid, block, lds, s, a); break;
                case 4: hipLaunchKernelGGL((q4k_gemv_tall_kernel<XQ8, NORM, ACC, MODE, 4>), grid, block, lds, s, a); break;
                default: hipLaunchKernelGGL((q4k_gemv_tall_kernel<XQ8, NORM, ACC, MODE, 5>), grid, block, lds, s, a); break;
            }
            return launch_status();
        }
    }
    if constexpr ((NORM && !ACC) || (XQ8 && MODE == 0)) {  // the launches of a decode step
        const Q4KOne o = a.tiles_per_wg == 1 ? q4k_one<XQ8, NORM, MODE>(a) : Q4KOne{};
        if (o.waves > 0) {
            a.log2S = o.ls;
            const int rows = o.waves * (8 >> o.ls);
            const auto kernel = XQ8 || o.pieces == 2 ? q4k_one_kernel<XQ8, NORM, ACC, MODE, 2>(o) : q4k_one_kernel<XQ8, NORM, ACC, MODE, XQ8 ? 2 : 1>(o);
            hipLaunchKernelGGL(kernel, dim3((a.total_rows + rows - 1) / rows), dim3(64 * o.waves), lds, s, a);
            return launch_status();
        }
    }
    const dim3 grid((n_tiles + a.tiles_per_wg - 1) / a.tiles_per_wg);
    switch (nb) {
        case 2: hipLaunchKernelGGL((q4k_gemv_kernel<XQ8, NORM, ACC, MODE, 2>), grid, block, lds, s, a); break;
        case 3: hipLaunchKernelGGL((q4k_gemv_kernel<XQ8, NORM, ACC, MODE, 3>), grid, block, lds, s, a); break;
        case 4: hipLaunchKernelGGL((q4k_gemv_kernel<XQ8, NORM, ACC, MODE, 4>), grid, block, lds, s, a); break;
        case 5: hipLaunchKernelGGL((q4k_gemv_kernel<XQ8, NORM, ACC, MODE, 5>), grid, block, lds, s, a); break;
        default: hipLaunchKernelGGL((q4k_gemv_kernel<XQ8, NORM, ACC, MODE, 10>), grid, block, lds, s, a); break;
    }
    return launch_status();
}

static int q4k_check(const void* W, const void* x, const void* y, int K, int N, int64_t stride) {
    if (!W || !x || !y) return PTM_E_NULL;
    if (K <= 0 || N <= 0 || (K % 256) != 0) return PTM_E_SHAPE;
    if (K > 32768) return PTM_E_UNSUPPORTED;  // Q8 activations must fit the 40 KB LDS budget used here
    if (stride < (int64_t)(K / 256) * 144) return PTM_E_SHAPE;
    if ((stride & 15) != 0 || !aligned16(W) || !aligned16(x) || (reinterpret_cast<uintptr_t>(y) & 3u)) return PTM_E_ALIGN;
    return PTM_OK;
}

// Shared by the C entry points and the decode runtime.
int q4k_gemv_multi(int n_mat, const void* const* W, float* const* y, const int* N, const void* x, bool x_is_q8,
                   const float* gamma, float eps, int add_one, int K, int64_t stride, bool accumulate,
                   hipStream_t s) {
    Q4KArgs a{};
    int total = 0;
    for (int i = 0; i < n_mat; ++i) {
        const int rc = q4k_check(W[i], x, y[i], K, N[i], stride);
        if (rc != PTM_OK) return rc;
        a.W[i] = static_cast<const uint8_t*>(W[i]);
        a.y[i] = y[i];
        total += N[i];
        a.row_end[i] = total;
    }
    a.n_mat = n_mat;
    a.total_rows = total;
    a.K = K;
    a.stride = stride;
    a.x = x;
    a.gamma = gamma;
    a.eps = eps;
    a.add_one = add_one;
    if (gamma) {
        if (x_is_q8) return PTM_E_UNSUPPORTED;
        if (!aligned16(gamma)) return PTM_E_ALIGN;
        return accumulate ? q4k_launch<false, true, true, 0>(a, s) : q4k_launch<false, true, false, 0>(a, s);
    }
    if (x_is_q8) return accumulate ? q4k_launch<true, false, true, 0>(a, s) : q4k_launch<true, false, false, 0>(a, s);
    if (n_mat == 1) {
        const Q4KLongrow sh = q4k_longrow_shape(N[0], K);
        if (sh.waves > 0) return accumulate ? q4k_launch_longrow<true>(a, sh, s) : q4k_launch_longrow<false>(a, sh, s);
    }
    return accumulate ? q4k_launch<false, false, true, 0>(a, s) : q4k_launch<false, false, false, 0>(a, s);
}

int q4k_gate_up_silu(const void* wg, const void* wu, const void* x, bool x_is_q8, const float* gamma, float eps,
                     int add_one, float* act, int K, int N, int64_t stride, hipStream_t s, bool gelu) {
    int rc = q4k_check(wg, x, act, K, N, stride);
    if (rc != PTM_OK) return rc;
    rc = q4k_check(wu, x, act, K, N, stride);
    if (rc != PTM_OK) return rc;
    if (N > 0x3fffffff) return PTM_E_UNSUPPORTED;
    Q4KArgs a{};
    a.W[0] = static_cast<const uint8_t*>(wg);
    a.W[1] = static_cast<const uint8_t*>(wu);
    a.y[0] = act;
    a.n_mat = 2;
    a.row_end[0] = N;
    a.total_rows = 2 * N;
    a.K = K;
    a.stride = stride;
    a.x = x;
    a.gamma = gamma;
    a.eps = eps;
    a.add_one = add_one;
    a.gelu = gelu ? 1 : 0;
    if (gamma) {
        if (x_is_q8) return PTM_E_UNSUPPORTED;
        if (!aligned16(gamma)) return PTM_E_ALIGN;
        return q4k_launch<false, true, false, 1>(a, s);
    }
    return x_is_q8 ? q4k_launch<true, false, false, 1>(a, s) : q4k_launch<false, false, false, 1>(a, s);
}

}  // namespace ptm

using namespace ptm;

extern "C" {

int ptm_q4k_gemv(const void* W, const float* x, float* y, int K, int N, int64_t stride, int accumulate,
                 ptm_stream_t stream) {
    return q4k_gemv_multi(1, &W, &y, &N, x, false, nullptr, 0.f, 0, K, stride, accumulate != 0, as_stream(stream));
}

int ptm_q4k_gemv_q8(const void* W, const void* x_q8, float* y, int K, int N, int64_t stride, int accumulate,
                    ptm_stream_t stream) {
    return q4k_gemv_multi(1, &W, &y, &N, x_q8, true, nullptr, 0.f, 0, K, stride, accumulate != 0, as_stream(stream));
}

int ptm_q4k_fused_gate_up_gemv(const void* w_gate, const void* w_up, const float* x, float* y_gate, float* y_up,
                               int K, int N_gate, int N_up, int64_t stride, ptm_stream_t stream) {
    const void* W[2] = {w_gate, w_up};
    float* y[2] = {y_gate, y_up};
    const int N[2] = {N_gate, N_up};
    return q4k_gemv_multi(2, W, y, N, x, false, nullptr, 0.f, 0, K, stride, false, as_stream(stream));
}

int ptm_q4k_fused_qkv_gemv(const void* w_q, const void* w_k, const void* w_v, const float* x, float* out_q,
                           float* out_k, float* out_v, int K, int N_q, int N_k, int N_v, int64_t stride,
                           ptm_stream_t stream) {
    const void* W[3] = {w_q, w_k, w_v};
    float* y[3] = {out_q, out_k, out_v};
    const int N[3] = {N_q, N_k, N_v};
    return q4k_gemv_multi(3, W, y, N, x, false, nullptr, 0.f, 0, K, stride, false, as_stream(stream));
}

int ptm_q4k_fused_rmsnorm_gemv(const float* x, const float* norm_w, const void* W, float* y, int K, int N,
                               int64_t stride, float eps, int add_one, ptm_stream_t stream) {
    if (!norm_w) return PTM_E_NULL;
    return q4k_gemv_multi(1, &W, &y, &N, x, false, norm_w, eps, add_one, K, stride, false, as_stream(stream));
}

int ptm_q4k_fused_rmsnorm_qkv_gemv(const float* x, const float* norm_w, const void* w_q, const void* w_k,
                                   const void* w_v, float* out_q, float* out_k, float* out_v, int K, int N_q,
                                   int N_k, int N_v, int64_t stride, float eps, int add_one,
                                   ptm_stream_t stream) {
    if (!norm_w) return PTM_E_NULL;
    const void* W[3] = {w_q, w_k, w_v};
    float* y[3] = {out_q, out_k, out_v};
    const int N[3] = {N_q, N_k, N_v};
    return q4k_gemv_multi(3, W, y, N, x, false, norm_w, eps, add_one, K, stride, false, as_stream(stream));
}

int ptm_q4k_fused_rmsnorm_gate_up_gemv(const float* x, const float* norm_w, const void* w_gate,
                                       const void* w_up, float* y_gate, float* y_up, int K, int N_gate,
                                       int N_up, int64_t stride, float eps, int add_one, ptm_stream_t stream) {
    if (!norm_w) return PTM_E_NULL;
    const void* W[2] = {w_gate, w_up};
    float* y[2] = {y_gate, y_up};
    const int N[2] = {N_gate, N_up};
    return q4k_gemv_multi(2, W, y, N, x, false, norm_w, eps, add_one, K, stride, false, as_stream(stream));
}

int ptm_q4k_fused_rmsnorm_gate_up_silu(const float* x, const float* norm_w, const void* w_gate,
                                       const void* w_up, float* act, int K, int N, int64_t stride, float eps,
                                       int add_one, ptm_stream_t stream) {
    if (!norm_w) return PTM_E_NULL;
    return q4k_gate_up_silu(w_gate, w_up, x, false, norm_w, eps, add_one, act, K, N, stride, as_stream(stream), false);
}

}  // extern "C"
