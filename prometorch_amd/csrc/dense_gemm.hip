// Prompt products over bfloat16 weights: C[M][N] = A[M][K] . W[N][K]^T on the matrix cores.
//
// dense_gemm_tiles_kernel (more than 64 bfloat16 rows): the tiles of gemm_tile.h, as plan_tiles lays them out.
// dense_gemm_few_kernel (up to 64 bfloat16 rows, outputs of up to 1280 tiles of 32 x 32).
// dense_gemm_kernel (up to 64 bfloat16 rows and more columns, outputs of few tiles, rows far apart): 4 waves, BM x BN output tile, 64 values of K per step.  Tiles go global -> registers ->
// LDS; two register sets and two LDS buffers, so a step has one barrier and the loads of the next two steps are in flight
// while its MFMAs run.
// LDS rows are 128 bytes, the eight 16-byte pieces of row r stored at piece ^ (r % 8): the fragment reads (32 rows, one
// piece) and the writes touch every bank evenly.  The product is formed transposed (W rows as the A operand), so that a lane
// holds four consecutive columns of one output row.
// dense_gemm_f32_kernel (fp32 rows): the same product in fp32 on v_mfma_f32_32x32x2_f32, 64 x 64 tiles.
#include "dense.h"
#include "gemm_tile.h"

#include <algorithm>
#include <mutex>

namespace ptm {

typedef __bf16 gm_b8 __attribute__((ext_vector_type(8)));
typedef float gm_f16 __attribute__((ext_vector_type(16)));

// workgroups are dealt to the 8 XCDs in turn: give each XCD a contiguous run of tiles (rows fastest, so a run shares columns of W)
__device__ __forceinline__ void tile_of(int wg, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n, per = total / 8, rem = total % 8, xcd = wg % 8, i = wg / 8;
    const int id = xcd * per + min(xcd, rem) + i;
    tm = id % tiles_m;
    tn = id / tiles_m;
}

// the same for the larger tiles: runs of bands of four row tiles, so that the 32 tiles an XCD works on are about as high as wide
__device__ __forceinline__ void band_tile_of(int wg, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int total = tiles_m * tiles_n, per = total / 8, rem = total % 8, xcd = wg % 8, i = wg / 8;
    const int id = xcd * per + min(xcd, rem) + i;
    const int band = id / (4 * tiles_n), r = id - band * 4 * tiles_n, rows = min(4, tiles_m - 4 * band);
    tm = 4 * band + r % rows;
    tn = r / rows;
}

__device__ __forceinline__ float relu2(float v) { return v > 0.0f ? v * v : 0.0f; }

// row of W behind column n of the product.  GEMM_SWIGLU: each 32 columns are 16 gate rows and the 16 up rows of the same values,
// which one lane's accumulators hold together.
__device__ __forceinline__ int weight_row(const DenseGemm& g, int n) {
    if (g.epilogue != GEMM_SWIGLU) return min(n, g.N - 1);
    const int ff = g.N / 2, v = min((n >> 5) * 16 + (n & 15), ff - 1);
    return (n & 16) ? ff + v : v;
}

// four consecutive columns n .. n + 3 of row m
template <bool F32>
__device__ __forceinline__ void store4(const DenseGemm& g, int split, int m, int n, float v0, float v1, float v2, float v3) {
    if (g.epilogue == GEMM_RELU2) {
        v0 = relu2(v0);
        v1 = relu2(v1);
        v2 = relu2(v2);
        v3 = relu2(v3);
    }
    if (g.epilogue == GEMM_DECAY) {
        auto decay = [&](float v, int k) { return k < g.N ? expf(-expf(v + g.bias[k])) : 0.0f; };
        v0 = decay(v0, n);
        v1 = decay(v1, n + 1);
        v2 = decay(v2, n + 2);
        v3 = decay(v3, n + 3);
    }
    const int64_t at = (int64_t)m * g.ldc + n + split * g.slab;
    if (F32 || g.epilogue == GEMM_F32 || g.epilogue == GEMM_DECAY) {
        float* c = static_cast<float*>(g.C) + at;
        if (n + 3 < g.N && (g.ldc & 3) == 0) {
            *reinterpret_cast<float4*>(c) = make_float4(v0, v1, v2, v3);
        } else {
            c[0] = v0;
            if (n + 1 < g.N) c[1] = v1;
            if (n + 2 < g.N) c[2] = v2;
            if (n + 3 < g.N) c[3] = v3;
        }
    } else {
        uint16_t* c = static_cast<uint16_t*>(g.C) + at;
        if (n + 3 < g.N && (g.ldc & 3) == 0) {
            *reinterpret_cast<uint2*>(c) = make_uint2((uint32_t)f_bf16(v0) | ((uint32_t)f_bf16(v1) << 16), (uint32_t)f_bf16(v2) | ((uint32_t)f_bf16(v3) << 16));
        } else {
            c[0] = f_bf16(v0);
            if (n + 1 < g.N) c[1] = f_bf16(v1);
            if (n + 2 < g.N) c[2] = f_bf16(v2);
            if (n + 3 < g.N) c[3] = f_bf16(v3);
        }
    }
}

// 32 columns of GEMM_SWIGLU: accumulators 0..7 are gates, 8..15 the ups of the same values
template <bool F32>
__device__ __forceinline__ void store_glu(const DenseGemm& g, int m, int n, int kh, const gm_f16& acc) {
    DenseGemm o = g;
    o.epilogue = GEMM_ELEM;
    o.N = g.N / 2;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int v = n / 2 + 8 * q + 4 * kh;
        if (v < o.N)
            store4<F32>(o, 0, m, v, silu_f(acc[4 * q]) * acc[8 + 4 * q], silu_f(acc[4 * q + 1]) * acc[9 + 4 * q],
                        silu_f(acc[4 * q + 2]) * acc[10 + 4 * q], silu_f(acc[4 * q + 3]) * acc[11 + 4 * q]);
    }
}

// Few rows: a workgroup has 32 rows and 32 columns, its four waves take steps of K in turn, and their sums meet at the end.  A wave's steps come to LDS
// of its own, two of them in flight, W and X alike in whole 128-byte rows, and nothing but the end has a barrier.
// What bounds it: how much of W is on its way, 4 KB a step, which is why a workgroup has few columns (64: 30 x 2560 x 2560 13.5 us where this takes
// 9.6, 30 x 10240 x 2560 15.7 and 17.5; 64 rows at a time: 48 x 2560 x 2560 11.8 and 8.6).  Weights from HBM, in a graph, against the tiles of
// dense_gemm_kernel: 30 x 10240 x 2560 24.3 -> 17.5 us, 30 x 19456 x 2560 30.8 -> 26.7, 30 x 2560 x 9728 70.7 -> 25.3, 19 x 5632 x 2560 23.0 -> 9.7,
// 64 x 2560 x 9728 68.3 -> 25.0.
constexpr int FEW_WAVES = 4, FEW_STEPS = 2;
__global__ __launch_bounds__(64 * FEW_WAVES, 2) void dense_gemm_few_kernel(const DenseGemm g) {
    constexpr int STEP = 8192, PIECES = 8;  // 32 rows of W, 32 of X, and a wave's instructions for them
    __shared__ __align__(16) uint8_t s_t[FEW_WAVES * FEW_STEPS * STEP];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), j = lane & 31, kh = lane >> 5;
    const int tiles_n = (g.tile_cols + 31) / 32, tiles_m = (g.M + 31) / 32, split = blockIdx.x / (tiles_m * tiles_n);
    int tm, tn;
    tile_of(blockIdx.x - split * tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    const int m0 = 32 * tm, n0 = 32 * tn, all = (g.K + 63) / 64, first = all * split / g.splits + wave, end = all * (split + 1) / g.splits;
    const uint16_t* A = static_cast<const uint16_t*>(g.A);
    if (g.section_n > 0) A += n0 / g.section_n * g.section_a;
    gt_i4 ws = gt_buffer(g.W), xs = gt_buffer(A);
    xs[0] = __builtin_amdgcn_readfirstlane(xs[0]);
    xs[1] = __builtin_amdgcn_readfirstlane(xs[1]);
    const int piece = ((lane & 7) ^ (lane >> 3)) << 4;  // piece p of row r lies at p ^ (r % 8)
    int wo[4], xo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3);
        wo[i] = weight_row(g, n0 + r) * (int)g.ldw * 2 + piece;
        xo[i] = min(m0 + r, g.M - 1) * (int)g.lda * 2 + piece;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)s_t + wave * (FEW_STEPS * STEP);
    auto fetch = [&](int slot, int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) gt_to_lds(lds0 + slot * STEP + i * 1024, wo[i], ws, st * 128);
#pragma unroll
        for (int i = 0; i < 4; ++i) gt_to_lds(lds0 + slot * STEP + 4096 + i * 1024, xo[i], xs, st * 128);
    };
    gm_f16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    auto step = [&](int slot, int st) {  // used, and its place given to the step FEW_STEPS on
        if (st + FEW_WAVES < end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PIECES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const uint8_t* t = s_t + (wave * FEW_STEPS + slot) * STEP + j * 128;
        gm_b8 w[4], x[4];
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int at = ((2 * ks + kh) ^ (j & 7)) << 4;
            w[ks] = *reinterpret_cast<const gm_b8*>(t + at);
            x[ks] = *reinterpret_cast<const gm_b8*>(t + 4096 + at);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (st + FEW_STEPS * FEW_WAVES < end) fetch(slot, st + FEW_STEPS * FEW_WAVES);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[ks], x[ks], acc, 0, 0, 0);
    };
    if (first < end) fetch(0, first);
    if (first + FEW_WAVES < end) fetch(1, first + FEW_WAVES);
    for (int st = first; st < end; st += 2 * FEW_WAVES) {
        step(0, st);
        if (st + FEW_WAVES < end) step(1, st + FEW_WAVES);
    }
    __syncthreads();
    float4* sums = reinterpret_cast<float4*>(s_t);  // [wave][four columns][lane]
#pragma unroll
    for (int q = 0; q < 4; ++q) sums[(4 * wave + q) * 64 + lane] = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    __syncthreads();
    auto sum = [&](int q) {
        float4 v = sums[q * 64 + lane];
#pragma unroll
        for (int w = 1; w < FEW_WAVES; ++w) {
            const float4 o = sums[(4 * w + q) * 64 + lane];
            v = make_float4(v.x + o.x, v.y + o.y, v.z + o.z, v.w + o.w);
        }
        return v;
    };
    const int m = m0 + j;
    const bool glu = g.epilogue == GEMM_SWIGLU;
    if (m >= g.M || (glu && wave >= 2)) return;
    const float4 v = sum(wave);
    if (glu) {  // columns 0 .. 15 of the 32 are gates
        const float4 u = sum(wave + 2);
        DenseGemm o = g;
        o.epilogue = GEMM_ELEM;
        o.N = g.N / 2;
        const int n = n0 / 2 + 8 * wave + 4 * kh;
        if (n < o.N) store4<false>(o, 0, m, n, silu_f(v.x) * u.x, silu_f(v.y) * u.y, silu_f(v.z) * u.z, silu_f(v.w) * u.w);
    } else {
        const int n = n0 + 8 * wave + 4 * kh;
        if (n < g.N) store4<false>(g, split, m, n, v.x, v.y, v.z, v.w);
    }
}

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256, 2) void dense_gemm_kernel(const DenseGemm g) {
    static_assert((BM / WM) * (BN / WN) == 4, "four waves");
    constexpr int TM = WM / 32, TN = WN / 32, PA = BM / 32, PB = BN / 32;  // pieces of 16 bytes a thread stages
    __shared__ __align__(16) uint8_t s_a[2][BM * 128];
    __shared__ __align__(16) uint8_t s_b[2][BN * 128];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, kh = lane >> 5;
    int tm, tn;
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.tile_cols + BN - 1) / BN, split = blockIdx.x / (tiles_m * tiles_n);
    tile_of(blockIdx.x - split * tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;
    const int all = (g.K + 63) / 64, steps = all * (split + 1) / g.splits, first = all * split / g.splits;
    const uint16_t* A = static_cast<const uint16_t*>(g.A);
    if (g.section_n > 0) A += n0 / g.section_n * g.section_a;
    const int pr = tid >> 3, pp = tid & 7;  // row and piece of this thread's first staged piece; the others 32 rows on
    const u32x4* pa[PA];
    const u32x4* pb[PB];
    uint32_t la[PA], lb[PB];
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        const int r = pr + 32 * i;
        pa[i] = reinterpret_cast<const u32x4*>(A + (int64_t)min(m0 + r, g.M - 1) * g.lda) + pp;
        la[i] = r * 128 + ((pp ^ (r & 7)) << 4);
    }
#pragma unroll
    for (int i = 0; i < PB; ++i) {
        const int r = pr + 32 * i;
        pb[i] = reinterpret_cast<const u32x4*>(g.W + (int64_t)weight_row(g, n0 + r) * g.ldw) + pp;
        lb[i] = r * 128 + ((pp ^ (r & 7)) << 4);
    }
    u32x4 ra0[PA], rb0[PB], ra1[PA], rb1[PB];
    auto fetch = [&](int st, u32x4 (&ra)[PA], u32x4 (&rb)[PB]) {
        st = st < steps ? st : steps - 1;
#pragma unroll
        for (int i = 0; i < PA; ++i) ra[i] = pa[i][st * 8];
#pragma unroll
        for (int i = 0; i < PB; ++i) rb[i] = pb[i][st * 8];
    };
    auto stage = [&](int buf, const u32x4 (&ra)[PA], const u32x4 (&rb)[PB]) {
#pragma unroll
        for (int i = 0; i < PA; ++i) *reinterpret_cast<u32x4*>(&s_a[buf][la[i]]) = ra[i];
#pragma unroll
        for (int i = 0; i < PB; ++i) *reinterpret_cast<u32x4*>(&s_b[buf][lb[i]]) = rb[i];
    };
    gm_f16 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;
    auto multiply = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int pc = ((2 * ks + kh) ^ (j & 7)) << 4;
            gm_b8 fa[TM], fb[TN];
#pragma unroll
            for (int a = 0; a < TM; ++a) fa[a] = *reinterpret_cast<const gm_b8*>(&s_a[buf][(wm + 32 * a + j) * 128 + pc]);
#pragma unroll
            for (int b = 0; b < TN; ++b) fb[b] = *reinterpret_cast<const gm_b8*>(&s_b[buf][(wn + 32 * b + j) * 128 + pc]);
#pragma unroll
            for (int a = 0; a < TM; ++a)
#pragma unroll
                for (int b = 0; b < TN; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[b], fa[a], acc[a][b], 0, 0, 0);
        }
    };
    fetch(first, ra0, rb0);
    fetch(first + 1, ra1, rb1);
    stage(0, ra0, rb0);
    __syncthreads();
    // two steps per trip; a step past the end repeats the last one's loads and is not multiplied
    for (int st = first; st < steps; st += 2) {
        fetch(st + 2, ra0, rb0);
        multiply(0);
        stage(1, ra1, rb1);
        __syncthreads();
        fetch(st + 3, ra1, rb1);
        if (st + 1 < steps) multiply(1);
        stage(0, ra0, rb0);
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        const int m = m0 + wm + 32 * a + j;
        if (m >= g.M) continue;
#pragma unroll
        for (int b = 0; b < TN; ++b) {
            if (g.epilogue == GEMM_SWIGLU) {
                store_glu<false>(g, m, n0 + wn + 32 * b, kh, acc[a][b]);
                continue;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int n = n0 + wn + 32 * b + 8 * q + 4 * kh;
                if (n < g.N) store4<false>(g, split, m, n, acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]);
            }
        }
    }
}

// The same product on the tiles of gemm_tile.h, which take rows of both sides from memory to LDS directly.  A launch covers its output
// with up to four regions of equal tiles.
typedef GemmTile<8, 4, 2, 2, 2> Tile0;
typedef GemmTile<4, 6, 4, 2, 2> Tile1;
typedef GemmTile<4, 4, 2, 2, 3> Tile2;
typedef GemmTile<2, 6, 4, 3, 3> Tile3;
typedef GemmTile<2, 4, 4, 3, 3> Tile4;
typedef GemmTile<2, 4, 2, 3, 3> Tile5;
typedef GemmTile<2, 2, 2, 3, 3> Tile6;

template <typename Tile>
__device__ __forceinline__ void dense_tile(const DenseGemm& g, const GemmRegion& r, int wg, uint8_t* lds) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int split = wg / (r.tiles_m * r.tiles_n);
    int tm, tn;
    band_tile_of(wg - split * r.tiles_m * r.tiles_n, r.tiles_m, r.tiles_n, tm, tn);
    const int m0 = r.m0 + tm * Tile::BM, n0 = r.n0 + tn * Tile::BN;
    const int all = (g.K + 63) / 64, first = all * split / g.splits, steps = all * (split + 1) / g.splits - first;
    const uint16_t* A = static_cast<const uint16_t*>(g.A) + (int64_t)m0 * g.lda + first * 64;
    if (g.section_n > 0) A += n0 / g.section_n * g.section_a;
    // two-byte results: a lane's two sums next to each other make one 16-byte store (1030 x 9728 x 2560 63.0 -> 57.7 us); fp32 sums of
    // one fragment are 16 bytes already, and the four lanes of a row then store 64 in a row
    const bool glu = g.epilogue == GEMM_SWIGLU, pairs = g.epilogue == GEMM_ELEM || g.epilogue == GEMM_RELU2;
    // Offsets count from the tile's first row, which no other of its rows lies in front of (GEMM_SWIGLU: tiles start with whole blocks of 32
    // columns), and where the ups, half of W further on, are more than 2 GiB away from the wave's first row: an instruction's 8 rows are
    // gates in the waves without bit 1 and ups in those with it.  (So everywhere, 2048 x 19456 x 2560 takes 185 us instead of 176.)
    const bool far = glu && (int64_t)g.N * g.ldw >= 0x7fffffff;
    const int w0 = weight_row(g, n0 + (far ? (wave & 2) << 3 : 0));
    const gt_i4 xs = gt_buffer(A), ws = gt_buffer(g.W + (int64_t)w0 * g.ldw + first * 64);
    const uint32_t piece = ((lane & 7) ^ (lane >> 3)) << 4;
    uint32_t xo[Tile::NX], wo[Tile::NW];
#pragma unroll
    for (int i = 0; i < Tile::NX; ++i) xo[i] = (uint32_t)min(8 * (wave + 8 * i) + (lane >> 3), g.M - 1 - m0) * (uint32_t)g.lda * 2 + piece;
#pragma unroll
    for (int i = 0; i < Tile::NW; ++i) wo[i] = (uint32_t)(weight_row(g, n0 + (pairs ? gt_column(8 * (wave + 8 * i) + (lane >> 3)) : 8 * (wave + 8 * i) + (lane >> 3))) - w0) * (uint32_t)g.ldw * 2 + piece;
    const uint32_t base = (uint32_t)(uintptr_t)lds + wave * 1024;
    Tile t;
    t.run(lds, steps, [&](int st, int i, int at) { gt_to_lds(base + at + i * 8192, (int)xo[i], xs, st * 128); },
          [&](int st, int i, int at) { gt_to_lds(base + at + i * 8192, (int)wo[i], ws, st * 128); });
    const int m1 = min(g.M, r.m0 + r.tiles_m * Tile::BM), n1 = min(g.N, r.n1);
    // Tiles that end within the columns (and rows that hold whole vectors): one place per lane, a test per row.  With its own place, its tests and its kind of
    // result decided for every store, the end of a 256 x 256 tile took 64 instructions per eight values.
    const int row0 = Tile::lane_row(), col0 = Tile::lane_col(), g4 = (lane >> 4) * 4;
    auto rows = [&](auto&& store) {
#pragma unroll
        for (int a = 0; a < Tile::ROWS; ++a)
            if (m0 + row0 + 16 * a < m1)
#pragma unroll
                for (int b = 0; b < Tile::COLS; b += 2) store(a, b, (int64_t)(16 * a) * g.ldc, t.acc[a][b], t.acc[a][b + 1]);
    };
    if (n0 + Tile::BN <= n1 && (!glu || (g.ldc & 3) == 0)) {
        const int64_t first = (int64_t)(m0 + row0) * g.ldc;
        auto pack = [](float lo, float hi) { return (uint32_t)f_bf16(lo) | ((uint32_t)f_bf16(hi) << 16); };
        if (glu) {
            uint16_t* p = static_cast<uint16_t*>(g.C) + first + (n0 + col0 - g4) / 2 + g4;
            rows([&](int, int b, int64_t at, const gt_f4& x, const gt_f4& u) {
                *reinterpret_cast<uint2*>(p + at + 8 * b) = make_uint2(pack(silu_f(x[0]) * u[0], silu_f(x[1]) * u[1]), pack(silu_f(x[2]) * u[2], silu_f(x[3]) * u[3]));
            });
            return;
        }
        if (pairs && (g.ldc & 7) == 0) {
            uint16_t* p = static_cast<uint16_t*>(g.C) + first + n0 + col0 + g4;
            auto put = [&](int b, int64_t at, const gt_f4& x, const gt_f4& y) {
                *reinterpret_cast<uint4*>(p + at + 16 * b) = make_uint4(pack(x[0], x[1]), pack(x[2], x[3]), pack(y[0], y[1]), pack(y[2], y[3]));
            };
            if (g.epilogue == GEMM_RELU2)
                rows([&](int, int b, int64_t at, const gt_f4& x, const gt_f4& y) {
                    put(b, at, gt_f4{relu2(x[0]), relu2(x[1]), relu2(x[2]), relu2(x[3])}, gt_f4{relu2(y[0]), relu2(y[1]), relu2(y[2]), relu2(y[3])});
                });
            else
                rows([&](int, int b, int64_t at, const gt_f4& x, const gt_f4& y) { put(b, at, x, y); });
            return;
        }
        if (g.epilogue == GEMM_F32 && (g.ldc & 3) == 0) {
            float* p = static_cast<float*>(g.C) + first + n0 + col0 + split * g.slab;
            rows([&](int, int b, int64_t at, const gt_f4& x, const gt_f4& y) {
                *reinterpret_cast<gt_f4*>(p + at + 16 * b) = x;
                *reinterpret_cast<gt_f4*>(p + at + 16 * b + 16) = y;
            });
            return;
        }
    }
    if (glu) {  // even W fragments are gates, the odd ones behind them the ups of the same values
        DenseGemm o = g;
        o.epilogue = GEMM_ELEM;
        o.N = g.N / 2;
        t.each([&](int a, int b, int row, int c) {
            const int m = m0 + row, n = n0 + c - 4 * (lane >> 4), v = n / 2 + 4 * (lane >> 4);
            if (m >= m1 || n >= r.n1 || v >= o.N) return;
            const gt_f4 x = t.acc[a][b], u = t.acc[a][b + 1];
            store4<false>(o, 0, m, v, silu_f(x[0]) * u[0], silu_f(x[1]) * u[1], silu_f(x[2]) * u[2], silu_f(x[3]) * u[3]);
        });
        return;
    }
    t.each([&](int a, int b, int row, int c) {
        const int m = m0 + row, n = n0 + (pairs ? gt_column(c) : c), next = pairs ? 4 : 16;
        if (m >= m1) return;
        const gt_f4 x = t.acc[a][b], y = t.acc[a][b + 1];
        if (pairs && n + 7 < g.N && (g.ldc & 7) == 0) {
            if (n >= n1) return;
            auto two = [&](float lo, float hi) {
                if (g.epilogue == GEMM_RELU2) lo = relu2(lo), hi = relu2(hi);
                return (uint32_t)f_bf16(lo) | ((uint32_t)f_bf16(hi) << 16);
            };
            *reinterpret_cast<uint4*>(static_cast<uint16_t*>(g.C) + (int64_t)m * g.ldc + n) = make_uint4(two(x[0], x[1]), two(x[2], x[3]), two(y[0], y[1]), two(y[2], y[3]));
            return;
        }
        if (n < n1) store4<false>(g, split, m, n, x[0], x[1], x[2], x[3]);
        if (n + next < n1) store4<false>(g, split, m, n + next, y[0], y[1], y[2], y[3]);
    });
}

__global__ __launch_bounds__(512, 2) void dense_gemm_tiles_kernel(const DenseGemm g, const GemmRegions rs) {
    extern __shared__ __align__(1024) uint8_t gt_lds[];
    int i = 0;
    while (i + 1 < rs.n && (int)blockIdx.x >= rs.r[i + 1].first) ++i;
    const GemmRegion r = rs.r[i];
    const int wg = blockIdx.x - r.first;
    switch (r.kind) {
        case 0: return dense_tile<Tile0>(g, r, wg, gt_lds);
        case 1: return dense_tile<Tile1>(g, r, wg, gt_lds);
        case 2: return dense_tile<Tile2>(g, r, wg, gt_lds);
        case 3: return dense_tile<Tile3>(g, r, wg, gt_lds);
        case 4: return dense_tile<Tile4>(g, r, wg, gt_lds);
        case 5: return dense_tile<Tile5>(g, r, wg, gt_lds);
        default: return dense_tile<Tile6>(g, r, wg, gt_lds);
    }
}

__global__ __launch_bounds__(256) void dense_gemm_f32_kernel(const DenseGemm g) {
    constexpr int BK = 32, P = BK + 1;
    __shared__ float s_a[64 * P], s_b[64 * P];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, j = lane & 31, kh = lane >> 5;
    int tm, tn;
    tile_of(blockIdx.x, (g.M + 63) / 64, (g.tile_cols + 63) / 64, tm, tn);
    const int m0 = tm * 64, n0 = tn * 64, wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
    const float* A = static_cast<const float*>(g.A);
    if (g.section_n > 0) A += n0 / g.section_n * g.section_a;
    gm_f16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.0f;
    const int r0 = tid >> 2, c0 = (tid & 3) * 8;
    const float* pa = A + (int64_t)min(m0 + r0, g.M - 1) * g.lda + c0;
    const uint16_t* pb = g.W + (int64_t)weight_row(g, n0 + r0) * g.ldw + c0;
    const int steps = (g.K + BK - 1) / BK;
    for (int st = 0; st < steps; ++st) {
        const float4 a0 = *reinterpret_cast<const float4*>(pa + st * BK), a1 = *reinterpret_cast<const float4*>(pa + st * BK + 4);
        const uint4 w = *reinterpret_cast<const uint4*>(pb + st * BK);
        __syncthreads();
        float* d = s_a + r0 * P + c0;
        d[0] = a0.x; d[1] = a0.y; d[2] = a0.z; d[3] = a0.w; d[4] = a1.x; d[5] = a1.y; d[6] = a1.z; d[7] = a1.w;
        d = s_b + r0 * P + c0;
        d[0] = bf16_lo(w.x); d[1] = bf16_hi(w.x); d[2] = bf16_lo(w.y); d[3] = bf16_hi(w.y);
        d[4] = bf16_lo(w.z); d[5] = bf16_hi(w.z); d[6] = bf16_lo(w.w); d[7] = bf16_hi(w.w);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < BK; k += 2)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s_b[(wn + j) * P + k + kh], s_a[(wm + j) * P + k + kh], acc, 0, 0, 0);
    }
    const int m = m0 + wm + j;
    if (m >= g.M) return;
    if (g.epilogue == GEMM_SWIGLU) return store_glu<true>(g, m, n0 + wn, kh, acc);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn + 8 * q + 4 * kh;
        if (n < g.N) store4<true>(g, 0, m, n, acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    }
}

// The times are those of 512 ... 2048 rows times 2560 ... 28672 columns, 40 and 152 steps, the chip nearly full (two thirds empty, a step
// takes a fifth less: the CUs share the power).  Against 128 x 128 tiles of four waves, rows through registers, two workgroups a CU:
// 2048 x 19456 x 2560 240 -> 175 us (gate, up; 1165 TFLOP/s), 2048 x 2560 x 9728 116 -> 85, 1030 x 9728 x 2560 84 -> 57 (895 TFLOP/s).
static const TileKind kinds[] = {tile_kind<Tile0>(1300, 14000), tile_kind<Tile1>(1080, 11000), tile_kind<Tile2>(850, 8500), tile_kind<Tile3>(740, 6000),
                                 tile_kind<Tile4>(500, 6000),   tile_kind<Tile5>(500, 6000),  tile_kind<Tile6>(340, 5000)};

// K splits of 64 x 64 tiles of four waves, 0 where the plan's tiles are done first.  With a CU for each workgroup their step is the shortest
// (330 ns and 4500 in the units above), and two that share a CU take 1.7 times one's: 128 x 1024 x 1024 9.0 us as the plan has it, 7.7 so,
// 300 x 2560 x 2560 17.4 and 15.1, 1030 x 1024 x 128 5.05 and 4.6; split, 128 x 1024 x 2816 6.7 and 5.6.  With more of them a larger tile
// wins: 512 x 2560 x 2560 (320 tiles) 18.1 and 23.1, 300 x 5000 x 320 (395) 6.5 and 7.0.
static int four_wave_splits(const DenseGemm& g, int64_t tiles, int steps, int most, float plan_cost) {
    int best = 0;
    for (int splits = 1; splits == 1 || (splits <= most && splits * 4 <= steps); ++splits) {
        if (tiles * splits > 512) break;
        const float step = tiles * splits > 256 ? 1.7f * 330.0f : 330.0f;
        const float sums = splits > 1 ? (float)splits * (float)g.M * (float)g.N * 2e-3f : 0.0f;
        const float cost = (float)((steps + splits - 1) / splits) * step + 4500.0f + sums;
        if (cost < plan_cost) best = splits, plan_cost = cost;
    }
    return best;
}

// columns that tiles cover: gates and ups in whole blocks of 16
static int tile_columns(const DenseGemm& g) { return g.epilogue == GEMM_SWIGLU ? (g.N / 2 + 15) / 16 * 32 : g.N; }

TilePlan dense_gemm_plan(const DenseGemm& g, bool may_split) {
    const int cols = tile_columns(g), steps = up64(g.K) / 64;
    const int most = may_split && g.slab > 0 ? (int)std::min<int64_t>(16, g.slab_room / g.slab) : 1;
    const int64_t small = ((int64_t)g.M + 63) / 64 * ((cols + 63) / 64);
    TilePlan p{};
    p.splits = 1;
    // offsets in a tile are 32 bits: 255 rows of up to 8 MiB stay under 2 GiB
    if (g.lda <= 1 << 22 && g.ldw <= 1 << 22) {
        // 32-bit results of 50 MB and more behind four steps or fewer are bound by their stores: a launch of two kinds takes 5 to 10 us more than
        // the times above add up to, one of a single kind 2 to 3 less (1500 x 16384 x 64 36.2 us in two kinds, 24.4 in one; 700 x 32768 x 256
        // 41.4 and 33.5).  From five steps on either may win by a tenth, and 16-bit results add up.
        const bool stores = steps <= 4 && (g.epilogue == GEMM_F32 || g.epilogue == GEMM_DECAY) && (int64_t)g.M * cols * 4 >= 50000000;
        p = plan_tiles(kinds, sizeof kinds / sizeof *kinds, g.M, cols, steps, most, g.section_n, stores ? 10000.0f : 0.0f);
        const int splits = four_wave_splits(g, small, steps, most, p.cost);
        if (splits == 0) return p;
        p = TilePlan{};
        p.splits = splits;
    }
    p.wgs = (int)(small * p.splits);
    return p;
}

// Up to so many tiles of 32 x 32 dense_gemm_few_kernel has the few rows; with more of them, larger tiles fill the chip, too, and read X less often:
// 32 x 28672 x 4096 (896) 51.7 us there and 51.3 with few, 64 x 19456 x 2560 (1216) 37.0 and 35.3, 64 x 28672 x 4096 (1792) 56.3 and 68.6, 30 x 65536 x
// 1024 (2048) 28.2 and 31.6.
constexpr int64_t FEW_TILES = 1280;

int dense_gemm(DenseGemm g, hipStream_t s, int* splits) {
    if (!g.A || !g.W || !g.C) return PTM_E_NULL;
    const int kp = up64(g.K);
    const bool glu = g.epilogue == GEMM_SWIGLU;
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.lda <= 0 || g.ldw < kp || g.ldc < (glu ? g.N / 2 : g.N)) return PTM_E_SHAPE;
    if ((glu && (g.N & 1)) || g.section_n < 0 || (g.section_n & 127) || (g.section_a & 7)) return PTM_E_SHAPE;
    if (g.epilogue != GEMM_F32 && splits) return PTM_E_SHAPE;  // partial sums have no epilogue
    if (g.epilogue == GEMM_DECAY && !g.bias) return PTM_E_NULL;
    if (!aligned16(g.A) || !aligned16(g.W) || !aligned16(g.C) || (g.lda & 7) || (g.ldw & 7)) return PTM_E_ALIGN;
    const int cols = g.tile_cols = tile_columns(g);
    auto tiles = [&](int bm, int bn) { return ((int64_t)g.M + bm - 1) / bm * ((cols + bn - 1) / bn); };
    if (tiles(32, 32) * 16 > 0x7fffffff) return PTM_E_UNSUPPORTED;
    // splits that bring `t` tiles to about `target` workgroups, each with at least four steps of K
    auto split = [&](int64_t t, int64_t target) {
        g.splits = 1;
        if (!splits || g.slab <= 0) return;
        int64_t n = (target + t / 2) / t;
        if (n > kp / 256) n = kp / 256;
        if (n > 16) n = 16;
        while (n > 1 && n * g.slab > g.slab_room) --n;
        g.splits = n > 1 ? (int)n : 1;
    };
    if (g.a_fp32) {
        g.splits = 1;
        hipLaunchKernelGGL(dense_gemm_f32_kernel, dim3((unsigned)tiles(64, 64)), dim3(256), 0, s, g);
    } else if (g.M <= 64 && tiles(32, 32) <= FEW_TILES && g.lda <= 1 << 22 && (int64_t)g.N * g.ldw < 1 << 30) {  // (offsets of 32 bits)
        split(tiles(32, 32), 512);
        if (g.splits > kp / 512) g.splits = kp / 512 > 1 ? kp / 512 : 1;  // two steps a wave
        hipLaunchKernelGGL(dense_gemm_few_kernel, dim3((unsigned)(tiles(32, 32) * g.splits)), dim3(64 * FEW_WAVES), 0, s, g);
    } else if (g.M <= 32) {
        split(tiles(32, 128), 512);
        hipLaunchKernelGGL((dense_gemm_kernel<32, 128, 32, 32>), dim3((unsigned)(tiles(32, 128) * g.splits)), dim3(256), 0, s, g);
    } else if (g.M <= 64) {
        split(tiles(64, 64), 512);
        hipLaunchKernelGGL((dense_gemm_kernel<64, 64, 32, 32>), dim3((unsigned)(tiles(64, 64) * g.splits)), dim3(256), 0, s, g);
    } else {
        const TilePlan p = dense_gemm_plan(g, splits != nullptr);
        g.splits = p.splits;
        if (p.regions.n == 0) {
            hipLaunchKernelGGL((dense_gemm_kernel<64, 64, 32, 32>), dim3((unsigned)p.wgs), dim3(256), 0, s, g);
        } else {
            static std::once_flag raised;
            std::call_once(raised, [] {
                (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&dense_gemm_tiles_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            });
            hipLaunchKernelGGL(dense_gemm_tiles_kernel, dim3((unsigned)p.wgs), dim3(512), p.lds, s, g, p.regions);
        }
    }
    if (splits) *splits = g.splits;
    return launch_status();
}

}  // namespace ptm

extern "C" int ptm_dense_gemm(const void* A, int a_fp32, int64_t lda, const void* W, int64_t ldw, float* C, int64_t ldc, int M,
                              int N, int K, ptm_stream_t stream) {
    if (M <= 0 || N <= 0 || K <= 0 || lda < ptm::up64(K)) return PTM_E_SHAPE;
    ptm::DenseGemm g;
    g.A = A;
    g.a_fp32 = a_fp32;
    g.lda = lda;
    g.W = static_cast<const uint16_t*>(W);
    g.ldw = ldw;
    g.M = M;
    g.N = N;
    g.K = K;
    g.C = C;
    g.ldc = ldc;
    return ptm::dense_gemm(g, ptm::as_stream(stream));
}
