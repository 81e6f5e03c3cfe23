// The main loop of the prompt products: one workgroup of eight waves, BM rows of X times BN rows of W, 64 values of K per step,
// bfloat16 operands, fp32 sums on v_mfma_f32_16x16x32.
//
// LDS holds two or three steps of either side.  A row of a step is 128 bytes, its eight 16-byte pieces stored at piece ^ (row % 8), so the
// fragment reads (16 rows, four pieces) use every bank evenly.  Rows go from memory to LDS without passing registers (buffer_load ... lds: a
// wave's instruction fills 8 rows, the lanes' global addresses carry the permutation); a step has one barrier, in front of its last quarter,
// and the fetches behind it are the ones into the LDS it freed.
//
// What bounds it: 8192 x 8192 x 8192 in 256 x 256 tiles runs at 1190 ... 1400 TFLOP/s on different boxes (a library's product: 1350 ... 1626).  The
// matrix cores are busy 71 % of the clocks, fragment reads have no bank conflicts, and a wave spends the rest at the barrier of a step and on its
// reads; 2048 x 19456 x 2560 177 us = 1153 TFLOP/s (the library's 188), busy 50 %, the last round of tiles included, before the tiles' ends took a sixth
// of the instructions (gates and ups so, under a tracer, 182 -> 171).  Reads and fetches in bursts
// behind the barrier cost 10 % more than spread between the MFMAs; four waves with twice the fragments each read a third less LDS and were slower
// (1160 where this has 1200); workgroups ordered by rows alone, without bands, 900.  Small tiles are bound by how long a fetch takes: three
// steps in LDS against two bring 128 x 128 from 545 to 760, 128 x 256 from 890 to 1050.
#pragma once
#include "gemm_plan.h"
#include "ptm_common.h"

namespace ptm {

typedef float gt_f4 __attribute__((ext_vector_type(4)));
typedef int gt_i4 __attribute__((ext_vector_type(4)));
typedef __bf16 gt_b8 __attribute__((ext_vector_type(8)));

// 16 bytes per lane from base + voff + soff to LDS bytes [lds, lds + 1024), lane after lane
__device__ __forceinline__ void gt_to_lds(uint32_t lds, int voff, gt_i4 base, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(base), "s"(soff) : "memory");
}
// 4 bytes per lane to LDS bytes [lds, lds + 256)
__device__ __forceinline__ void gt_word_to_lds(uint32_t lds, int voff, gt_i4 base, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(lds), "v"(voff), "s"(base), "s"(soff) : "memory");
}
__device__ __forceinline__ gt_i4 gt_buffer(const void* p) {
    const uint64_t a = reinterpret_cast<uint64_t>(p);
    return gt_i4{(int)(uint32_t)a, (int)((a >> 32) & 0xffffu), -1, 0x00020000};
}

// all but the last N of this wave's fetches have arrived and it has what it read from LDS; then the same of the workgroup's other waves
template <int N>
__device__ __forceinline__ void gt_arrived() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory"); }

// Where row r of a tile of W lies in the product: a lane's sums of two fragments are then eight consecutive columns.
__device__ __forceinline__ int gt_column(int r) { return (r & ~31) + ((r & 12) << 1) + ((r & 16) >> 2) + (r & 3); }

// RX, RW: 16-row fragments of X and W of a wave; WX waves along the rows of X, 8 / WX along those of W; XN, WN: steps of X and W in LDS
template <int RX, int RW, int WX, int XN, int WN>
struct GemmTile {
    static_assert((16 * RX * WX) % 64 == 0 && (16 * RW * (8 / WX)) % 64 == 0 && RX % 2 == 0 && RW % 2 == 0, "whole fetch instructions, halves of X, pairs of sums");
    static_assert(XN <= WN && (XN == 2 || XN == 3) && (WN == 2 || WN == 3), "the wait counts");
    static constexpr int BM = 16 * RX * WX, BN = 16 * RW * (8 / WX), THREADS = 512;
    static constexpr int XB = BM * 128, WB = BN * 128;  // LDS bytes of a step
    static constexpr int LDS = XN * XB + WN * WB;
    static constexpr int NX = BM / 64, NW = BN / 64;    // fetch instructions of a wave for a step
    gt_f4 acc[RX][RW];

    // fetch_x / fetch_w (step, piece, LDS offset): one instruction's share of a step's rows
    template <typename FetchX, typename FetchW>
    __device__ __forceinline__ void run(uint8_t* lds, int steps, FetchX&& fetch_x, FetchW&& fetch_w) {
        constexpr int HX = RX / 2;
        constexpr int LATER = WN == 2 ? 0 : NW + (XN == 3 ? NX : 0);  // fetches of step st + 2 that are out when step st + 1 is waited for
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int j = lane & 15, g = lane >> 4;
        const int wx = (wave % WX) * 16 * RX, ww = (wave / WX) * 16 * RW;
#pragma unroll
        for (int a = 0; a < RX; ++a)
#pragma unroll
            for (int b = 0; b < RW; ++b) acc[a][b] = gt_f4{0.f, 0.f, 0.f, 0.f};
        const int p0 = (g ^ (j & 7)) << 4, p1 = ((4 + g) ^ (j & 7)) << 4;
        const uint8_t* x0 = lds + (wx + j) * 128;
        const uint8_t* w0 = lds + XN * XB + (ww + j) * 128;
        gt_b8 x[2][HX], w[2][RW];
        auto read_x = [&](int half, int k, int at, int a) { x[half][a] = *reinterpret_cast<const gt_b8*>(x0 + at + (k ? p1 : p0) + (half * HX + a) * 2048); };
        auto read_w = [&](int k, int at, int b) { w[k][b] = *reinterpret_cast<const gt_b8*>(w0 + at + (k ? p1 : p0) + b * 2048); };
        // a quarter of a step: half of the wave's X rows times half of the step's K.  Memory instructions go out between the MFMAs of two X
        // fragments, a few at a time: in one burst behind the barrier they hold up the MFMAs of all eight waves.
        auto quarter = [&](int half, int k, auto&& between) {
#pragma unroll
            for (int a = 0; a < HX; ++a) {
                between(a);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int b = 0; b < RW; ++b) acc[half * HX + a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k][b], x[half][a], acc[half * HX + a][b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        // the a-th of HX equal shares of n things
        auto share = [](int a, int n, auto&& f) {
#pragma unroll
            for (int i = 0; i < n; ++i)
                if (i * HX / n == a) f(i);
        };
#pragma unroll
        for (int st = 0; st < WN; ++st) {
            if (st >= steps) break;
            if (st < XN)
                for (int i = 0; i < NX; ++i) fetch_x(st, i, st * XB);
            for (int i = 0; i < NW; ++i) fetch_w(st, i, XN * XB + st * WB);
        }
        if (steps >= WN) gt_arrived<(XN - 1) * NX + (WN - 1) * NW>();
        else gt_arrived<0>();
        int xb = 0, wb = 0, wfree = 0;
#pragma unroll
        for (int b = 0; b < RW; ++b) read_w(0, 0, b);
#pragma unroll
        for (int a = 0; a < HX; ++a) read_x(0, 0, 0, a);
        for (int st = 0; st < steps; ++st) {
            const int xnext = xb == (XN - 1) * XB ? 0 : xb + XB, wnext = wb == (WN - 1) * WB ? 0 : wb + WB;
            quarter(0, 0, [&](int a) {
                if (st > 0 && st - 1 + WN < steps) share(a, NW, [&](int i) { fetch_w(st - 1 + WN, i, XN * XB + wfree); });
                read_x(1, 0, xb, a);
            });
            quarter(1, 0, [&](int a) {
                share(a, RW + HX, [&](int i) {
                    if (i < RW) read_w(1, wb, i);
                    else read_x(0, 1, xb, i - RW);
                });
            });
            quarter(0, 1, [&](int a) { read_x(1, 1, xb, a); });
            // this step's LDS has been read by every wave, the next step's rows have arrived
            if (LATER > 0 && st + 2 < steps) gt_arrived<LATER>();
            else gt_arrived<0>();
            quarter(1, 1, [&](int a) {
                if (st + 1 < steps) share(a, RW + HX, [&](int i) {
                    if (i < RW) read_w(0, wnext, i);
                    else read_x(0, 0, xnext, i - RW);
                });
                if (st + XN < steps) share(a, NX, [&](int i) { fetch_x(st + XN, i, xb); });
            });
            wfree = wb;
            xb = xnext;
            wb = wnext;
        }
    }

    // where the lane's sums acc[0][0] lie: row of X, first of four rows of W; acc[a][b] are 16 a and 16 b on
    static __device__ __forceinline__ int lane_row() { return ((threadIdx.x >> 6) % WX) * 16 * RX + (threadIdx.x & 15); }
    static __device__ __forceinline__ int lane_col() { return ((threadIdx.x >> 6) / WX) * 16 * RW + 4 * ((threadIdx.x >> 4) & 3); }
    static constexpr int ROWS = RX, COLS = RW;
    // use(a, b, row of X, row of W): the sums acc[a][b] and acc[a][b + 1] are of rows .. + 0, 1, 2, 3 and .. + 16, 17, 18, 19 of W in LDS
    template <typename Use>
    __device__ __forceinline__ void each(Use&& use) const {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int wx = (wave % WX) * 16 * RX + (lane & 15), ww = (wave / WX) * 16 * RW + 4 * (lane >> 4);
#pragma unroll
        for (int a = 0; a < RX; ++a)
#pragma unroll
            for (int b = 0; b < RW; b += 2) use(a, b, wx + 16 * a, ww + 16 * b);
    }
};

// step, ends: what a workgroup takes for a step of 64 values and for its start and end (ns)
template <typename Tile>
constexpr TileKind tile_kind(float step, float ends) {
    return {Tile::BM, Tile::BN, step, ends, Tile::LDS};
}

}  // namespace ptm
