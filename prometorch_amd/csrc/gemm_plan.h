// Products of bfloat16 rows and weights: what a call describes, and how a launch covers its output.  Host side, no device code.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace ptm {

// C = epilogue(A . W^T): GEMM_F32 fp32 C; otherwise element type of the rows (bfloat16, or fp32 when a_fp32).
// GEMM_SWIGLU: W holds N / 2 gate rows, then N / 2 up rows; C [M][N / 2] = silu(gate) * up.
// GEMM_DECAY: fp32 C = exp(-exp(product + bias)).
enum { GEMM_F32 = 0, GEMM_ELEM = 1, GEMM_RELU2 = 2, GEMM_SWIGLU = 3, GEMM_DECAY = 4 };
struct DenseGemm {
    const void* A = nullptr;
    int a_fp32 = 0;
    int64_t lda = 0;
    const uint16_t* W = nullptr;
    int64_t ldw = 0;
    int M = 0, N = 0, K = 0;
    int epilogue = GEMM_F32;
    void* C = nullptr;
    int64_t ldc = 0;
    // K split over workgroups where the output has too few tiles (GEMM_F32 only): split z leaves its partial sums at
    // C + z * slab; slab_room floats are available for all of them
    int64_t slab = 0, slab_room = 0;
    int splits = 1, tile_cols = 0;  // set by dense_gemm
    // rows n of W take A + n / section_n * section_a (section_n a multiple of 128; 0: one section)
    int section_n = 0;
    int64_t section_a = 0;
    const float* bias = nullptr;  // [N], GEMM_DECAY
};
int dense_gemm(DenseGemm g, hipStream_t s, int* splits = nullptr);

// ---- how a launch covers its output ----------------------------------------------------------------------------------------
// Rows m0 .. and columns n0 .. n1 - 1 in tiles_m x tiles_n tiles of one kind, workgroups first .. (the K splits one after the other).
struct GemmRegion {
    int kind, first, m0, n0, n1, tiles_m, tiles_n;
};
struct GemmRegions {
    int n;
    GemmRegion r[4];
};

// A kind of tile: its size, what a workgroup takes for a step of 64 values and for its start and end (ns), its LDS.
struct TileKind {
    int bm, bn;
    float step, ends;
    int lds;
};
struct TilePlan {
    GemmRegions regions;
    int splits, wgs, lds;
    float cost;
};

// When the last of 256 CUs is done that take workgroups one after the other, `count` of `each` ns at a time
class ChipTime {
    struct Part { float t; int n; };
    Part p[10];
    int parts = 1;

public:
    ChipTime() { p[0] = {0.0f, 256}; }
    void run(int64_t count, float each) {
        while (count > 0) {
            int i = 0;
            for (int k = 1; k < parts; ++k)
                if (p[k].t < p[i].t) i = k;
            if (count >= p[i].n || parts == 10) {
                count -= p[i].n;
                p[i].t += each;
            } else {
                p[i].n -= (int)count;
                p[parts++] = {p[i].t + each, (int)count};
                count = 0;
            }
        }
    }
    float last() const {
        float t = 0.0f;
        for (int k = 0; k < parts; ++k) t = p[k].t > t ? p[k].t : t;
        return t;
    }
};

// The regions, kinds and K splits (at most most_splits) that bring M x N outputs of `steps` steps of K to the shortest time: whole
// rounds of the chip in one kind of tile, the columns and rows left over in smaller ones, where a last round of the large tiles would leave
// most of the chip idle or work on rows that are not there.  section_n > 0: no tile crosses a multiple of it.  second_kind: what a
// launch of more than one kind takes beyond that (ns).
TilePlan plan_tiles(const TileKind* kinds, int n_kinds, int M, int N, int steps, int most_splits, int section_n, float second_kind);

// What dense_gemm launches for more than 64 bfloat16 rows; may_split: the caller takes partial sums.  No regions: `splits` K splits of
// 64 x 64 tiles of four waves.
TilePlan dense_gemm_plan(const DenseGemm& g, bool may_split);

}  // namespace ptm
