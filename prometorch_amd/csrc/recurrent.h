// Recurrent mixers (recurrent.hip): what their calls describe.  Host side, no device code.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace ptm {

bool recurrent_supported(int keys);
int64_t recurrent_state_floats(int heads, int keys, int columns);

struct WkvStep {
    const float* proj;        // [r | k | v | g | low-rank]
    const uint16_t* w2;       // [heads * dim][w2_ld]
    int64_t w2_ld;
    int heads, dim, rank;
    const float *w0, *u, *norm;
    float eps;
    const int64_t* d_past;
    float* state;
    float* out;               // [heads * dim]
};
int wkv_step(const WkvStep& a, hipStream_t s);

struct WkvRows {
    const float* proj;        // [M][ld]: r, k, v, g and the decays w, `section` floats apart
    int64_t ld, section;
    int M, heads, dim;
    const float *u, *norm;
    float eps;
    int64_t pos0;
    float* state;
    float* tiles;             // wkv_tile_floats, 16-byte aligned
    float* o;                 // [M][o_ld]
    int64_t o_ld;
    int keys;                 // set by wkv_rows
    void* out;                // [M][out_ld]
    int64_t out_ld;
    const float* h_last;      // the mixer's last input row, kept for the next token's shift
    float* shift;
    int wp;
};
int wkv_rows(WkvRows a, bool fp32, hipStream_t s);
int64_t wkv_tile_floats(int heads, int dim, int rows);
int token_shift_rows(const float* h, const float* shift, const float* mu, int n, int rows, int64_t pos0, int wp, bool fp32, void* out, hipStream_t s);
int tanh_rows(const float* g, int slabs, int64_t slab, int rows, int n, bool fp32, void* out, hipStream_t s);

struct SsmShape {
    int heads, vdim, state, groups, taps, norm_groups;
    const float *conv, *conv_b, *dt_bias, *neg_a, *D, *norm;  // neg_a: -exp(A_log)
    float scale;
};
struct SsmStep {
    SsmShape m;
    const float* proj;        // [z | x | B | C | dt]
    const int64_t* d_past;
    float *ring, *state;      // [taps][channels]; state
    float* out;               // [heads * vdim], before its norm
};
int ssm_step(const SsmStep& a, hipStream_t s);
struct SsmRows {
    SsmShape m;
    const float* proj;        // [M][ld]
    int64_t ld;
    int M;
    int64_t pos0;
    float eps;
    float *ring, *state;
    float* conv;              // [M][ssm_conv_row]: x | B | C, 16-byte aligned
    float* decay;             // [M][2][heads]
    float* tiles;             // ssm_tile_floats, 16-byte aligned
    float* y;                 // [M][heads * vdim]
    int64_t conv_ld;          // these two set by ssm_rows
    int keys;
    void* out;                // [M][out_ld]
    int64_t out_ld;
};
int ssm_rows(SsmRows a, bool fp32, hipStream_t s);
int64_t ssm_conv_row(const SsmShape& m);
int64_t ssm_tile_floats(int heads, int rows);

}  // namespace ptm
