// Products of bfloat16 weights and one vector: what a call describes.  Host side, no device code.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace ptm {

enum { GEMV_STORE = 0, GEMV_RELU2 = 1, GEMV_SIDE = 2, GEMV_ARGMAX = 3, GEMV_SWIGLU = 4 };
constexpr int GEMV_SECTIONS = 8;

// y = epilogue(W . prologue(x)).  Vectors are fp32, zero-padded to a multiple of 64 values.
// Prologue: x' = x + RMS(h) * hw + add0 + add1 (each part optional; x' stored to xout by one workgroup), then RMS(x') * gamma if
// gamma is given (stored to xn_out by one workgroup).
// With streams > 0, x is that many vectors x_stride floats apart: x' = sum_s blend[s] x_s + blend[streams] h, and with h the first
// workgroups store the new streams sum_s store[t][s] x_s + store[t][streams] h to xout (K-padded rows); layer norm if beta is
// given; then the token shift: rows of section i take x' + (x'_before - x') * mu[i], x'_before from the ring slot of the previous position.
// With tail_n > 0 (no other prologue), values tail0 .. of x are RMS-normed in tail_parts equal parts, times tail_norm * tail_scale.
// GEMV_SWIGLU: W holds N gate rows, then N up rows; y = silu(gate) * up.
struct DenseGemv {
    // what a plain product reads lies in one cache line of kernel arguments, a norm's vectors in the next: a line first read late in the
    // kernel is a round trip to memory there
    const uint16_t* W = nullptr;
    const float* x = nullptr;
    float* y = nullptr;
    int64_t ld = 0;
    int N = 0, K = 0;
    int epilogue = GEMV_STORE;
    float out_scale = 1.0f;          // factor of every stored y
    int waves = 0, wgs = 0;          // of the launch, set by dense_gemv
    float eps = 0.0f;
    int sections = 0;
    const float *h = nullptr, *hw = nullptr, *add0 = nullptr, *add1 = nullptr;
    float* xout = nullptr;
    const float* gamma = nullptr;
    float* xn_out = nullptr;
    const uint16_t* side = nullptr;  // GEMV_SIDE: row *d_token of the table, from column side_off
    int64_t side_ld = 0;
    int side_off = 0;
    const int* d_token = nullptr;
    float* part_val = nullptr;       // GEMV_ARGMAX: one (value, index) per workgroup
    int* part_idx = nullptr;
    int streams = 0;
    int64_t x_stride = 0;
    const float *blend = nullptr, *store = nullptr, *beta = nullptr;
    const float* mu = nullptr;       // [sections][padded K]
    float* shift = nullptr;          // [2][padded K], by position parity
    const int64_t* d_past = nullptr;
    int section_row[GEMV_SECTIONS + 1] = {};  // first rows; the last entry is N
    int section_wg[GEMV_SECTIONS + 1] = {};   // first workgroups, set by dense_gemv
    int tail0 = 0, tail_n = 0, tail_parts = 0;
    const float* tail_norm = nullptr;
    float tail_scale = 1.0f;
};
int dense_gemv_workgroups(const DenseGemv& g);
int dense_gemv(DenseGemv g, hipStream_t s);
void dense_gemv_init();

}  // namespace ptm
