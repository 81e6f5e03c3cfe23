// What the attention kernels of the block decoders share (mixer_attention.hip, prompt_attention.hip).
#pragma once
#include "dense.h"

namespace ptm {

typedef __bf16 at_b8 __attribute__((ext_vector_type(8)));
typedef short at_s4 __attribute__((ext_vector_type(4)));
typedef float at_f4 __attribute__((ext_vector_type(4)));
typedef float at_f16 __attribute__((ext_vector_type(16)));
constexpr float LOG2E = 1.44269504088896340736f;

// ds_read_b64_tr_b16: within each group of 16 lanes, lane i passes the address of four 16-bit values (row i / 4 of a 4-row
// block, columns 4 (i % 4) .. +3 of a 16-column block) and receives column i of the four rows.
__device__ __forceinline__ at_s4 lds_tr16(const uint8_t* p) {
    typedef __attribute__((address_space(3))) at_s4 lds_s4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
}
__device__ __forceinline__ short bf_bits(float f) { return (short)f_bf16(f); }
__device__ __forceinline__ float bf_val(short s) { return bf16_f((uint16_t)s); }
// cap * tanh(s / cap); 1 - 2 / (e^2y + 1) ends at +-1 for large arguments
__device__ __forceinline__ float soft_cap(float s, float cap, float inv_cap) {
    const float e = __builtin_amdgcn_exp2f(s * inv_cap * (2.0f * LOG2E));
    return cap * (1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f));
}

// factor of value dimension v of a finished result: output gate and scale
__device__ __forceinline__ float out_factor(const ptm_attention_args& a, int64_t row, int head, int v) {
    const float s = a.out_scale != 0.0f ? a.out_scale : 1.0f;
    return a.gate && v < a.gate_head ? s * sigmoid_f(a.gate[row * a.gate_row + (int64_t)head * a.gate_head + v]) : s;
}

// prompt rows, bfloat16, heads of up to 256 (attention_rows has checked the arguments)
int attention_mfma(const ptm_attention_args& a, hipStream_t s);

}  // namespace ptm
