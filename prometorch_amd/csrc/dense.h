// Interfaces between the block-decoder runtime (blocks.hip) and its kernels (dense_gemv.hip, dense_gemm.hip,
// mixer_attention.hip).  Host side; not part of the C ABI.
#pragma once
#include "dense_gemv.h"
#include "recurrent.h"
#include "gemm_plan.h"
#include "ptm_common.h"

namespace ptm {

inline int up8(int n) { return (n + 7) & ~7; }
inline int up64(int n) { return (n + 63) & ~63; }

__device__ __forceinline__ float bf16_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ float bf16_f(uint16_t u) { return __uint_as_float((uint32_t)u << 16); }
__device__ __forceinline__ uint16_t f_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }  // nearest even

// element access of an activation / cache buffer: bfloat16 or fp32
template <bool F32>
__device__ __forceinline__ void put_elem(void* p, int64_t i, float v) {
    if constexpr (F32) static_cast<float*>(p)[i] = v;
    else static_cast<uint16_t*>(p)[i] = f_bf16(v);
}
template <bool F32>
__device__ __forceinline__ float get_elem(const void* p, int64_t i) {
    if constexpr (F32) return static_cast<const float*>(p)[i];
    else return bf16_f(static_cast<const uint16_t*>(p)[i]);
}

__device__ __forceinline__ float gelu_tanh(float z) {
    return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }

// block-wide sum for `waves` waves; red: `waves` floats of LDS
__device__ __forceinline__ float block_sum(float v, float* red, int waves) {
    v = sum64(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    float s = 0.0f;
    for (int w = 0; w < waves; ++w) s += red[w];
    return s;
}
template <int WAVES>
__device__ __forceinline__ float block_sum(float v, float* red) {
    return block_sum(v, red, WAVES);
}

// One decode step of a latent mixer around its attention.
struct LatentStep {
    const float* proj;        // [heads * (dim + rot_dim)] q, then kv_rank latent values and rot_dim key values
    const float* c_norm;      // [kv_rank]
    const float* rope;        // [max_seq][rot.dims / 2][2]
    const uint16_t* expand;   // W_uk rows, then W_uv rows (per head padded to 8 rows)
    int64_t ld;
    int heads, dim, rot_dim, rot_dims, kv_rank, vdim;
    float eps;
    const int64_t* d_past;
    void* q;                  // [heads][up8(kv_rank) + up8(rot_dim)]: fp32, or two bfloat16 planes of that (tiled attention)
    int q_planes;
    void* cache;              // [max_seq][up8(kv_rank) + up8(rot_dim)]
    int fp32;
};
int latent_absorb(const LatentStep& a, hipStream_t s);
// out[h * up8(vdim) + v] = W_uv[h] . merged latent of head h; pM / pL NULL: pO is the finished latent [heads][o_row]
int latent_out(const LatentStep& a, const float* pO, const float* pM, const float* pL, int splits, int o_row, float* out,
               hipStream_t s);

// Attention of one decode token, position *d_past.  bfloat16 caches with tile classes the matrix-core kernel has: splits
// partial results (decode_attention_splits); otherwise one finished result.
struct DecodeAttention {
    ptm_attention_args a;      // rows 1; Q (unless raw is given): two bfloat16 planes [2][heads][dim1 + dim2] that add up to q
    const int64_t* d_past;
    int max_seq;
    // attention mixer: un-normed projections, finished in the prologue, and the rows appended to the caches
    const float* raw = nullptr;  // [q | k | v]
    const float *q_norm = nullptr, *k_norm = nullptr, *rope = nullptr;
    int dim = 0, vdim_true = 0, rot_dims = 0;
    float eps = 0.0f;
    int head_norm = 0, values_are_keys = 0;  // q and k normed per head; v = the un-normed k
    void *k_cache = nullptr, *v_cache = nullptr;
    float *pO = nullptr, *pM = nullptr, *pL = nullptr;  // [splits][heads][vdim], [splits][heads] twice
};
bool decode_attention_tiled(const ptm_attention_args& a);
int decode_attention_splits(const ptm_attention_args& a, int max_seq);
int decode_attention(const DecodeAttention& a, hipStream_t s);
// a: heads, vdim, and the sink, gate and scale of the finished values
int decode_attention_merge(const float* pO, const float* pM, const float* pL, int splits, const ptm_attention_args& a, float* out,
                           hipStream_t s);
int attention_rows(const ptm_attention_args& a, const int64_t* d_past, bool q_fp32_out_fp32, hipStream_t s);

int argmax_finish(const float* part_val, const int* part_idx, int n, int64_t* out_index, const ArgmaxAdvance adv, hipStream_t s);

}  // namespace ptm
