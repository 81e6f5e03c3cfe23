// Test harness (not part of the library): the block decoders' prompt product as their runtime calls it, with its epilogues, sections and K
// splits, which the C ABI's plain product does not have, how a launch would cover its output, their decode product with its epilogues, and the quantised
// models' prompt attention, QK-norm, q / k / v and gate / up products and down projection as theirs calls them.  Host C++ only; built by
// __graft_entry__.build() into tests/libshim_harness.so and driven through ctypes by tests/gemm_helpers.py.
#include "dense_gemv.h"
#include "gemm_plan.h"
#include "ptm.h"
#include "recurrent.h"

namespace ptm {
int attention_mfma_order(int dq, int dv, int id, int grid);
int prefill_attention_rows(const float* Q, const void* K_cache, const void* V_cache, float* O, void* rows16, float* rowscale,
                           bool q8round, bool* wrote16, int rows, int n_heads, int n_kv_heads, int head_dim, int64_t pos0, int max_seq,
                           float scale, int kv_fp16, int window, hipStream_t s);
int qgemm_f16_impl(uint32_t ggml_type, const void* W, const void* X, bool x_is_f32, float* Y, int M, int K, int N,
                   int64_t stride, void* workspace, bool accumulate, float* split_ws, size_t split_ws_bytes, bool reuse_rows,
                   hipStream_t s, int* deferred_splits, bool split_scales);
int qgemm_f16_blocks_per_split(int N, int K, int M, size_t split_ws_bytes);
int64_t qgemm_f16_split_scale_bytes(int M);
int qknorm_slabs_per_batch(int most, int64_t waves);
int qknorm_rope_kv_rows_from_parts(const float* const* P, const int* splits, const float* const* bias, float* Q,
                                   const float* q_norm_w, const float* k_norm_w, void* K_cache, void* V_cache,
                                   const float* rope_table, int rows, int n_heads, int n_kv_heads, int head_dim, int64_t pos0,
                                   int max_seq, float eps, int add_one, int kv_fp16, int rope_interleaved, hipStream_t s);
int qgemm_f16_prepare_fused(int pre, const float* X, const float* X2, float eps, int add_one, void* ws_round, void* ws_plain, int M, int K, hipStream_t s);
int qgemm_f16_multi(int n, const uint32_t* types, const void* const* W, const int64_t* strides, const int* N, float* const* Y,
                    int M, int K, void* ws_round, void* ws_plain, float* split_ws, size_t split_ws_bytes, hipStream_t s,
                    const float** deferred_P, int* deferred_splits);
size_t qgemm_f16_multi_split_bytes(int n, const int* N, const uint32_t* types, int K, int M);
void qgemm_f16_multi_plan(int n, const int* N, const uint32_t* types, int K, int M, int* splits);
bool attn_five_waves(int head_dim, int n_heads, int n_kv_heads, int max_seq);
bool q4k_rows_in_order(int N, int K, int waves);
int q6k_rows_waves(int N, int K, bool accumulate);
int qgemm_f16_act_rows(const float* G, const float* U, int sg, int su, bool gelu, bool rounded, void* ws, int bps, int M, int K, hipStream_t s);
}

extern "C" {

struct GemmCall {
    const void* A;
    const void* W;
    void* C;
    const float* bias;
    int64_t lda, ldw, ldc, section_a, slab, slab_room;
    int32_t M, N, K, epilogue, section_n, may_split;
};

static ptm::DenseGemm dense(const GemmCall* c) {
    ptm::DenseGemm g;
    g.A = c->A;
    g.W = static_cast<const uint16_t*>(c->W);
    g.C = c->C;
    g.bias = c->bias;
    g.lda = c->lda;
    g.ldw = c->ldw;
    g.ldc = c->ldc;
    g.section_a = c->section_a;
    g.slab = c->slab;
    g.slab_room = c->slab_room;
    g.M = c->M;
    g.N = c->N;
    g.K = c->K;
    g.epilogue = c->epilogue;
    g.section_n = c->section_n;
    return g;
}

int gemm_run(const GemmCall* c, int32_t* splits, void* stream) {
    int n = 1;
    const int rc = ptm::dense_gemm(dense(c), static_cast<hipStream_t>(stream), c->may_split ? &n : nullptr);
    *splits = n;
    return rc;
}

// splits, workgroups, regions, and of each region its seven numbers
void gemm_plan(const GemmCall* c, int32_t* out) {
    const ptm::TilePlan p = ptm::dense_gemm_plan(dense(c), c->may_split != 0);
    *out++ = p.splits;
    *out++ = p.wgs;
    *out++ = p.regions.n;
    for (int i = 0; i < p.regions.n; ++i) {
        const ptm::GemmRegion& r = p.regions.r[i];
        for (int v : {r.kind, r.first, r.m0, r.n0, r.n1, r.tiles_m, r.tiles_n}) *out++ = v;
    }
}

// y = W . x with one of the epilogues a decode step has; blend (optional): x is a stream of that weight.  GEMV_ARGMAX: (value, index) of
// every workgroup to part_val, part_idx (room for 512); the number of workgroups is returned in *wgs.
int gemv_run(const void* W, const float* x, float* y, int K, int N, int64_t ld, int epilogue, const float* blend, float* part_val, int* part_idx, int* wgs,
             void* stream) {
    ptm::DenseGemv g;
    g.W = static_cast<const uint16_t*>(W);
    g.x = x;
    g.y = y;
    g.K = K;
    g.N = N;
    g.ld = ld;
    g.epilogue = epilogue;
    g.streams = blend ? 1 : 0;
    g.blend = blend;
    g.part_val = part_val;
    g.part_idx = part_idx;
    *wgs = ptm::dense_gemv_workgroups(g);
    return ptm::dense_gemv(g, static_cast<hipStream_t>(stream));
}

// prompt attention that leaves the rows of the next product; *wrote: whether it did (else O has the rows)
int prefill_rows16(const float* Q, const void* K, const void* V, float* O, void* rows16, float* rowscale, int q8round, int* wrote, int rows,
                   int n_heads, int n_kv_heads, int head_dim, int64_t pos0, int max_seq, float scale, int kv_fp16, int window, void* stream) {
    bool w = false;
    const int rc = ptm::prefill_attention_rows(Q, K, V, O, rows16, rowscale, q8round != 0, &w, rows, n_heads, n_kv_heads, head_dim, pos0,
                                               max_seq, scale, kv_fp16, window, static_cast<hipStream_t>(stream));
    *wrote = w ? 1 : 0;
    return rc;
}

// QK-norm, rotation and append of rows that are still splits[i] slabs of q, k, v
int qk_rows(const float* const* P, const int* splits, const float* const* bias, float* Q, const float* qw, const float* kw, void* K, void* V, const float* rope,
            int rows, int n_heads, int n_kv_heads, int head_dim, int64_t pos0, int max_seq, int kv_fp16, int interleaved, void* stream) {
    return ptm::qknorm_rope_kv_rows_from_parts(P, splits, bias, Q, qw, kw, K, V, rope, rows, n_heads, n_kv_heads, head_dim, pos0, max_seq, 1e-6f, 0, kv_fp16,
                                               interleaved, static_cast<hipStream_t>(stream));
}
int qk_rows_batch(int most, int64_t waves) { return ptm::qknorm_slabs_per_batch(most, waves); }

// Y[i] = RMSNorm(X; gamma) . W[i]^T of up to three matrices in one launch; P / splits (optional): their slabs instead
int multi_run(int n, const uint32_t* types, const void* const* W, const int64_t* strides, const int* N, float* const* Y, const float* X, const float* gamma, int M,
              int K, void* ws_round, void* ws_plain, float* split_ws, int64_t split_bytes, const float** P, int* splits, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int rc = ptm::qgemm_f16_prepare_fused(1, X, gamma, 1e-6f, 0, ws_round, ws_plain, M, K, s);
    return rc ? rc : ptm::qgemm_f16_multi(n, types, W, strides, N, Y, M, K, ws_round, ws_plain, split_ws, (size_t)split_bytes, s, P, splits);
}
int64_t multi_split_bytes(int n, const int* N, const uint32_t* types, int K, int M) { return (int64_t)ptm::qgemm_f16_multi_split_bytes(n, N, types, K, M); }
void multi_plan(int n, const int* N, const uint32_t* types, int K, int M, int* splits) { ptm::qgemm_f16_multi_plan(n, N, types, K, M, splits); }

int attn_five_waves(int head_dim, int n_heads, int n_kv_heads, int max_seq) { return ptm::attn_five_waves(head_dim, n_heads, n_kv_heads, max_seq) ? 1 : 0; }
int q4k_rows_in_order(int N, int K, int waves) { return ptm::q4k_rows_in_order(N, K, waves) ? 1 : 0; }
int q6k_rows_waves(int N, int K, int accumulate) { return ptm::q6k_rows_waves(N, K, accumulate != 0); }

int64_t act_down_bytes(int M, int K) { return ptm_qgemm_f16_workspace_bytes(M, K) + ptm::qgemm_f16_split_scale_bytes(M); }
// Y = down . (act(gate) . up) of rows that are still slabs, in ws of act_down_bytes
int act_down(uint32_t type, const void* W, int64_t stride, const float* G, const float* U, int sg, int su, int gelu, float* Y, int M, int K, int N, void* ws,
             float* split_ws, int64_t split_bytes, void* stream) {
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int bps = ptm::qgemm_f16_blocks_per_split(N, K, M, (size_t)split_bytes);
    const int rc = ptm::qgemm_f16_act_rows(G, U, sg, su, gelu != 0, type == PTM_TYPE_Q4_K, ws, bps, M, K, s);
    return rc ? rc : ptm::qgemm_f16_impl(type, W, G, true, Y, M, K, N, stride, ws, false, split_ws, (size_t)split_bytes, true, s, nullptr, true);
}

// prompt rows of a state-space mixer, fp32: weights w = conv, conv_b, dt_bias, neg_a, D, norm; scratch = conv rows, decays, tiles, y
int64_t ssm_scratch(int heads, int vdim, int state, int groups, int M, int what) {
    ptm::SsmShape m{};
    m.heads = heads;
    m.vdim = vdim;
    m.state = state;
    m.groups = groups;
    return what == 0 ? ptm::ssm_conv_row(m) * M : what == 1 ? 2 * (int64_t)heads * M : what == 2 ? ptm::ssm_tile_floats(heads, M) : (int64_t)heads * vdim * M;
}
int ssm_run(const int* shape, const float* const* w, const float* proj, int M, int64_t pos0, float* ring, float* state, float* const* scratch, float* out, void* stream) {
    ptm::SsmRows r{};
    r.m = {shape[0], shape[1], shape[2], shape[3], shape[4], 1, w[0], w[1], w[2], w[3], w[4], w[5], 1.0f};
    const int inner = r.m.heads * r.m.vdim;
    r.proj = proj;
    r.ld = 2 * inner + 2 * r.m.groups * r.m.state + r.m.heads;
    r.M = M;
    r.pos0 = pos0;
    r.eps = 1e-6f;
    r.ring = ring;
    r.state = state;
    r.conv = scratch[0];
    r.decay = scratch[1];
    r.tiles = scratch[2];
    r.y = scratch[3];
    r.out = out;
    r.out_ld = inner;
    return ptm::ssm_rows(r, true, static_cast<hipStream_t>(stream));
}
// prompt rows of a WKV mixer, fp32: proj rows of r, k, v, g and decays
int64_t wkv_scratch(int heads, int dim, int M, int what) { return what == 0 ? ptm::wkv_tile_floats(heads, dim, M) : (int64_t)heads * dim * M; }
int wkv_run(int heads, int dim, const float* proj, const float* u, const float* norm, int M, int64_t pos0, float* state, float* const* scratch, const float* h_last, float* shift,
            float* out, void* stream) {
    ptm::WkvRows w{};
    w.proj = proj;
    w.section = (int64_t)heads * dim;
    w.ld = 5 * w.section;
    w.M = M;
    w.heads = heads;
    w.dim = dim;
    w.u = u;
    w.norm = norm;
    w.eps = 1e-6f;
    w.pos0 = pos0;
    w.state = state;
    w.tiles = scratch[0];
    w.o = scratch[1];
    w.o_ld = w.section;
    w.out = out;
    w.out_ld = w.section;
    w.h_last = h_last;
    w.shift = shift;
    w.wp = 64;
    return ptm::wkv_rows(w, true, static_cast<hipStream_t>(stream));
}
int64_t ssm_state_floats(int heads, int state, int vdim) { return ptm::recurrent_state_floats(heads, state, vdim); }

int attention_order(int dq, int dv, int id, int grid) { return ptm::attention_mfma_order(dq, dv, id, grid); }

}  // extern "C"
