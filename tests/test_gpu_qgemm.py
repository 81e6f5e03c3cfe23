"""GPU parity of the prefill GEMM (MFMA) against M single-row oracle GEMVs, which is what the
reference's matmul_q computes for M > 1 (torch/io/gguf_model.h:7029-7036): every output row must equal the
GEMV of that row of X.

Bars: Q4_K rows bit-identical to the oracle for even N (exact integer sub-block dots, same fp32 chain
order), within 1e-3 of rms(y) otherwise; Q6_K within 1e-3 of rms(y) (the path's stated bar is 1e-2)."""
import numpy as np
import pytest
import torch

from conftest import bits
from prometorch_amd import ops
from prometorch_amd.testing import synth
from prometorch_amd._lib import PtmError

pytestmark = pytest.mark.gpu

QGEMM_TOL = 1e-3


def bf16_round(x):
    """fp32 -> nearest-even bf16, returned as (uint16 bits, fp32 value)."""
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    u = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
    b = u.astype(np.uint16)
    return b, (b.astype(np.uint32) << 16).view(np.float32)


def gpu_qgemm(qt, W, xb, M, K, N):
    Wd = torch.from_numpy(W).cuda()
    Xd = torch.from_numpy(xb.view(np.int16)).cuda()
    Y = torch.full((M, N), 77.0, device="cuda")
    ws = torch.empty(max(16, ops.qgemm_workspace_bytes(M, K)), dtype=torch.uint8, device="cuda")
    ops.matmul_q(qt, Wd, Xd, Y, M, K, N, W.shape[1], ws)
    torch.cuda.synchronize()
    return Y.cpu().numpy()


def gpu_qgemm_f16(qt, W, xb, M, K, N):
    Wd = torch.from_numpy(W).cuda()
    Xd = torch.from_numpy(xb.view(np.int16)).cuda()
    Y = torch.full((M, N), 77.0, device="cuda")
    ws = torch.empty(ops.qgemm_f16_workspace_bytes(M, K), dtype=torch.uint8, device="cuda")
    ops.matmul_q_f16(qt, Wd, Xd, Y, M, K, N, W.shape[1], ws)
    torch.cuda.synchronize()
    return Y.cpu().numpy()


def oracle_rows(po, qt, W, xf):
    return np.stack([po.gemv(qt, W, xf[m]) for m in range(xf.shape[0])])


def rel_err(y, ref):
    ref = ref.astype(np.float64)
    return float(np.abs(y.astype(np.float64) - ref).max() / max(np.sqrt((ref ** 2).mean()), 1e-30))


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 256, 16), (5, 512, 48), (64, 512, 128), (70, 1024, 130), (129, 2560, 334),
                                   (33, 256, 7)])
def test_qgemm_rows_equal_gemv(dev, po, qt, M, K, N):
    r = synth.rng_for(41, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, xf = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    Y = gpu_qgemm(qt, W, xb, M, K, N)
    ref = oracle_rows(po, qt, W, xf)
    e = rel_err(Y, ref)
    print(qt, M, K, N, "rel err", e, flush=True)
    assert e <= QGEMM_TOL
    if qt == 12:
        # the odd last row of the reference GEMV uses a single accumulation chain; all others must match exactly
        n_pair = N - (N & 1)
        assert np.array_equal(bits(Y[:, :n_pair]), bits(ref[:, :n_pair]))


def test_qgemm_zero_and_extreme_rows(dev, po):
    M, K, N = 20, 512, 64
    r = synth.rng_for(42)
    x = r.standard_normal((M, K), dtype=np.float32)
    x[3] = 0.0
    x[4] *= 1e20
    x[5] *= 1e-30
    x[6, ::2] = 0.0
    xb, xf = bf16_round(x)
    for qt in (12, 14):
        W = synth.make_weight(r, qt, N, K)
        Y = gpu_qgemm(qt, W, xb, M, K, N)
        ref = oracle_rows(po, qt, W, xf)
        assert np.all(Y[3] == 0.0)
        for m in range(M):
            assert rel_err(Y[m], ref[m]) <= QGEMM_TOL, (qt, m)


@pytest.mark.parametrize("qt,N,K", [(12, 4096, 4096), (12, 1024, 4096), (14, 4096, 14336)])
def test_qgemm_llama3_8b_layer_shapes_m512(dev, po, qt, N, K):
    """The prefill case the path is specified on: one Llama-3-8B layer's matrices, 512 bf16 rows."""
    M = 512
    r = synth.rng_for(43, qt, N, K)
    W = synth.make_weight(r, qt, N, K)
    xb, xf = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    Y = gpu_qgemm(qt, W, xb, M, K, N)
    rows = np.unique(np.concatenate([np.arange(0, M, 37), [63, 64, 511]]))
    ref = oracle_rows(po, qt, W, xf[rows])
    e = rel_err(Y[rows], ref)
    print(qt, N, K, "rel err", e, flush=True)
    assert e <= QGEMM_TOL
    if qt == 12:
        assert np.array_equal(bits(Y[rows]), bits(ref))
    # linearity in the rows: row m only depends on row m of X (checked on the rows the oracle did not cover)
    perm = r.permutation(M)
    Yp = gpu_qgemm(qt, W, np.ascontiguousarray(xb[perm]), M, K, N)
    assert np.array_equal(bits(Yp), bits(Y[perm]))


def test_qgemm_argument_errors(dev):
    W = torch.zeros(16 * 144, dtype=torch.uint8, device="cuda")
    X = torch.zeros(4 * 256, dtype=torch.int16, device="cuda")
    Y = torch.zeros(4 * 16, device="cuda")
    ws = torch.zeros(ops.qgemm_workspace_bytes(4, 256), dtype=torch.uint8, device="cuda")
    with pytest.raises(PtmError):
        ops.matmul_q(12, W, X, Y, 4, 200, 16, 144, ws)      # K not a multiple of 256
    with pytest.raises(PtmError):
        ops.matmul_q(12, W, X, Y, 4, 256, 16, 100, ws)      # stride shorter than a row
    with pytest.raises(PtmError):
        ops.matmul_q(12, W, X, Y, 0, 256, 16, 144, ws)      # empty M
    with pytest.raises(PtmError):
        ops.matmul_q(13, W, X, Y, 4, 256, 16, 144, ws)      # not a K-quant this path handles


# ---- fast path: fp16 MFMA on dequantised weights -------------------------------------------------------------
QGEMM_F16_TOL = 1e-2   # the prefill path's stated bar: max |y - y_cpu| / rms(y_cpu) against the reference GEMV per row
QGEMM_F16_EXPECT = 5e-3  # what fp16 rounding of both operands should stay under (measured ~1e-3)


def oracle_rows_q8x(po, qt, W, xf):
    """Reference rows.  Q6_K: the reference uses fp32 activations; the fast path rounds them to Q8 values first, so
    its error against the reference's Q6_K GEMV includes that rounding (it is what the reference's Q4_K path does)."""
    return np.stack([po.gemv(qt, W, xf[m]) for m in range(xf.shape[0])])


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 256, 16), (5, 512, 48), (128, 512, 256), (130, 1024, 300), (257, 2560, 334),
                                   (33, 256, 7)])
def test_qgemm_f16_rows_vs_gemv(dev, po, qt, M, K, N):
    r = synth.rng_for(44, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, xf = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    Y = gpu_qgemm_f16(qt, W, xb, M, K, N)
    ref = oracle_rows(po, qt, W, xf)
    e = rel_err(Y, ref)
    print(qt, M, K, N, "rel err", e, flush=True)
    assert np.all(np.isfinite(Y))
    assert e <= (QGEMM_F16_EXPECT if qt == 12 else QGEMM_F16_TOL)


def test_qgemm_f16_large_and_zero_rows(dev, po):
    M, K, N = 20, 512, 64
    r = synth.rng_for(45)
    x = r.standard_normal((M, K), dtype=np.float32)
    x[3] = 0.0
    x[4] *= 1e20      # far beyond fp16: exercised by the per-row power-of-two scale
    x[5] *= 1e-3
    xb, xf = bf16_round(x)
    W = synth.make_weight(r, 12, N, K)
    Y = gpu_qgemm_f16(12, W, xb, M, K, N)
    ref = oracle_rows(po, 12, W, xf)
    assert np.all(np.isfinite(Y)) and np.all(Y[3] == 0.0)
    for m in range(M):
        assert rel_err(Y[m], ref[m]) <= QGEMM_F16_EXPECT, m


@pytest.mark.parametrize("qt,N,K", [(12, 4096, 4096), (12, 1024, 4096), (12, 14336, 4096), (14, 4096, 14336)])
def test_qgemm_f16_llama3_8b_layer_shapes_m512(dev, po, qt, N, K):
    M = 512
    r = synth.rng_for(43, qt, N, K)
    W = synth.make_weight(r, qt, N, K)
    xb, xf = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    Y = gpu_qgemm_f16(qt, W, xb, M, K, N)
    rows = np.unique(np.concatenate([np.arange(0, M, 61), [127, 128, 511]]))
    ref = oracle_rows(po, qt, W, xf[rows])
    e = rel_err(Y[rows], ref)
    fro = float(np.linalg.norm(Y[rows] - ref) / np.linalg.norm(ref))
    print(qt, N, K, "max/rms", e, "frobenius", fro, flush=True)
    assert e <= QGEMM_F16_TOL and fro <= 3e-3
    # against the bit-exact kernel on ALL rows (Q4_K): same bar
    if qt == 12:
        Yx = gpu_qgemm(qt, W, xb, M, K, N)
        assert rel_err(Y, Yx) <= QGEMM_F16_EXPECT


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 512, 127), (31, 2560, 129), (32, 512, 385), (33, 4096, 128), (63, 768, 255), (64, 2560, 641),
                                   (33, 256, 128 * 256 + 1)])
def test_short_prompt_tiles(dev, po, qt, M, K, N):
    """Workgroups of 128 columns (up to 32 rows always, up to 64 where 256 columns leave CUs idle) and the last size's 256: rows are the
    rows of a 65-row call, which no 128-column tile serves, bit for bit (K unsplit: a call without room for partial sums)."""
    r = synth.rng_for(46, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, _ = bf16_round(r.standard_normal((65, K), dtype=np.float32))
    few = gpu_qgemm_f16(qt, W, xb[:M], M, K, N)
    many = gpu_qgemm_f16(qt, W, xb, 65, K, N)
    assert np.array_equal(bits(few), bits(many[:M]))


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 768, 127), (31, 768, 129), (32, 1024, 385), (17, 1024, 1), (8, 768, 4096)])
def test_short_prompts_with_all_blocks_requested_at_once(dev, po, qt, M, K, N):
    """K of three and four super-blocks: rows are the rows of a 65-row call bit for bit."""
    r = synth.rng_for(47, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, _ = bf16_round(r.standard_normal((65, K), dtype=np.float32))
    assert np.array_equal(bits(gpu_qgemm_f16(qt, W, xb[:M], M, K, N)), bits(gpu_qgemm_f16(qt, W, xb, 65, K, N)[:M]))


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(19, 9728, 2560), (32, 14336, 1000), (5, 9728, 2561)])
def test_short_prompts_whose_last_split_is_shorter(dev, po, qt, M, K, N):
    """13 splits of three blocks with two in the last, and others: rows are the rows of a 40-row call, which has the same splits, bit for bit."""
    r = synth.rng_for(48, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    x = torch.from_numpy(r.standard_normal((40, K), dtype=np.float32)).cuda()
    Wd, out = torch.from_numpy(W).cuda(), []
    for m in (M, 40):
        ws = torch.empty(ops.qgemm_f16_f32_workspace_bytes(m, K, N), dtype=torch.uint8, device="cuda")
        y = torch.full((m, N), 3.0, device="cuda")
        ops.matmul_q_f16_f32(qt, Wd, x[:m].contiguous(), y, m, K, N, W.shape[1], ws, accumulate=False)
        out.append(y.cpu().numpy()[:M])
    assert np.array_equal(bits(out[0]), bits(out[1]))


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 256, 129), (32, 256, 127), (19, 512, 1), (31, 512, 385), (19, 1280, 130), (32, 4096, 2560)])
def test_short_prompts_of_one_and_two_blocks(dev, po, qt, M, K, N):
    """Splits of one and of two super-blocks, the last shorter or not: rows are the rows of a 40-row call, which has the same splits, bit for bit."""
    r = synth.rng_for(50, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, _ = bf16_round(r.standard_normal((40, K), dtype=np.float32))
    assert np.array_equal(bits(gpu_qgemm_f16(qt, W, xb[:M], M, K, N)), bits(gpu_qgemm_f16(qt, W, xb, 40, K, N)[:M]))


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(1, 256, 31), (5, 768, 128), (32, 768, 33), (33, 768, 129), (64, 512, 256), (65, 768, 255), (128, 256, 513), (129, 768, 256), (192, 512, 20000),
                                   (257, 768, 6500), (260, 512, 40000)])
def test_sums_onto_what_is_there(dev, po, qt, M, K, N):
    """Every tile height, whole tiles and ones with rows and columns past the edge: added onto Y is what is stored plus Y, bit for bit, and
    nothing behind the last row is written."""
    r = synth.rng_for(51, qt, M, K, N)
    W = torch.from_numpy(synth.make_weight(r, qt, N, K)).cuda()
    x = torch.from_numpy(r.standard_normal((M, K), dtype=np.float32)).cuda()
    old = torch.from_numpy(r.standard_normal((M + 1, N), dtype=np.float32)).cuda()
    ws = torch.empty(ops.qgemm_f16_f32_workspace_bytes(M, K, N), dtype=torch.uint8, device="cuda")
    out = []
    for accumulate in (False, True):
        y = old.clone()
        ops.matmul_q_f16_f32(qt, W, x, y, M, K, N, W.shape[1], ws, accumulate=accumulate)
        assert torch.equal(y[M], old[M])
        out.append(y[:M])
    assert torch.equal(out[1], out[0] + old[:M]) or torch.equal(out[1], old[:M] + out[0])


# super-blocks of the longest split of each matrix; types in file order, K that does not divide evenly among the splits, N off the 128-column tiles
@pytest.mark.parametrize("K,N,types,blocks", [(2560, (4097, 1000, 129), (12, 12, 14), (3, 3, 2)), (2560, (13000, 1000, 515), (14, 12, 12), (3, 4, 4)),
                                              (4096, (13000, 1000, 515), (12, 14, 14), (4, 2, 3)), (4096, (5000, 700), (14, 12), (2, 3)), (2560, (20000, 300), (12, 14), (4, 2)),
                                              (1792, (9728, 9728), (12, 12), (3, 3)), (1024, (1000, 70000), (12, 14), (4, 4))])
def test_short_prompts_of_several_matrices(dev, po, K, N, types, blocks):
    """q / k / v and gate / up of up to 32 rows: unequal K splits and kinds of weights side by side, shorter last splits.  Rows are the rows of a 40-row call, which
    has the same splits and another kernel, bit for bit, as sums and as the slabs that a later launch adds; and the product in 64 bits."""
    import ctypes as C
    from gemm_helpers import harness
    h, n, nblk = harness(), len(N), K // 256
    h.multi_split_bytes.restype = C.c_int64
    Ns, ts, sp = (C.c_int * n)(*N), (C.c_uint32 * n)(*types), (C.c_int * n)()
    h.multi_plan(n, Ns, ts, K, 32, sp)
    assert tuple(-(-nblk // s) for s in sp) == blocks
    r = synth.rng_for(49, K, *N)
    Wh = [synth.make_weight(r, t, rows, K) for t, rows in zip(types, N)]
    W = [torch.from_numpy(w).cuda() for w in Wh]
    gamma = torch.from_numpy((1 + 0.1 * r.standard_normal(K)).astype(np.float32)).cuda()
    X = torch.from_numpy(r.standard_normal((40, K), dtype=np.float32)).cuda()
    ptrs = lambda ts: (C.c_void_p * n)(*[t.data_ptr() for t in ts])
    p = lambda t: C.c_void_p(t.data_ptr())

    def run(M, deferred):
        ws = [torch.zeros(ops.qgemm_f16_workspace_bytes(M, K), dtype=torch.uint8, device="cuda") for _ in range(2)]
        room = h.multi_split_bytes(n, Ns, ts, K, M)
        split = torch.full((max(room // 4, 4),), 5.0, device="cuda")
        Y = [torch.full((M, rows), 3.0, device="cuda") for rows in N]
        P, s = (C.c_void_p * n)(), (C.c_int * n)()
        rc = h.multi_run(n, ts, ptrs(W), (C.c_int64 * n)(*[w.shape[1] for w in Wh]), Ns, ptrs(Y), p(X), p(gamma), M, K, p(ws[0]), p(ws[1]), p(split),
                         C.c_int64(split.numel() * 4), P if deferred else None, s if deferred else None, None)
        assert rc == 0
        torch.cuda.synchronize()
        if not deferred:
            return Y
        out = []
        for i in range(n):
            at = (P[i] - split.data_ptr()) // 4
            out.append(Y[i][None] if s[i] == 1 else split[at:at + s[i] * M * N[i]].reshape(s[i], M, N[i]))
        return out

    many, slabs = run(40, False), run(40, True)
    for M in (1, 19, 32):
        for i, (a, b) in enumerate(zip(run(M, False), many)):
            assert torch.equal(a, b[:M]), (M, i)
        for i, (a, b) in enumerate(zip(run(M, True), slabs)):
            assert torch.equal(a, b[:, :M]), (M, i)
    x = X.double() / (X.double().pow(2).mean(1, keepdim=True) + 1e-6).sqrt() * gamma.double()
    for i, (t, rows) in enumerate(zip(types, N)):
        xt = x
        if t == 12:
            b = x.reshape(40, -1, 32)
            d = b.abs().amax(2, keepdim=True) / 127
            xt = (torch.round(b / d) * d).reshape(40, K)
        want = xt @ torch.from_numpy(po.dequant(t, Wh[i])).cuda().double().reshape(rows, K).T
        err = float((many[i].double() - want).abs().max() / want.pow(2).mean().sqrt())
        print("max err / rms: %.2e" % err, flush=True)
        assert err <= QGEMM_F16_TOL, (i, err)


@pytest.mark.parametrize("K,N,types", [(1024, (1000, 129, 257), (12, 12, 14)), (2560, (4097, 1000), (14, 12)), (256, (300, 300), (12, 12))])
def test_several_matrices_in_128_columns_and_several_row_tiles(dev, po, K, N, types):
    """65 to 128 rows in workgroups of 64 rows and 128 columns: their first 40 rows are those of a 40-row call, which has the same splits, bit for
    bit, and so are rows 64 on of those of a call of them alone."""
    import ctypes as C
    from gemm_helpers import harness
    h, n = harness(), len(N)
    h.multi_split_bytes.restype = C.c_int64
    Ns, ts = (C.c_int * n)(*N), (C.c_uint32 * n)(*types)
    r = synth.rng_for(52, K, *N)
    W = [torch.from_numpy(synth.make_weight(r, t, rows, K)).cuda() for t, rows in zip(types, N)]
    gamma = torch.from_numpy((1 + 0.1 * r.standard_normal(K)).astype(np.float32)).cuda()
    X = torch.from_numpy(r.standard_normal((128, K), dtype=np.float32)).cuda()
    ptrs = lambda ts: (C.c_void_p * n)(*[t.data_ptr() for t in ts])
    p = lambda t: C.c_void_p(t.data_ptr())

    def run(x):
        M = x.shape[0]
        ws = [torch.zeros(ops.qgemm_f16_workspace_bytes(M, K), dtype=torch.uint8, device="cuda") for _ in range(2)]
        split = torch.full((max(h.multi_split_bytes(n, Ns, ts, K, M) // 4, 4),), 5.0, device="cuda")
        Y = [torch.full((M + 1, rows), 3.0, device="cuda") for rows in N]
        assert h.multi_run(n, ts, ptrs(W), (C.c_int64 * n)(*[w.shape[1] for w in W]), Ns, ptrs(Y), p(x), p(gamma), M, K, p(ws[0]), p(ws[1]), p(split),
                           C.c_int64(split.numel() * 4), None, None, None) == 0
        torch.cuda.synchronize()
        assert all(bool((y[M] == 3.0).all()) for y in Y)
        return [y[:M] for y in Y]

    few = run(X[:40].contiguous())
    for M in (65, 100, 128):
        tail = run(X[64:M].contiguous())
        for i, y in enumerate(run(X[:M].contiguous())):
            assert torch.equal(y[:40], few[i]), (M, i)
            assert torch.equal(y[64:], tail[i]), (M, i)


@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(65, 768, 257), (128, 2560, 1000), (127, 9728, 129)])
def test_128_columns_and_several_row_tiles(dev, po, qt, M, K, N):
    """65 to 128 rows in workgroups of 64 rows and 128 columns: rows are those of a 40-row call, which has the same splits, bit for bit."""
    r = synth.rng_for(53, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, _ = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    y = gpu_qgemm_f16(qt, W, xb, M, K, N)
    assert np.array_equal(bits(y[:40]), bits(gpu_qgemm_f16(qt, W, xb[:40], 40, K, N)))
    assert np.array_equal(bits(y[64:]), bits(gpu_qgemm_f16(qt, W, xb[64:], M - 64, K, N)))


@pytest.mark.parametrize("M,K,N", [(257, 1024, 8449), (320, 2560, 9728), (321, 1280, 10751), (384, 1024, 10752), (385, 1024, 9000), (300, 4096, 8200), (300, 4352, 8200), (300, 768, 9000),
                                   (300, 1024, 8192), (190, 1024, 13001)])
def test_64_rows_of_256_columns_in_several_row_tiles(dev, po, M, K, N):
    """Q4_K products in one split, and beside the rule for these tiles: rows are those of calls of 64 rows, which have 128 columns, bit for bit."""
    r = synth.rng_for(54, M, K, N)
    W = synth.make_weight(r, 12, N, K)
    xb, _ = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    y = gpu_qgemm_f16(12, W, xb, M, K, N)
    for m in (0, 64, 100, M - 64):
        assert np.array_equal(bits(y[m:m + 64]), bits(gpu_qgemm_f16(12, W, np.ascontiguousarray(xb[m:m + 64]), 64, K, N))), m


# tiles of 256 rows: all (236 pairs of row tiles), whole rounds and 128-row tiles behind them (K splits off and on), an odd last row tile, ragged N; of 192
# rows: 3 and 2 row tiles, whole and ragged, one of 129 rows
@pytest.mark.parametrize("qt", [12, 14])
@pytest.mark.parametrize("M,K,N", [(509, 512, 19456), (385, 256, 38000), (953, 512, 19441), (1030, 256, 19456), (2047, 256, 9728), (641, 1024, 14337), (510, 512, 30001), (384, 256, 28672),
                                   (129, 512, 65000), (192, 768, 40001), (576, 256, 19456)])
def test_tiles_of_256_rows(dev, po, qt, M, K, N):
    """Rows are the rows of calls of 128 rows, which have tiles of 128, bit for bit (K unsplit)."""
    r = synth.rng_for(50, qt, M, K, N)
    W = synth.make_weight(r, qt, N, K)
    xb, _ = bf16_round(r.standard_normal((M, K), dtype=np.float32))
    y = gpu_qgemm_f16(qt, W, xb, M, K, N)
    for m in list(range(0, M - 127, 384)) + [M - 128]:
        assert np.array_equal(bits(y[m:m + 128]), bits(gpu_qgemm_f16(qt, W, np.ascontiguousarray(xb[m:m + 128]), 128, K, N))), m


@pytest.mark.parametrize("K,N,types,M", [(512, (9728, 9728), (12, 12), 509), (512, (5000, 5001, 5100), (12, 14, 14), 1000), (1024, (4096, 1024, 1000), (12, 12, 14), 2048),
                                         (512, (14336, 14300), (14, 12), 2000)])
def test_tiles_of_256_rows_of_several_matrices(dev, po, K, N, types, M):
    """Slabs and sums are those of calls of fewer rows of the same class (same K splits) in tiles of 128, bit for bit."""
    import ctypes as C
    from gemm_helpers import harness
    h, n, few = harness(), len(N), 260 if M <= 1024 else 1025
    h.multi_split_bytes.restype = C.c_int64
    Ns, ts = (C.c_int * n)(*N), (C.c_uint32 * n)(*types)
    r = synth.rng_for(51, K, *N)
    Wh = [synth.make_weight(r, t, rows, K) for t, rows in zip(types, N)]
    W = [torch.from_numpy(w).cuda() for w in Wh]
    gamma = torch.from_numpy((1 + 0.1 * r.standard_normal(K)).astype(np.float32)).cuda()
    X = torch.from_numpy(r.standard_normal((M, K), dtype=np.float32)).cuda()
    ptrs = lambda ts: (C.c_void_p * n)(*[t.data_ptr() for t in ts])
    p = lambda t: C.c_void_p(t.data_ptr())

    def run(x):
        m = x.shape[0]
        ws = [torch.zeros(ops.qgemm_f16_workspace_bytes(m, K), dtype=torch.uint8, device="cuda") for _ in range(2)]
        split = torch.full((max(h.multi_split_bytes(n, Ns, ts, K, m) // 4, 4),), 5.0, device="cuda")
        Y = [torch.full((m, rows), 3.0, device="cuda") for rows in N]
        assert h.multi_run(n, ts, ptrs(W), (C.c_int64 * n)(*[w.shape[1] for w in Wh]), Ns, ptrs(Y), p(x), p(gamma), m, K, p(ws[0]), p(ws[1]), p(split),
                           C.c_int64(split.numel() * 4), None, None, None) == 0
        torch.cuda.synchronize()
        return Y

    y = run(X)
    for m in (0, M - few):
        for i, (a, b) in enumerate(zip(run(X[m:m + few].contiguous()), y)):
            assert torch.equal(a, b[m:m + few]), (m, i)
