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
