"""Prompt products of more than 64 rows: every kind of tile, alone and beside others in one launch, at the edges of rows, columns and K."""
import numpy as np
import pytest
import torch

from folder_helpers import errors, portions
from nadozen_models import model as nadozen, parallel, wkv
from tovasun_models import attention, latent, layer, model as tovasun
from oracle import nadozen_oracle, tovasun_oracle
from prometorch_amd import _lib, model as registry
from prometorch_amd.testing import folder_writer as fw

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available()
    return _lib.load()


# rows and columns around multiples of 64, 128, 192 and 256; launches of a few tiles, of one round of the chip and a little more, of several
# rounds with columns and rows left over; K of one step, of two, of many, and not whole
@pytest.mark.parametrize("M,N,K", [(65, 64, 64), (65, 1, 8), (128, 129, 65), (129, 257, 128), (191, 320, 200), (255, 512, 64), (257, 700, 192), (64 * 7, 6000, 64),
                                   (512, 2560, 1030), (513, 9728, 130), (1030, 9728, 64), (1030, 6144, 128), (1100, 2560, 4096), (2048, 8200, 64),
                                   (2047, 19456, 64), (3001, 5000, 320), (70, 33000, 64)])
def test_tiles(dev, M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K)
    kp = (K + 63) // 64 * 64
    A, W = (torch.zeros(n, kp, dtype=torch.bfloat16, device="cuda") for n in (M, N))
    A[:, :K], W[:, :K] = torch.randn(M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g)
    ldc = N + (M & 3)  # whole and broken 16-byte rows
    C = torch.full((M + 1, ldc), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _lib.check(dev.ptm_dense_gemm(A.data_ptr(), 0, kp, W.data_ptr(), kp, C.data_ptr(), ldc, M, N, K, None), "dense_gemm")
    torch.cuda.synchronize()
    assert torch.isnan(C[M]).all() and torch.isnan(C[:M, N:]).all()
    want = A.double() @ W.double().T
    # products are exact in fp32, a sum of K of them in any order is off by at most K units in the last place of the sum of sizes
    bound = (A.double().abs() @ W.double().abs().T) * (K * 2.0 ** -24) + 1e-30
    assert ((C[:M, :N].double() - want).abs() <= bound).all()


# rows so far apart that the last of 64 lies 4 GiB and more behind the first, on either side; the longest rows that tiles take, and the next
@pytest.mark.parametrize("lda,ldw", [(36 << 20, 128), (128, 36 << 20), (1 << 22, 1 << 22), ((1 << 22) + 8, 1 << 22)])
def test_rows_far_apart(dev, lda, ldw):
    M, N, K = 130, 140, 100
    g = torch.Generator(device="cuda").manual_seed(9)
    rows = {}
    for name, n, ld in (("A", M, lda), ("W", N, ldw)):
        flat = torch.empty((n - 1) * ld + 128, dtype=torch.bfloat16, device="cuda")
        rows[name] = flat.as_strided((n, 128), (ld, 1))
        rows[name].copy_(torch.randn(n, 128, device="cuda", generator=g))
        rows[name][:, K:] = 0
    C = torch.full((M, N), float("nan"), device="cuda")
    torch.cuda.synchronize()
    _lib.check(dev.ptm_dense_gemm(rows["A"].data_ptr(), 0, lda, rows["W"].data_ptr(), ldw, C.data_ptr(), N, M, N, K, None), "dense_gemm")
    torch.cuda.synchronize()
    a, w = rows["A"].double(), rows["W"].double()
    bound = (a.abs() @ w.abs().T) * (K * 2.0 ** -24) + 1e-30  # as above
    assert ((C.double() - a @ w.T).abs() <= bound).all()


# the results that are not plain sums (squared ReLU, gated SiLU, decays, 16-bit rows, sections of one product) and their odd sizes
@pytest.mark.parametrize("design", ["tovasun", "nadozen"])
def test_prompts_of_many_rows(dev, tmp_path, design):
    if design == "tovasun":
        cfg = tovasun([layer(latent(3, 40, 8, 72, 36, window=50, sharp=1.0), 333), layer(attention(6, 2, 40, 24, rot=10, window=70, keep=3, sharp=1.0), 200)], 136, 101, side=11)
        oracle = tovasun_oracle
    else:
        cfg = nadozen([wkv(4, 64, 33, ff=333), parallel(6, 2, 40, 60, (4, 33, 32, 2, 3, 4), ff=130, sharp=1.0)], 256, 101, 2)
        oracle = nadozen_oracle
    weights = fw.random_weights(cfg, 5)
    m = registry.load(fw.write_model_folder(str(tmp_path / "m"), cfg, weights), max_seq=320)
    tokens = [int(t) for t in np.random.default_rng(3).integers(0, 101, 300)]
    want = oracle.logits(tokens, weights, cfg)
    for sizes in ([300], [129, 171], [67]):
        e = errors(portions(m, tokens, sizes), want)
        # bfloat16 rows and caches: the bars of the two models' own tests
        assert e.mean() < 0.02 and np.percentile(e, 97) < 0.1, (sizes, e.mean(), e.max())
    m.close()
