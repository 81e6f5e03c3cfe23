"""Prompt products of more than 64 rows: every kind of tile, alone and beside others in one launch, at the edges of rows, columns and K."""
import ctypes as C

import numpy as np
import pytest
import torch

from folder_helpers import errors, portions
from gemm_helpers import DECAY, ELEM, F32, RELU2, SWIGLU, Call, harness
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


def check_product(M, N, K, epilogue=F32, section=0, slabs=0, pad=0, ldw=0):
    """One product as the block decoders' runtime calls it against 64 bits; how many K splits it took."""
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N * 3 + K + epilogue)
    kp, S = (K + 63) // 64 * 64, N // section if section else 1
    A = torch.zeros(S, M, kp, dtype=torch.bfloat16, device="cuda")
    ldw = ldw or kp
    W = torch.empty((N - 1) * ldw + kp, dtype=torch.bfloat16, device="cuda").as_strided((N, kp), (ldw, 1))
    W[:, K:] = 0
    A[..., :K], W[:, :K] = torch.randn(S, M, K, device="cuda", generator=g), torch.randn(N, K, device="cuda", generator=g) * K ** -0.5
    cols = N // 2 if epilogue == SWIGLU else N
    ldc, bias = cols + pad, torch.randn(N, device="cuda", generator=g) - 1
    out = torch.full((max(1, slabs), M, ldc), float("nan"), device="cuda", dtype=torch.float32 if epilogue in (F32, DECAY) else torch.bfloat16)
    c = Call(A=A.data_ptr(), W=W.data_ptr(), C=out.data_ptr(), bias=bias.data_ptr(), lda=kp, ldw=ldw, ldc=ldc, section_a=M * kp, slab=M * ldc,
             slab_room=M * ldc * slabs, M=M, N=N, K=K, epilogue=epilogue, section_n=section, may_split=int(slabs > 0))
    splits = C.c_int32()
    torch.cuda.synchronize()
    _lib.check(harness().gemm_run(C.byref(c), C.byref(splits), None), "gemm_run")
    torch.cuda.synchronize()
    splits = splits.value
    assert splits <= max(1, slabs) and torch.isnan(out[:splits, :, cols:]).all() and torch.isnan(out[splits:]).all()
    got = out[:splits, :, :cols].double().sum(0)
    v, off = [], []  # the products, and how far sums of K of them in any order can be from them (as above; partial sums are added exactly here)
    for i in range(S):
        a, w = A[i].double(), W[i * (N // S):(i + 1) * (N // S)].double()
        v.append(a @ w.T)
        off.append(a.abs() @ w.abs().T * (K * 2.0 ** -24) + 1e-30)
    v, off = torch.cat(v, 1), torch.cat(off, 1)
    half = 2.0 ** -8  # bfloat16 has 8 significant bits: half of its last place is 2^-8 of the value, or less
    if epilogue == F32:
        want, bound = v, off
    elif epilogue == ELEM:
        want, bound = v, off + (v.abs() + off) * half
    elif epilogue == RELU2:
        want = v.clamp(min=0) ** 2
        slack = 2 * v.abs() * off + off ** 2 + want * 2.0 ** -23
        bound = slack + (want + slack) * half
    elif epilogue == SWIGLU:  # |silu'| < 1.1; exponential, division and two products in 32 bits: 2^-20 of the result
        (gate, up), (og, ou) = v.split(N // 2, 1), off.split(N // 2, 1)
        want = gate / (1 + torch.exp(-gate)) * up
        slack = 1.1 * og * (up.abs() + ou) + gate.abs() * ou + want.abs() * 2.0 ** -20
        bound = slack + (want.abs() + slack) * half
    else:  # the derivative of exp(-exp(v)) is at most 1 / e; each exponential 2^-22 off, the inner one times x exp(-x) <= 1 / e
        want, bound = torch.exp(-torch.exp(v + bias.double())), 0.4 * (off + 2.0 ** -23 * (v.abs() + bias.double().abs())) + 2.0 ** -21
    assert ((got - want).abs() <= bound).all(), float(((got - want).abs() / bound).max())
    return splits


# up to 64 rows in tiles of 32 x 32 and a step: one, fewer steps than waves, steps that are no multiple of the waves, K split, sections, every epilogue,
# and the last output that these tiles take with the first that they do not
@pytest.mark.parametrize("M,N,K,epilogue,section,slabs", [
    (1, 1, 8, F32, 0, 0), (1, 32, 64, ELEM, 0, 0), (31, 257, 100, F32, 0, 0), (32, 64, 576, RELU2, 0, 0), (33, 65, 320, DECAY, 0, 0), (64, 96, 1030, SWIGLU, 0, 0),
    (17, 90, 200, SWIGLU, 0, 0), (30, 512, 2560, F32, 128, 0), (64, 40, 9728, F32, 0, 16), (30, 2560, 1536, F32, 0, 16), (32, 40960, 64, F32, 0, 0),
    (32, 40961, 64, F32, 0, 0), (64, 20480, 192, ELEM, 0, 0), (64, 20481, 192, ELEM, 0, 0)])
def test_few_rows(dev, M, N, K, epilogue, section, slabs):
    check_product(M, N, K, epilogue, section, slabs)


# outputs of more tiles than that, in tiles of 32 x 128 and 64 x 64: gated, with a bias, sections, steps of K with a rest
@pytest.mark.parametrize("M,N,K,epilogue,section", [(33, 28672, 330, SWIGLU, 0), (64, 28672, 330, SWIGLU, 0), (19, 41002, 330, SWIGLU, 0), (32, 41000, 200, DECAY, 0),
                                                    (1, 41001, 130, F32, 0), (40, 24001, 200, RELU2, 0), (30, 49152, 330, F32, 16384), (50, 24576, 330, ELEM, 8192)])
def test_few_rows_of_wide_outputs(dev, M, N, K, epilogue, section):
    check_product(M, N, K, epilogue, section)


# gates and ups just under and over 2 GiB apart, and 4.6 GiB
@pytest.mark.parametrize("ldw", [558656, 558664, 1200000])
def test_ups_far_from_their_gates(dev, ldw):
    check_product(1041, 3844, 64, SWIGLU, ldw=ldw)


# outputs of few tiles (64 x 64, four waves each): one, all 256 of a round and a little more, split, and every kind of result
FEW = [(65, 64, 64, F32, 0, 0, 0), (1024, 1024, 100, F32, 0, 0, 3), (1030, 1024, 128, ELEM, 0, 0, 0), (255, 4090, 1000, F32, 0, 0, 2), (129, 1023, 1030, F32, 0, 16, 1),
       (128, 512, 2816, F32, 0, 16, 0), (97, 1500, 320, ELEM, 0, 0, 4), (200, 1001, 640, RELU2, 0, 0, 7), (130, 2022, 1024, SWIGLU, 0, 0, 5), (300, 999, 64, DECAY, 0, 0, 1),
       (150, 1024, 256, F32, 256, 0, 0)]


@pytest.mark.parametrize("case", FEW, ids=str)
def test_few_tiles(dev, case):
    assert check_product(*case) > 1 or not case[5]


# (rows, columns, K, result, section, partial sums): each kind of tile alone with each kind of result, two and three kinds in a launch with
# columns or rows left over, sections, K splits; tests/test_gemm_plan_cpu.py holds the list against the plans
LARGE = [(1158, 9988, 72, F32, 0, 0), (555, 13646, 61, F32, 0, 0), (389, 13212, 71, F32, 0, 16), (266, 13268, 64, F32, 0, 16), (133, 11662, 65, F32, 0, 0), (75, 8204, 141, F32, 0, 0),
         (1472, 8616, 60, ELEM, 0, 0), (515, 13976, 67, ELEM, 0, 0), (464, 12394, 74, ELEM, 0, 0), (259, 13920, 73, ELEM, 0, 0), (257, 6690, 91, ELEM, 0, 0), (67, 8376, 176, ELEM, 0, 0),
         (1333, 9462, 79, RELU2, 0, 0), (680, 10786, 61, RELU2, 0, 0), (514, 10650, 64, RELU2, 0, 0), (385, 9742, 71, RELU2, 0, 0), (229, 8348, 80, RELU2, 0, 0), (72, 9262, 145, RELU2, 0, 0),
         (1370, 8996, 69, SWIGLU, 0, 0), (529, 13306, 63, SWIGLU, 0, 0), (393, 13092, 85, SWIGLU, 0, 0), (1041, 3844, 64, SWIGLU, 0, 0), (131, 12082, 98, SWIGLU, 0, 0), (79, 8604, 149, SWIGLU, 0, 0),
         (1170, 10054, 89, DECAY, 0, 0), (678, 11300, 72, DECAY, 0, 0), (441, 13136, 63, DECAY, 0, 0), (286, 13490, 62, DECAY, 0, 0), (138, 11264, 73, DECAY, 0, 0), (75, 8672, 147, DECAY, 0, 0),
         (1343, 8192, 79, F32, 2048, 0), (1355, 4608, 83, F32, 1152, 0), (592, 7168, 78, F32, 1792, 0), (406, 10752, 63, F32, 2688, 0), (1468, 11264, 115, F32, 2816, 0), (80, 9216, 150, F32, 2304, 0),
         (1488, 13894, 124, ELEM, 0, 0), (1468, 12982, 446, SWIGLU, 0, 0), (1175, 13112, 146, RELU2, 0, 0), (1426, 12016, 275, DECAY, 0, 0), (1364, 12288, 357, F32, 3072, 0),
         (1059, 13522, 97, ELEM, 0, 0), (843, 12602, 69, SWIGLU, 0, 0), (1103, 10638, 147, RELU2, 0, 0), (1356, 8318, 135, DECAY, 0, 0), (1299, 10800, 266, F32, 0, 0), (1132, 10752, 114, F32, 2688, 0),
         (1325, 13874, 81, ELEM, 0, 0), (1310, 11976, 118, SWIGLU, 0, 0), (1192, 8192, 89, F32, 2048, 0), (1030, 9728, 1000, ELEM, 0, 0), (513, 19458, 500, SWIGLU, 0, 0),
         (71, 11412, 3312, F32, 0, 16), (68, 9600, 1997, F32, 0, 16), (141, 5788, 2340, F32, 0, 16), (71, 3502, 1168, F32, 0, 16), (138, 13930, 3795, F32, 0, 16)]


@pytest.mark.parametrize("i,case", list(enumerate(LARGE)), ids=lambda v: str(v) if isinstance(v, tuple) else "")
def test_kinds_and_regions(dev, i, case):
    check_product(*case, pad=i % 8)


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
