"""CPU: which tiles cover a prompt product of more than 64 rows, and where a launch of 64 x 64 tiles of four waves takes it instead."""
import ctypes
import random

import pytest

from gemm_helpers import DECAY, ELEM, F32, RELU2, SWIGLU, TILES, harness, plan
from test_gpu_gemm_tiles import LARGE


# outputs of few tiles: up to 256 of 64 x 64, up to 512 where K is short; split, tiles x splits
@pytest.mark.parametrize("M,N,K,slabs,splits", [(65, 64, 64, 0, 1), (128, 1024, 1024, 0, 1), (300, 2560, 2560, 0, 1), (256, 4096, 2560, 0, 1), (129, 2560, 9728, 0, 1),
                                                (1500, 64, 2560, 0, 1), (1030, 1024, 128, 0, 1), (128, 1024, 1024, 16, 4), (128, 512, 1024, 16, 4)])
def test_few_tiles_are_four_waves_each(M, N, K, slabs, splits):
    got = plan(M, N, K, slabs=slabs)
    assert got == (splits, (M + 63) // 64 * ((N + 63) // 64) * splits, [])


@pytest.mark.parametrize("M,N,K,slabs", [(512, 2560, 2560, 0), (300, 5000, 320, 0), (2048, 2560, 1024, 0), (65, 2560, 9728, 16), (1030, 9728, 64, 0)])
def test_more_tiles_are_not(M, N, K, slabs):
    assert plan(M, N, K, slabs=slabs)[2]


@pytest.mark.parametrize("M,N,K,epilogue,kinds", [(1500, 16384, 64, F32, 1), (700, 32768, 256, F32, 1), (700, 32768, 257, F32, 2), (1500, 16384, 64, ELEM, 2), (648, 8320, 64, F32, 2),
                                                  (2048, 19456, 2560, F32, 2)])
def test_large_32_bit_results_of_short_products_are_of_one_kind(M, N, K, epilogue, kinds):
    assert len({r[0] for r in plan(M, N, K, epilogue)[2]}) == kinds


def test_rows_far_apart_are_four_waves_each():
    """A tile's offsets are 32 bits; K of 2^22 + 8 values makes rows longer than the longest they take."""
    assert plan(1000, 5000, (1 << 22) + 8)[2] == [] and plan(1000, 5000, 1 << 22)[2]


def test_plans_cover_each_output():
    r = random.Random(4)
    for _ in range(4000):
        M, N, K = r.randint(65, 3000), r.randint(1, 20000), r.randint(1, 10000)
        epilogue, section, slabs = r.choice([(F32, 0, 16), (F32, 0, 0), (ELEM, 0, 0), (SWIGLU, 0, 0), (DECAY, 0, 0), (F32, 1, 0)])
        if section:
            section = 128 * r.randint(1, 40)
            N = 4 * section
        N += N & 1
        cols = (N // 2 + 15) // 16 * 32 if epilogue == SWIGLU else N
        splits, wgs, regions = plan(M, N, K, epilogue, section, slabs)
        assert 1 <= splits <= max(1, slabs) and (splits == 1 or splits * 4 <= (K + 63) // 64)
        at, covered = 0, {}
        for kind, first, m0, n0, n1, tm, tn in regions:
            bm, bn = TILES[kind]
            assert first == at and tm > 0 and tn > 0 and m0 % 32 == n0 % 32 == 0
            assert not section or (section % bn == 0 and n0 % bn == 0)
            at += tm * tn * splits
            m1, n1 = min(M, m0 + tm * bm), min(n1, n0 + tn * bn, cols)
            for n in list(range(n0, n1, 32)):
                covered.setdefault(n, []).append((m0, m1))
        assert not regions or at == wgs
        for n in range(0, cols, 32) if regions else ():
            end = 0
            for lo, hi in sorted(covered[n]):
                assert lo <= end, (M, N, K, n)
                end = max(end, hi)
            assert end == M, (M, N, K, n)


def test_the_gpu_cases_reach_every_kind_of_tile_and_region():
    alone, rows, columns, splits = set(), set(), set(), set()
    for M, N, K, epilogue, section, slabs in LARGE:
        n, _, regions = plan(M, N, K, epilogue, section, slabs)
        kinds = [r[0] for r in regions]
        assert kinds, (M, N, K)
        if len(kinds) == 1:
            alone.add((kinds[0], epilogue, section > 0))
        rows |= {(epilogue, section > 0) for r in regions if r[2] > 0}
        columns |= {(epilogue, section > 0) for r in regions if r[3] > 0}
        splits |= {(k, len(kinds) > 1) for k in kinds if n > 1}
    kinds = {0, 1, 2, 3, 4, 6}  # (64 rows of 256 columns are best where something is left over, or in sections)
    assert alone >= {(k, e, False) for k in kinds for e in (F32, ELEM, RELU2, SWIGLU, DECAY)} and (5, F32, True) in alone
    assert rows >= {(e, False) for e in (F32, ELEM, RELU2, SWIGLU, DECAY)} | {(F32, True)}
    assert columns >= {(e, False) for e in (ELEM, RELU2, SWIGLU, DECAY)} | {(F32, True)}
    assert splits >= {(3, False), (4, False), (6, False), (5, True)}
    assert max(len(plan(*c)[2]) for c in LARGE) == 3


def test_slabs_of_a_qknorm_batch():
    """A batch takes no more slabs than leave all of a launch's waves on the chip (1024 SIMDs with 2 / 4 / 7 waves of eight / four / two slabs), and never
    fetches a slab twice over where a smaller batch has them all."""
    h = harness()
    h.qk_rows_batch.argtypes = [ctypes.c_int, ctypes.c_int64]
    for most in range(1, 17):
        for waves in (1, 2048, 2049, 4096, 4097, 7168, 7169, 20480, 1 << 33):
            b = h.qk_rows_batch(most, waves)
            assert b in (1, 2, 4, 8) and (b == 1 or waves <= {8: 2048, 4: 4096, 2: 7168}[b]) and b < 2 * most
    assert [h.qk_rows_batch(m, 190) for m in (1, 2, 3, 4, 5, 16)] == [1, 2, 4, 4, 8, 8]
    assert [h.qk_rows_batch(5, w) for w in (2048, 2049, 4096, 4097)] == [8, 4, 4, 1]


# ---- prompt attention -----------------------------------------------------------------------------
@pytest.mark.parametrize("dq,dv,resident", [(64, 64, 2), (128, 64, 2), (104, 128, 2), (192, 128, 2), (128, 200, 1), (200, 128, 1), (256, 256, 1)])
@pytest.mark.parametrize("heads,blocks", [(8, 16), (8, 33), (8, 50), (8, 64), (4, 128), (8, 65), (4, 200)])
def test_row_blocks_that_take_long_do_not_come_last(dq, dv, resident, heads, blocks):
    """Row block i of a causal prompt takes about i + 1 turns.  `resident` workgroups share a CU, which then takes as long as both together; 256 CUs take the
    workgroups in the order of their ids.  None is left out, and the launch is no longer than with the longest first."""
    h, grid = harness(), heads * blocks
    got = [h.attention_order(dq, dv, i, grid) for i in range(grid)]
    assert sorted(got) == list(range(grid))

    def lasts(order):
        cus = [[] for _ in range(256)]  # what is left of a CU's workgroups
        todo, t = [blocks - o // heads for o in order], 0
        for s in range(resident):
            for cu in cus:
                if todo:
                    cu.append(todo.pop(0))
        while any(cus):
            step = min(min(cu) * len(cu) for cu in cus if cu)
            t += step
            for cu in cus:
                n = len(cu)
                for i in range(n - 1, -1, -1):
                    cu[i] -= step / n
                    if cu[i] < 1e-9:
                        del cu[i]
                        if todo:
                            cu.append(todo.pop(0))
        return t

    assert lasts(got) <= lasts(range(grid)) + 1e-6


@pytest.mark.parametrize("rows", [1, 32, 33, 64, 65, 128, 129, 256, 300, 2048])
def test_several_quantised_matrices_fit_one_round(rows):
    """All (column tile, K split) slots of a launch of several matrices in one round of the chip over the row tiles of the rows' class, but for the one split a
    matrix has at least: a split more leaves CUs with two workgroups of half the blocks, and adds its partial sums."""
    h, r = harness(), random.Random(5)
    of_class = 1 if rows <= 128 else 2 if rows <= 256 else 4 if rows <= 1024 else 8
    shapes = [((24576, 24576), 2048), ((22016, 22016), 4096), ((28672, 28672), 8192), ((9728, 9728), 2560), ((4096, 1024, 1024), 2560)]
    shapes += [(tuple(256 * r.randint(1, 120) - r.randint(0, 255) for _ in range(r.randint(1, 3))), 256 * r.randint(1, 64)) for _ in range(300)]
    for N, K in shapes:
        n = len(N)
        types = [r.choice([12, 14]) for _ in N]
        sp = (ctypes.c_int * n)()
        h.multi_plan(n, (ctypes.c_int * n)(*N), (ctypes.c_uint32 * n)(*types), K, rows, sp)
        tiles = [-(-x // 256) for x in N]
        assert sum(t * s for t, s in zip(tiles, sp)) <= max(256 // of_class, sum(tiles)), (N, K, list(sp))
        assert all(1 <= s <= max(1, min(16 if of_class == 1 else 8, K // 512)) for s in sp)
