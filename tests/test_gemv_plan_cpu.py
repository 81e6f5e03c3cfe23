"""CPU: which kernel takes a product of few long rows, or a step's attention, where two of them could."""
import pytest

from gemm_helpers import harness


def _waves(N):
    rows = -(-N // 256)
    return rows if rows <= 16 else -(-rows // 2)


@pytest.mark.parametrize("N,K,in_order", [(512, 4096, 0), (768, 6144, 0), (768, 20480, 0), (1024, 6144, 1), (769, 4096, 1), (2816, 4096, 1), (2817, 4096, 0), (4096, 4096, 0),
                                          (4096, 4352, 1), (4097, 4096, 0), (6144, 4096, 0), (6145, 4096, 1), (8192, 4096, 1), (2560, 9728, 1), (8192, 14336, 1)])
def test_q4k_long_rows(N, K, in_order):
    """Sides of the lines as they were measured: few waves, and rows of 4096 values in the largest workgroups, go in passes."""
    assert harness().q4k_rows_in_order(N, K, _waves(N)) == in_order


@pytest.mark.parametrize("N,K,stored,added", [(1536, 256, 6, 6), (1537, 256, 0, 0), (4096, 512, 0, 0), (3072, 768, 12, 12), (3073, 1024, 0, 0), (4096, 1280, 16, 16), (1, 2048, 2, 2),
                                              (4096, 2560, 0, 0), (3584, 2560, 0, 14), (1280, 2304, 5, 5), (1536, 3840, 6, 6), (1537, 2816, 0, 7), (2816, 3328, 11, 11), (2817, 3840, 0, 12),
                                              (4096, 4352, 0, 0), (3841, 5120, 0, 0), (3840, 4608, 15, 15), (4096, 5376, 16, 16), (4096, 3584, 0, 16),
                                              (3073, 4096, 13, 13), (3072, 4096, 0, 12), (2560, 9728, 10, 10), (3072, 8192, 0, 12), (3073, 6400, 13, 13), (2816, 14336, 11, 11),
                                              (3072, 13312, 0, 12), (4096, 14336, 16, 16), (4096, 16384, 0, 16), (4097, 2304, 0, 0), (2560, 20736, 0, 0)])
def test_q6k_rows_a_wave(N, K, stored, added):
    """Waves of the kernel with a row per wave, 0 where the ones before it are faster: sides of the lines as they were measured."""
    h = harness()
    assert (h.q6k_rows_waves(N, K, 0), h.q6k_rows_waves(N, K, 1)) == (stored, added)


@pytest.mark.parametrize("dim,heads,kv_heads,room,five", [(128, 32, 8, 2048, 0), (128, 32, 8, 2112, 0), (128, 32, 8, 2113, 1), (128, 32, 8, 2560, 1), (128, 32, 8, 2561, 0), (128, 8, 8, 2304, 0),
                                                          (128, 40, 10, 1664, 0), (128, 40, 10, 1700, 1), (128, 32, 16, 1025, 1), (128, 32, 32, 600, 0), (128, 64, 32, 600, 1),
                                                          (64, 32, 8, 2304, 0), (128, 20, 5, 4096, 0), (128, 20, 5, 4080, 1), (128, 32, 4, 4096, 0), (128, 32, 8, 1 << 30, 0)])
def test_attention_in_chunks_of_80(dim, heads, kv_heads, room, five):
    """Sides of the lines as they were measured over the positions of a cache: not for a few workgroups more than CUs, nor for one query head a kv head."""
    assert harness().attn_five_waves(dim, heads, kv_heads, room) == five
