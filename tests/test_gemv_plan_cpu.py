"""CPU: which kernel takes a product of few long rows, where two of them could."""
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
