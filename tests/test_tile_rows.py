"""How many rows of x the tile products take before the library does (ops/kernels.py), on a chip of 256 compute units."""
import pytest

from pytriton_llama_amd import ops


@pytest.mark.parametrize("N,K,most", [(768, 768, 768), (1024, 1024, 768), (1536, 1536, 768), (2048, 2048, 768),
                                      (3072, 3072, 768), (4096, 4096, 640), (5120, 5120, 512), (768, 2048, 768),
                                      (1024, 2816, 768), (1024, 4096, 1088), (2048, 8192, 1088), (3072, 8192, 1088),
                                      (4096, 14336, 1088), (5120, 13824, 870), (8192, 28672, 544)])
def test_products_with_the_norm_behind_them(N, K, most):
    """In a step of more rows than that, the tiles were slower than the library's product and the norm."""
    assert ops.tile_most_rows_sums(N, K) == most


@pytest.mark.parametrize("I,K,most", [(1408, 512, 576), (4096, 1024, 576), (5632, 2048, 576), (8192, 2048, 448), (8192, 3072, 448),
                                      (8960, 1536, 432), (10240, 2560, 432), (12288, 2048, 288), (16384, 1024, 288),
                                      (14336, 2048, 96), (14336, 4096, 96), (28672, 8192, 96), (40000, 512, 0)])
def test_gate_up(I, K, most):
    """As for the sums; and as long as the largest tiles lie on the chip at once."""
    assert ops.tile_most_rows_gate_up(2 * I, K, 256) == most


@pytest.mark.parametrize("rows_w,most", [(3072, 2048), (5120, 1228), (6144, 1024), (98304, 64)])
def test_qkv(rows_w, most):
    """As long as tiles of 128 x 192 lie on the chip at once."""
    assert ops.tile_most_rows_qkv(rows_w, 256) == most


@pytest.mark.parametrize("I,K,least", [(8192, 2048, 49), (8192, 3072, 33), (14336, 4096, 33), (5632, 2048, 49), (8704, 2048, 33),
                                       (8192, 2304, 33), (7168, 3072, 33), (9728, 2048, 33)])
def test_gate_up_from(I, K, least):
    """Matrices up to that of 2 x 8,192 x 2,048, where the kernel for tens of rows is the faster one below, and larger ones."""
    assert ops.tile_least_rows_gate_up(2 * I, K) == least
