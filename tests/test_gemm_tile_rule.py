"""The tile rule of the 2-byte GEMMs through its host-only queries (no GPU): on a
256-CU device.  Constants may be refitted; these are the products where a wrong
choice has cost a factor or a launch."""
import os

import pytest

BF16 = 2
GENERAL, T256, T256M, T128X256, T128, T128K2, T64, T64X128K2 = range(8)


@pytest.fixture(scope="module")
def lib():
    from zorse_amd import _abi
    if not os.path.exists(_abi.LIB_PATH):
        pytest.fail("libzorse_amd.so is not built: run python -m zorse_amd.build")
    return _abi.lib()


def _tile(lib, M, N, K, a_km=0, b_km=0):
    return lib.zk_gemm_tile(M, N, K, M if a_km else K, a_km, N if b_km else K, b_km, N, -1, BF16)


@pytest.mark.parametrize("b_km", [0, 1])
@pytest.mark.parametrize("M,N,K", [(3848, 2744, 24), (1064, 12088, 16), (8192, 1024, 8),
                                   (16384, 512, 24)])
def test_few_k_steps_count_their_stores(lib, M, N, K, b_km):
    """A product of one K step is bound by storing its output: 64 x 64 tiles
    take 1.1 to 1.5 times the general kernel's time, 128 x 128 tiles less."""
    assert _tile(lib, M, N, K, 0, b_km) == T128


@pytest.mark.parametrize("M,F,K", [(696, 6976, 64), (696, 11008, 128), (1536, 11008, 64),
                                   (2048, 6976, 64)])
def test_few_k_steps_gate_up(lib, M, F, K):
    """The same of gate|up, three outputs: 64 x 64 tiles 1.2 to 1.6 times the time."""
    assert lib.zk_gemm_swiglu_tile(M, F, K, K, K, 2 * F, BF16) == T128


@pytest.mark.parametrize("M,N,K,tile", [((1 << 30) - 64, 8, 8, T128), (1 << 30, 8, 8, GENERAL),
                                        (8, (1 << 30) + 8, 16, GENERAL), (1 << 29, 72, 8, GENERAL)])
def test_masked_tiles_fit_one_grid_dimension(lib, M, N, K, tile):
    """A launch holds fewer than 2^32 threads along its grid, 2^24 tiles of 256:
    products of as many 64 x 64 tiles keep to the general kernel's larger ones."""
    assert _tile(lib, M, N, K) == tile


@pytest.mark.parametrize("M,N,K", [(2048, 2048, 16), (2152, 1568, 48), (2048, 2048, 512),
                                   (1536, 2048, 256)])
def test_weight_gradients_of_few_tokens_fill_the_chip(lib, M, N, K):
    """63 tiles of 256 x 256 leave three quarters of the CUs idle: 14 us where the
    general kernel took 10 and 128 x 128 or 64 x 64 tiles take 7."""
    assert _tile(lib, M, N, K, 1, 1) in (T128, T64)
