"""Which kernel takes a matrix product: the rules' lines, which are drawn for 256 compute units (what the library
assumes without a device)."""

import pytest
import torch

from pagedserve_amd.ops import kernels, library


@pytest.fixture
def lib():
    if torch.cuda.is_available() and kernels.compute_units() != 256:
        pytest.skip("the lines are drawn for 256 compute units")
    return library.load_library()


def _even(lib, m, n, k, epilogue):
    """(tile, ranges of k) of a float product."""
    choice = lib.ps_gemm_nt_even_choice(m, n, k, kernels.EPILOGUES[epilogue])
    assert choice >= 16
    return choice % 16, choice // 16


@pytest.mark.parametrize("m,n,k,ranges", [
    (224, 768, 768, 1), (160, 1024, 1024, 1), (400, 512, 1024, 1), (160, 1600, 1024, 1),        # a short k
    (300, 768, 3072, 4), (544, 1024, 4096, 4), (544, 1600, 6400, 3),
    (2100, 768, 3072, 1), (1700, 1024, 4096, 1), (1024, 1600, 6400, 1), (6000, 1600, 6400, 1)])   # more than 384 tiles of 64 x 64
def test_ranges_of_k_of_float_products(lib, m, n, k, ranges):
    """Ranges of k, whose sums atomics add in no fixed order: rows that are added to, a k of more than 1,024, tiles of
    64 x 64 for one and a half to a unit at most."""
    assert _even(lib, m, n, k, "residual")[1] == ranges
    assert _even(lib, m, n, k, "none")[1] == _even(lib, m, n, k, "gelu_tanh")[1] == 1


@pytest.mark.parametrize("m,n,k,columns", [
    (65, 192, 64, 32), (129, 192, 64, 32), (300, 1000, 96, 32), (2048, 256, 32, 32), (500, 1024, 64, 32),        # 128 tiles of 64 x 64
    (513, 1024, 64, 64), (2049, 256, 32, 64), (4096, 4096, 64, 64)])
def test_tiles_of_float_products_of_a_short_k(lib, m, n, k, columns):
    """A k of up to 96: 64 x 32 by pairs of k tiles where tiles of 64 x 64 come to half of the units at most."""
    assert lib.ps_gemm_nt_even_choice(m, n, k, kernels.EPILOGUES["none"]) == -1
    assert lib.ps_gemm_nt_f32_ring_columns(m, n, k) == columns
