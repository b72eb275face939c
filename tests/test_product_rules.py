"""Which kernel takes a matrix product: the rules' lines, which are drawn for 256 compute units (what the library
assumes without a device)."""

import ctypes

import pytest
import torch

from pagedserve_amd.ops import kernels, library


@pytest.fixture
def lib():
    if torch.cuda.is_available() and kernels.compute_units() != 256:
        pytest.skip("the lines are drawn for 256 compute units")
    return library.load_library()


FEW, K_WAVES, TWO_SIZES, LARGE, WIDE, RING, PLAIN = range(7)


def _choice(lib, m, n, k, outputs="bfloat16", epilogue="none", packed=True, scatter=False):
    """(kernel, tile or columns of the first size, ranges of k) of a product of bfloat16 operands."""
    tile, ranges = ctypes.c_int(), ctypes.c_int()
    kernel = lib.ps_linear_choice(m, n, k, 0 if outputs == "float32" else 1, kernels.EPILOGUES[epilogue], int(packed), int(scatter),
                                  ctypes.byref(tile), ctypes.byref(ranges))
    return kernel, tile.value, ranges.value


@pytest.mark.parametrize("m,n,k,plain,floats,added", [
    (64, 2304, 768, None, None, None), (65, 2304, 768, 0, 0, None),                       # 65 rows; few rows added to: 97
    (97, 2304, 448, None, None, None), (97, 2304, 512, 0, 0, 0), (97, 2304, 544, None, None, None),      # whole stages, eight of them
    (224, 2304, 768, 0, 0, 0), (225, 2304, 768, 1, 1, 1), (320, 2304, 768, 1, 1, 1),      # one round of 32 x 64, 32 x 96,
    (321, 2304, 768, 2, 2, 2), (448, 2304, 768, 2, 2, 2), (449, 2304, 768, 3, 3, 3),      # 64 x 64,
    (576, 2304, 768, 3, 3, 3), (577, 2304, 768, None, 3, 3), (640, 2304, 768, None, 3, 3), (641, 2304, 768, None, None, None),
    (392, 3072, 1024, 3, 3, 3), (449, 3072, 1024, None, 3, 3),      # 7/8 of the units (bfloat16), all
    (2048, 768, 3072, None, 3, 3), (2049, 768, 3072, None, None, None),
    (128, 6400, 1600, 2, 2, 2), (160, 6400, 1600, None, None, None), (168, 6400, 1024, 3, 3, 3), (193, 4800, 1600, 3, 3, 3),   # three rows
    (110, 9600, 1024, 3, 3, 3),                                                           # of 64 x 96: a k of up to 1,024
    (260, 4092, 768, 3, 3, 3), (260, 4097, 768, 3, 3, None), (256, 4097, 768, 3, 3, 3)])      # rows in no pieces of four
def test_who_splits_k_over_its_waves(lib, m, n, k, plain, floats, added):
    """The tile of a product whose waves split k, None where it goes elsewhere: both sides of the rule's lines."""
    for outputs, epilogue, tile in (("bfloat16", "none", plain), ("bfloat16", "gelu_tanh", plain), ("float32", "none", floats),
                                    ("float32", "residual", added)):
        choice = _choice(lib, m, n, k, outputs, epilogue)
        assert choice == (K_WAVES, tile, 1) if tile is not None else choice[0] != K_WAVES


@pytest.mark.parametrize("m,n,k,plain,floats,added", [
    (393, 3456, 1024, LARGE, "64x96", "64x96"), (393, 3456, 1088, LARGE, "64x96", LARGE), (392, 3008, 1088, "64x96", "64x96", "64x96"),
    (576, 2304, 768, "64x96", "64x96", "64x96"), (169, 6400, 1024, LARGE, "64x96", "64x96"), (168, 6400, 1024, "64x96", "64x96", "64x96"),
    (281, 4800, 1280, LARGE, LARGE, LARGE), (280, 4096, 1280, "64x96", "64x96", "64x96"), (384, 3072, 1280, "64x96", "64x96", "64x96"),
    (805, 1600, 3520, "64x96", "64x96", "64x96"), (805, 1600, 3584, LARGE, "64x96", "64x96"), (805, 1792, 3584, LARGE, "64x96", LARGE),
    (704, 768, 4096, "64x64", "64x64", "64x64"), (704, 768, 4160, RING, "64x64", RING), (768, 768, 4160, RING, "64x64", RING),
    (729, 768, 4160, "64x64", "64x64", "64x64"), (730, 768, 4160, RING, "64x64", RING), (832, 768, 4160, "64x64", "64x64", "64x64"),
    (1088, 512, 4160, "64x64", "64x64", "64x64"), (250, 2304, 6400, "64x64", "64x64", "64x64"),
    (1088, 1024, 3456, "64x96", "64x96", "64x96"), (1088, 1024, 3520, RING, RING, RING), (1066, 1024, 3520, "64x96", "64x96", "64x96"),
    (1472, 768, 5120, "64x96", "64x96", "64x96"), (1536, 768, 5120, RING, RING, RING), (1600, 768, 5120, "64x96", "64x96", "64x96")])
def test_who_splits_k_over_its_waves_in_full_tiles(lib, m, n, k, plain, floats, added):
    """Tiles that the rows nearly fill: the kernel of a product that goes elsewhere, the tile of one that stays."""
    for outputs, epilogue, expected in (("bfloat16", "none", plain), ("bfloat16", "gelu_tanh", plain), ("float32", "none", floats),
                                        ("float32", "residual", added)):
        kernel, tile, ranges = _choice(lib, m, n, k, outputs, epilogue)
        assert (("32x64", "32x96", "64x64", "64x96")[tile] if kernel == K_WAVES else kernel) == expected
        assert (kernel != LARGE or tile == 11) and ranges == 1


@pytest.mark.parametrize("m,n,k,waves", [
    (96, 512, 512, False), (97, 512, 512, True), (97, 64, 576, True), (97, 320, 640, False),          # a k of up to 576: any outputs
    (128, 512, 1024, False), (136, 512, 1024, False), (137, 512, 1024, True), (97, 768, 1024, True),  # 70,000 outputs
    (128, 768, 1536, False), (131, 768, 1536, True), (97, 768, 1408, True), (137, 512, 1600, True),   # a k in two ranges of 768
    (133, 768, 2048, False), (134, 768, 2048, True), (160, 64, 5120, False), (128, 768, 3072, True),  # 2.1e8 products
    (97, 1030, 1024, False), (97, 1028, 1024, True), (130, 321, 6400, False)])                        # not in pieces of four
def test_who_takes_few_rows_added_to(lib, m, n, k, waves):
    """Rows added to that the kernel for few rows could take: whether they go to the one whose waves split k."""
    assert _choice(lib, m, n, k, "float32", "residual")[0] == (K_WAVES if waves else FEW)
    # ranges of k, whose sums are added by atomics, only where the other kernel has them too
    assert _choice(lib, m, n, k, "float32", "residual")[2] == 1 or k > 1024


@pytest.mark.parametrize("m,n,k,columns", [
    (3840, 6400, 1600, 0), (3841, 6400, 1600, 5120), (4096, 6400, 1600, 5120), (4097, 6400, 1600, 0),
    (7680, 6400, 1600, 0), (7681, 6400, 1600, 5120), (8192, 6400, 1600, 5120), (8193, 6400, 1600, 0),
    (2048, 12800, 1600, 10240), (4096, 6400, 1536, 5120), (4096, 6400, 1472, 0), (1023, 12800, 1600, 0)])
def test_who_takes_two_sizes_of_tiles(lib, m, n, k, columns):
    """The columns of the first size, 0: one size; bfloat16 outputs that nothing is added to, without key/value scatter."""
    choice = _choice(lib, m, n, k)
    assert choice[:2] == (TWO_SIZES, columns) if columns else choice[0] != TWO_SIZES
    assert _choice(lib, m, n, k, epilogue="gelu_tanh") == choice
    assert _choice(lib, m, n, k, scatter=True)[0] != TWO_SIZES
    assert _choice(lib, m, n, k, "float32")[0] != TWO_SIZES and _choice(lib, m, n, k, "float32", "residual")[0] != TWO_SIZES


@pytest.mark.parametrize("m,n,k,tile", [(17, 2304, 768, 0), (544, 2304, 768, 0), (193, 3072, 1024, 1), (544, 1024, 4096, 1),
                                        (1163, 1600, 1600, 2), (2048, 3072, 768, 0), (2500, 3072, 1024, 3), (1200, 4800, 1600, 4)])
def test_tiles_of_float_products(lib, m, n, k, tile):
    """32 x 64, 48 x 64, 64 x 64, 80 x 64 or 64 x 96, by the fitted time."""
    assert _even(lib, m, n, k, "residual" if k > n else "none")[0] == tile


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
