"""The machine code of the kernels whose loads are written in assembly: no register is used before its load is there.
And what the tiled products take, which decides how many of their blocks a compute unit holds."""

import os

import pytest

import kernel_code
from pagedserve_amd.ops import library

LISTING = """
0000000000001000 <waits>:
\tds_read_b128 v[4:7], v0                                     // 000000001000: D9FE0000 04000000
\tds_read_b128 v[8:11], v0 offset:16                          // 000000001008: D9FE0010 08000000
\ts_waitcnt lgkmcnt(1)                                        // 000000001010: BF8CC17F
\t{first}                            // 000000001014: 7E000304
\ts_cbranch_scc1 65530                                        // 000000001018: BF85FFFA <waits>
\ts_waitcnt lgkmcnt(0)                                        // 00000000101C: BF8CC07F
\tglobal_load_dwordx4 v[4:7], v[8:9], off                     // 000000001020: DC5C8000 047F0008
\tglobal_store_dword v[8:9], v10, off                         // 000000001028: DC708000 007F0A08
\ts_waitcnt vmcnt({left})                                        // 000000001030: BF8C0F70
\tv_mov_b32_e32 v1, v5                                        // 000000001034: 7E020305
\ts_endpgm                                                    // 000000001038: BF810000
"""


@pytest.mark.parametrize("first,left,registers", [
    ("v_mov_b32_e32 v0, v4", 1, set()),
    ("v_mov_b32_e32 v0, v4", 2, {("v", 5)}),             # the store is behind the load: two may be left
    ("v_mov_b32_e32 v0, v9", 0, {("v", 9)}),             # the second read, one may be left
    ("v_mov_b32_e32 v9, v4", 0, {("v", 9)}),             # what is on its way overwrites it
    ("global_store_dword v[0:1], v11, off", 1, {("v", 11)}),
])
def test_the_scan_finds_uses_before_the_wait(first, left, registers):
    (name, code), = kernel_code.kernels(LISTING.format(first=first, left=left))
    assert name == "waits" and len(code) == 11
    assert {register for _, _, register in kernel_code.early_uses(code)} == registers


INSTANCES = {"gemm_nt_bf16_two_sizes_kernel": 4}      # one for every epilogue but rows added to


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
@pytest.mark.parametrize("kernel", ["gemm_nt_bf16_large_kernel", "gemm_nt_bf16_two_sizes_kernel", "gemm_nt_ring_kernel",
                                    "attention_prefill_kernel", "attention_mixed_kernel"])
def test_no_register_is_used_before_its_load(kernel, tmp_path):
    """Every instance of the kernels that read their operands from LDS by assembly, as built.  (The wide product's
    last tiles wait by counts known at run time, which the scan cannot follow.)"""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    images = [image for image in kernel_code.code_objects(path, library.ARCH) if kernel.encode() in image]
    assert images, "no source file holds this kernel"
    seen = 0
    for image in images:
        for name, code in kernel_code.kernels(kernel_code.disassemble(image, library.ARCH, tmp_path)):
            if kernel in name:
                seen += 1
                assert any(operation.startswith("ds_read") for _, operation, _, _ in code), name
                assert not kernel_code.early_uses(code), (name, kernel_code.early_uses(code)[:4])
    assert seen == INSTANCES.get(kernel, seen) and seen


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
@pytest.mark.parametrize("kernel", ["gemm_nt_bf16_large_kernel", "gemm_nt_bf16_two_sizes_kernel", "gemm_nt_ring_kernel",
                                    "gemm_nt_bf16_wide_kernel"])
def test_tiled_products_call_nothing(kernel, tmp_path):
    """Their epilogue (gemm_tile.h) holds accumulators, bias, rows and pages in arrays: called and not inlined, it would
    take them through scratch memory, and would lie where the test above does not look."""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    seen = 0
    for image in kernel_code.code_objects(path, library.ARCH):
        if kernel.encode() not in image:
            continue
        for name, taken in kernel_code.resources(image, tmp_path).items():
            if kernel in name:
                seen += 1
                assert taken["vgpr"] > 0 and taken["scratch"] == 0, (name, taken)
        for name, code in kernel_code.kernels(kernel_code.disassemble(image, library.ARCH, tmp_path)):
            assert kernel not in name or not any(operation.startswith("s_swappc") for _, operation, _, _ in code), name
    assert seen == INSTANCES.get(kernel, seen) and seen


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
def test_float_rows_added_to_share_a_unit(tmp_path):
    """Tiles of 64 x 64 in two stages are taken where many blocks share a compute unit, four at least: 160 KB of LDS hold
    five, the registers of a SIMD, 512 to a lane, four waves of up to 128."""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    kernel, form = "gemm_nt_ring_kernel", "If" + "".join(f"Li{i}E" for i in (1, 1, 2))    # float, 1 x 1, two stages
    seen = 0
    for image in kernel_code.code_objects(path, library.ARCH):
        if kernel.encode() not in image:
            continue
        for name, taken in kernel_code.resources(image, tmp_path).items():
            if kernel + form in name:
                seen += 1
                assert taken["vgpr"] <= 128 and taken["lds"] <= 160 * 1024 // 4, (name, taken)
    assert seen == 5


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
def test_rows_added_to_by_two_tiles_of_columns_share_a_unit(tmp_path):
    """The skinny bfloat16 product of rows added to, two tiles of columns to a block: two of its blocks share a compute unit,
    256 registers to a lane each, but where 5 steps of 64 rows travel at once."""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    kernel = "gemm_nt_skinny_kernel"
    forms = {f"Li3ELi{rows}ELi2ELi{steps}E": (rows, steps) for rows in (2, 3, 4) for steps in (2, 3, 4, 5)}
    seen = set()
    for image in kernel_code.code_objects(path, library.ARCH):
        if kernel.encode() not in image:
            continue
        for name, taken in kernel_code.resources(image, tmp_path).items():
            for form in forms if kernel in name else ():
                if form in name:
                    seen.add(form)
                    assert taken["scratch"] == 0 and (taken["vgpr"] <= 256 or forms[form] == (4, 5)), (name, taken)
    assert len(seen) == len(forms)


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
def test_float_products_in_even_tiles_wait_for_their_operands(tmp_path):
    """Every instance: no register is used before its read from LDS is there, nothing goes through scratch memory, and as
    many blocks share a compute unit as the rule that picks a tile counts on (two, or three of 32 x 64)."""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    kernel = "gemm_nt_even_f32_kernel"
    resident = {"Li1ELi2ELi1ELi4E": 3, "Li1ELi3ELi1ELi4E": 2, "Li1ELi4ELi1ELi3E": 2, "Li1ELi5ELi1ELi3E": 2, "Li2ELi2ELi3ELi3E": 2}
    seen = []
    for image in kernel_code.code_objects(path, library.ARCH):
        if kernel.encode() not in image:
            continue
        for name, taken in kernel_code.resources(image, tmp_path).items():
            for form, blocks in resident.items():
                if kernel + "I" + form in name:
                    seen.append(form)
                    assert taken["scratch"] == 0 and taken["lds"] * blocks <= 160 * 1024, (name, taken)
                    assert (taken["vgpr"] + 7) // 8 * 8 * blocks <= 512, (name, taken)
        for name, code in kernel_code.kernels(kernel_code.disassemble(image, library.ARCH, tmp_path)):
            if kernel in name:
                assert not kernel_code.early_uses(code), (name, kernel_code.early_uses(code)[:4])
    assert len(seen) == 6 * len(resident)


@pytest.mark.skipif(kernel_code.disassembler() is None, reason="no disassembler")
def test_products_whose_waves_split_k_wait_for_their_operands(tmp_path):
    """Every instance: no register is used before its read from LDS is there, nothing goes through scratch memory."""
    path = os.path.join(library.in_tree_dir(), library.LIB_NAME)
    if not os.path.isfile(path):
        pytest.skip("the library is not built in the tree")
    kernel, seen = "gemm_nt_k_waves_kernel", 0
    for image in kernel_code.code_objects(path, library.ARCH):
        if kernel.encode() not in image:
            continue
        for name, taken in kernel_code.resources(image, tmp_path).items():
            if kernel in name:
                assert taken["scratch"] == 0, (name, taken)
        for name, code in kernel_code.kernels(kernel_code.disassemble(image, library.ARCH, tmp_path)):
            if kernel in name:
                seen += 1
                assert not kernel_code.early_uses(code), (name, kernel_code.early_uses(code)[:4])
    assert seen == 4 * 9
