"""Registers and scratch of the built kernels: figures that decide how many waves a SIMD holds, and
that a change of a kernel can move without any result showing it.  Read from the library; no GPU."""
import os
import re

import pytest

import kernel_resources
from karume_amd import _ffi


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(_ffi.LIB_PATH):
        pytest.skip("the library has not been built")
    found = kernel_resources.kernels()
    assert len(found) > 500
    return found


def arguments(name):
    return [a.strip() for a in re.search(r"<(.*)>", name).group(1).split(",")]


def test_one_head_decode_attention_leaves_room_for_two_waves_a_simd(kernels):
    checked = 0
    for name, kernel in kernels.items():
        if name.startswith("attention_decode_kernel<") and arguments(name)[2] == "1":
            assert kernel_resources.registers(kernel) <= 256, name
            checked += 1
    assert checked == 4 * 5 * 2    # element types, lanes a row, single and ragged


def test_tiles_of_w4a8_groups_up_to_128_keep_their_state_in_registers(kernels):
    tiles = {n: k for n, k in kernels.items() if n.startswith("linear_w4a8_tall_kernel<")}
    assert {arguments(n)[1] for n in tiles} == {"5", "6", "7"}
    for name, kernel in tiles.items():
        assert kernel_resources.scratch(kernel) == 0, name


def test_w4a8_groups_of_64_and_128_have_tiles_for_any_k(kernels):
    """Past a K of 2^24 the tiles above do not reach all rows with their offsets of 32 bits."""
    tiles = {(arguments(n)[1], arguments(n)[3]) for n in kernels if n.startswith("linear_w4a8_tile_kernel<")}
    assert tiles == {("6", "1")} | {(group, wide) for group in ("7", "8", "0") for wide in ("1", "2")}


def test_rows_to_quantize_have_threads_by_their_length(kernels):
    """A thread has up to three quads more than it needs: not sixteen waves for rows that eight hold."""
    forms = {tuple(int(a.rstrip("u")) for a in arguments(n)) for n in kernels if n.startswith("quantize_rows_kernel<")}
    assert forms == {(256, 1), (512, 1), (512, 2), (512, 3), (512, 4), (512, 6), (1024, 3)}


def test_norms_read_at_most_half_as_much_again_as_a_row_has(kernels):
    """Pieces past a row are loads all the same: forms for rows of up to 4, 8, 12, 16, 24, 32 and 48 pieces."""
    forms = {tuple(arguments(n)) for n in kernels if n.startswith("rms_norm_kernel<")}
    types = (("float", "float"), ("__half", "__half"), ("float", "__half"))
    assert forms == {(*t, kept) for t in types for kept in ("0", "4", "8", "12", "16", "24", "32", "48")}


# The forms that spill: the large f32-activation forms of the GEMM on fp16 weights (f32 x is rounded in the
# loop, beside a 64 x 64 tile a wave).
SPILL = ("gemm_i4_f16_kernel<float, __half, 2, 2, 64, 1, 4, true,",
         "gemm_i4_f16_kernel<float, float, 2, 2, 64, 1, 4, true,")


def test_no_other_kernel_uses_scratch_memory(kernels):
    spilling = {n for n, k in kernels.items() if kernel_resources.scratch(k) > 0}
    assert {n for n in spilling if not n.startswith(SPILL)} == set()


def test_every_form_that_may_spill_does(kernels):
    spilling = {n for n, k in kernels.items() if kernel_resources.scratch(k) > 0}
    assert [p for p in SPILL if not any(n.startswith(p) for n in spilling)] == []


def test_rows_of_the_gemv_brought_to_lds_are_built_without_a_norm(kernels):
    """Rows of x in LDS (a step count of -1) are picked without a norm alone: no other instance is built."""
    staged = [arguments(n) for n in kernels if n.startswith("gemv_i4_kernel<") and arguments(n)[5] == "-1"]
    assert len(staged) == 12
    assert {(a[6], a[7]) for a in staged} == {("false", "false")}
