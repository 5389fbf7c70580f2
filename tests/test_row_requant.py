"""The row-streaming kernel's requantizing epilogue, bit-exact against the
oracle: both channel slice widths, one to four fragments per row, one-row
blocks, two and four channel groups, byte stores where N % 4 != 0."""
import numpy as np
import pytest

import int8_kernel_lab_amd as lab
from oracle import oracle
from tests.conftest import say
from tests.test_gpu_parity import assert_bit_exact, run_kernel
from tests.test_requant import _qparams

CASES = {
    "c64_k64_nfr4": lab.ConvShape(8, 20, 56, 64, 64, 3, 3, 1, 1, 1, 1, 1, 1),
    "c64_k128_nfr1": lab.ConvShape(3, 14, 15, 64, 128, 3, 3, 1, 1, 1, 1, 1, 1),
    "c64_k100_nfr2": lab.ConvShape(2, 9, 29, 64, 100, 3, 3, 1, 1, 1, 1, 1, 1),
    "c64_k63_nfr3": lab.ConvShape(1, 17, 40, 64, 63, 3, 3, 1, 1, 1, 1, 1, 1),
    "c64_k32_rows": lab.ConvShape(32, 19, 13, 64, 32, 3, 3, 1, 1, 1, 1, 1, 1),
    "c64_one_pixel": lab.ConvShape(2, 1, 1, 64, 36, 3, 3, 1, 1, 1, 1, 1, 1),
    "c256_k72_pad0": lab.ConvShape(1, 12, 18, 256, 72, 3, 3, 0, 0, 1, 1, 1, 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
@pytest.mark.parametrize("form", ["odd", "mixed"])
def test_row_requant_bit_exact(name, form):
    shape = CASES[name]
    assert lab.describe("halo", shape).startswith("halo row-streaming:"), name
    assert lab.dispatch(shape) == "halo", name
    x, w, b = lab.make_case_data(shape, seed=41)
    if form == "odd":
        rng = np.random.default_rng(42)
        mult = (rng.integers(2 ** 29, 2 ** 30, size=shape.k) * 2 + 1).astype(np.int32)
        shift = rng.integers(44, 47, size=shape.k).astype(np.int32)
    else:
        mult, shift = _qparams(shape.k, seed=43)
    say(f"[gpu] row requant {name} {form} {shape}")
    got = lab.conv2d_requant(x, w, b, mult, shift, -6, shape)
    exp = oracle.requantize(oracle.conv(shape, x, w, b), mult, shift, -6)
    np.testing.assert_array_equal(got, exp)


ONE_ROUND = {
    # grids of just over 256 workgroups: fewer blocks per image, uneven ones
    # among them, one and two channel slices
    "c64_k64_12_blocks": (lab.ConvShape(21, 35, 36, 64, 64, 3, 3, 1, 1, 1, 1, 1, 1), "12 row blocks"),
    "c64_k192_9_blocks": (lab.ConvShape(9, 50, 50, 64, 192, 3, 3, 1, 1, 1, 1, 1, 1), "9 row blocks"),
    "c128_k416_2_blocks": (lab.ConvShape(13, 29, 30, 128, 416, 3, 3, 1, 1, 1, 1, 1, 1), "2 row blocks"),
    "c256_k60_6_blocks": (lab.ConvShape(37, 20, 20, 256, 60, 3, 3, 1, 1, 1, 1, 1, 1), "6 row blocks"),
}


@pytest.mark.parametrize("name", sorted(ONE_ROUND))
def test_row_plan_of_one_round(name):
    shape, blocks = ONE_ROUND[name]
    assert blocks in lab.describe("halo", shape)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(ONE_ROUND))
def test_row_one_round_bit_exact(name):
    shape = ONE_ROUND[name][0]
    x, w, b = lab.make_case_data(shape, seed=44)
    say(f"[gpu] row kernel {name} {shape}")
    acc = oracle.conv(shape, x, w, b)
    assert_bit_exact(run_kernel("halo", shape, x, w, b), acc, name)
    mult, shift = _qparams(shape.k, seed=45)
    np.testing.assert_array_equal(lab.conv2d_requant(x, w, b, mult, shift, 4, shape),
                                  oracle.requantize(acc, mult, shift, 4))
