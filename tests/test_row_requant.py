"""The row-streaming kernel's requantizing epilogue, bit-exact against the
oracle: both channel slice widths, one to four fragments per row, one-row
blocks, two and four channel groups, byte stores where N % 4 != 0."""
import numpy as np
import pytest

import int8_kernel_lab_amd as lab
from oracle import oracle
from tests.conftest import say
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
