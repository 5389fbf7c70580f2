"""The generic kernel's 32 x 32 x 32 MFMA form, bit-exact against the oracle
with int32 and int8 output: each of its tiles at their edges (pixel and channel
tails, a k tail inside a stage, stages that span taps), through `generic` and
through the dispatched requantized launch."""
import numpy as np
import pytest

import int8_kernel_lab_amd as lab
from oracle import oracle
from tests.conftest import say
from tests.test_gpu_parity import assert_bit_exact, run_kernel
from tests.test_requant import _qparams

CASES = {
    # 64 x 64: one pixel past a tile and one channel past a tile, C = 80;
    # C = 16 with 27 bytes short of two stages; a strided C = 384 layer whose
    # pipelined grid would be small; gemm_k of exactly one stage
    "64_m65_n65_c80": ("64px x 64oc", lab.ConvShape(1, 5, 13, 80, 65, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_c16_5x3": ("64px x 64oc", lab.ConvShape(3, 19, 23, 16, 68, 5, 3, 2, 0, 2, 1, 1, 2)),
    "64_c384_s2": ("64px x 64oc", lab.ConvShape(2, 23, 21, 384, 132, 3, 3, 1, 1, 2, 2, 1, 1)),
    # groups of waves on a tile's stages: two (7 and 15 stages: the second
    # group's last one past the reduction), four (25 and 26 stages); one round
    # of tiles, and with two groups a second tile for some workgroups (512)
    "64_g2_c96": ("64px x 64oc, grid 4x2, 7 k-stages, 2 wave groups",
                  lab.ConvShape(1, 15, 14, 96, 72, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_g2_c208_k33": ("64px x 64oc, grid 38x1, 15 k-stages, 2 wave groups",
                       lab.ConvShape(3, 27, 30, 208, 33, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_g2_450_tiles": ("64px x 64oc, grid 225x2, 6 k-stages, 2 wave groups",
                        lab.ConvShape(10, 40, 36, 80, 100, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_g2_632_tiles": ("64px x 64oc, grid 316x2, 8 k-stages, 2 wave groups",
                        lab.ConvShape(6, 58, 58, 112, 100, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_g4_c352": ("64px x 64oc, grid 4x2, 25 k-stages, 4 wave groups",
                   lab.ConvShape(2, 11, 10, 352, 68, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_g4_c656_5x1": ("64px x 64oc, grid 6x3, 26 k-stages, 4 wave groups",
                       lab.ConvShape(5, 9, 8, 656, 132, 5, 1, 2, 0, 1, 1, 1, 1)),
    # ... and of a layer that the pipelined kernel would run on 22 tiles
    "64_g4_c512_k132": ("64px x 64oc, grid 21x3, 36 k-stages, 4 wave groups",
                        lab.ConvShape(1, 35, 37, 512, 132, 3, 3, 1, 1, 1, 1, 1, 1)),
    "64_k128": ("64px x 64oc", lab.ConvShape(18, 31, 33, 32, 36, 2, 2, 0, 0, 1, 1, 1, 1)),
    # 128 x 64: C = 32 and 48, odd channel counts, padding wider than the image
    "128x64_c32_k63": ("128px x 64oc", lab.ConvShape(5, 121, 119, 32, 63, 3, 3, 1, 1, 1, 1, 1, 1)),
    # ... more tiles than the 768 workgroups
    "128x64_k40_851_tiles": ("128px x 64oc, grid 851x1",
                             lab.ConvShape(1, 330, 330, 32, 40, 3, 3, 1, 1, 1, 1, 1, 1)),
    # 128 x 32: at most 32 channels, also of pixel rows past the image; more
    # tiles than workgroups
    "128x32_k20_851_tiles": ("128px x 32oc, grid 851x1",
                             lab.ConvShape(1, 330, 330, 32, 20, 3, 3, 1, 1, 1, 1, 1, 1)),
    "128x32_c48_k4": ("128px x 32oc", lab.ConvShape(1, 250, 263, 48, 4, 7, 7, 3, 3, 1, 1, 1, 1)),
    "128x32_c32_k32": ("128px x 32oc", lab.ConvShape(3, 151, 149, 32, 32, 3, 3, 1, 1, 1, 1, 1, 1)),
    "128x64_c48_k36": ("128px x 64oc", lab.ConvShape(1, 250, 263, 48, 36, 5, 5, 3, 3, 1, 1, 1, 1)),
    # 128 x 128: N = 65 and 255 (one, then two channel tiles), 1x3 dilated
    "128_k65": ("128px x 128oc", lab.ConvShape(2, 129, 130, 64, 65, 3, 3, 1, 1, 1, 1, 1, 1)),
    "128_k255": ("128px x 128oc", lab.ConvShape(1, 130, 131, 64, 255, 1, 3, 0, 2, 1, 1, 1, 2)),
    "128_k250_652_tiles": ("128px x 128oc, grid 326x2",
                           lab.ConvShape(1, 205, 203, 48, 250, 1, 3, 0, 1, 1, 1, 1, 1)),
    "128_k260": ("128px x 128oc", lab.ConvShape(1, 123, 125, 112, 260, 1, 1, 0, 0, 1, 1, 1, 1)),
    # 256 x 256: 514 tiles (two full rounds and a partial one), N = 132; three
    # channel chunks of a 1x3 filter and a stride-2 layer, both with a pixel
    # tail and N = 388 (a second channel tile of which half is dead)
    "256_c384_1x3_k388": ("256px x 256oc, grid 256x2, 9 k-stages",
                          lab.ConvShape(1, 255, 257, 384, 388, 1, 3, 0, 1, 1, 1, 1, 1)),
    "256_s2_k388": ("256px x 256oc, grid 256x2, 9 k-stages",
                    lab.ConvShape(1, 509, 513, 128, 388, 3, 3, 1, 1, 2, 2, 1, 1)),
    "256_k132": ("256px x 256oc", lab.ConvShape(2, 256, 257, 128, 132, 3, 3, 1, 1, 1, 1, 1, 1)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_gemm32_runs_these_layers(name):
    tile, shape = CASES[name]
    assert f"32x32 MFMA tile {tile}" in lab.describe("generic", shape)


@pytest.mark.parametrize("n,hw,c,k,r,small", [
    # one 64 x 64 tile per compute unit at most, from six stages on
    (1, 128, 256, 64, 3, True), (1, 129, 256, 64, 3, False), (2, 40, 256, 192, 3, True),
    (1, 36, 512, 256, 3, True), (1, 36, 512, 256, 1, False), (1, 36, 768, 256, 1, True)])
def test_64_wide_tiles_of_deep_layers_in_one_round(n, hw, c, k, r, small):
    s = lab.ConvShape(n, hw, hw, c, k, r, r, r // 2, r // 2, 1, 1, 1, 1)
    assert ("32x32 MFMA tile 64px x 64oc" in lab.describe("generic", s)) == small


@pytest.mark.parametrize("n,hw,c,k,tile", [
    # at least 256 tiles of 128 x 128: 64 x 64 up to 896 tiles, from eight stages on
    (1, 130, 224, 160, 64), (4, 56, 160, 288, 128), (8, 64, 160, 72, 128), (4, 57, 160, 320, 128),
    (1, 130, 96, 160, 128), (1, 128, 224, 160, 64)])
def test_64_wide_tiles_up_to_two_rounds(n, hw, c, k, tile):
    s = lab.ConvShape(n, hw, hw, c, k, 3, 3, 1, 1, 1, 1, 1, 1)
    assert f"32x32 MFMA tile {tile}px x {tile}oc" in lab.describe("generic", s)


@pytest.mark.parametrize("n,hw,c,k,r,wide", [
    # 256-wide tiles where they compute at most 8/7 of the columns that 128-wide
    # ones do
    (1, 512, 128, 129, 3, True), (1, 512, 128, 256, 3, True), (1, 512, 128, 385, 3, True),
    (1, 512, 128, 257, 3, False), (1, 512, 128, 384, 3, False), (1, 512, 128, 128, 3, False),
    (1, 512, 128, 640, 3, False), (1, 512, 128, 896, 3, True),
    # rounds of 256: 1024 tiles are four; 520 leave most of a third empty,
    # which only short reductions make up for
    (1, 512, 256, 256, 3, True), (1, 364, 256, 256, 3, False), (1, 364, 128, 256, 3, True),
    # 960 tiles: 15/16 of four rounds
    (15, 128, 256, 256, 3, True)])
def test_256_wide_tiles_where_they_pay(n, hw, c, k, r, wide):
    shape = lab.ConvShape(n, hw, hw, c, k, r, r, r // 2, r // 2, 1, 1, 1, 1)
    assert ("256px x 256oc" in lab.describe("generic", shape)) == wide


@pytest.mark.parametrize("hw,c,k,r,tile", [
    # at most 32 channels: 128 x 32 from 256 tiles on, below that
    # register-staged up to three stages; more channels or stages: 64 x 64
    (181, 32, 32, 1, "32x32 MFMA tile 128px x 32oc"), (181, 160, 32, 3, "32x32 MFMA tile 128px x 32oc"),
    (180, 32, 32, 1, "register-staged"), (180, 32, 32, 3, "register-staged"),
    (180, 48, 32, 3, "32x32 MFMA tile 64px x 64oc"), (180, 32, 33, 1, "32x32 MFMA tile 64px x 64oc"),
    (181, 32, 33, 1, "32x32 MFMA tile 64px x 64oc"), (120, 32, 64, 1, "register-staged")])
def test_narrow_short_layers(hw, c, k, r, tile):
    shape = lab.ConvShape(1, hw, hw, c, k, r, r, r // 2, r // 2, 1, 1, 1, 1)
    assert tile in lab.describe("generic", shape)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_gemm32_bit_exact(name):
    _, shape = CASES[name]
    x, w, b = lab.make_case_data(shape, seed=31)
    expected = oracle.conv(shape, x, w, b)
    say(f"[gpu] generic (32x32 MFMA) on {name} {shape}")
    assert_bit_exact(run_kernel("generic", shape, x, w, b), expected, name)
    if lab.dispatch(shape) != "generic":
        return
    for seed, zp in ((32, 5), (None, -9)):
        if seed is None:
            # every channel in the odd-multiplier form's domain
            rng = np.random.default_rng(33)
            mult = (rng.integers(2 ** 29, 2 ** 30, size=shape.k) * 2 + 1).astype(np.int32)
            shift = rng.integers(44, 47, size=shape.k).astype(np.int32)
        else:
            mult, shift = _qparams(shape.k, seed=seed)
        say(f"[gpu] requantized, seed {seed}")
        got = lab.conv2d_requant(x, w, b, mult, shift, zp, shape)
        np.testing.assert_array_equal(got, oracle.requantize(expected, mult, shift, zp))


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["64_m65_n65_c80", "128_k260"])
def test_gemm32_output_at_four_bytes(name):
    # an output 4 bytes past an allocation's start, nothing written around it
    _, shape = CASES[name]
    x, w, b = lab.make_case_data(shape, seed=34)
    count = shape.output_elements
    bufs = [lab.DeviceBuffer.from_array(a) for a in (x, w, b)]
    yb = lab.DeviceBuffer(4 * count + 16)
    try:
        yb.fill(0xA5)
        say(f"[gpu] generic (32x32 MFMA) on {name} with the output at +4 bytes")
        lab.launch("generic", shape, *bufs, yb.ptr + 4)
        lab.synchronize()
        raw = yb.download(np.int32, count + 4)
    finally:
        for buf in bufs + [yb]:
            buf.close()
    poison = np.uint32(0xA5A5A5A5).view(np.int32)
    assert raw[0] == poison and np.all(raw[count + 1:] == poison)
    assert_bit_exact(raw[1:count + 1].reshape(shape.output_shape), oracle.conv(shape, x, w, b), name)


BYTE_CASES = {
    # byte stores of int8: channel tails in each tile and wave grouping, a
    # pixel tail, more tiles than workgroups, and layers whose int32 output
    # the pipelined kernel computes
    "64_k67": lab.ConvShape(1, 13, 11, 80, 67, 3, 3, 1, 1, 1, 1, 1, 1),
    "64_k95_two_groups": lab.ConvShape(1, 14, 13, 144, 95, 3, 3, 1, 1, 1, 1, 1, 1),
    "64_k33_four_groups": lab.ConvShape(2, 27, 25, 368, 33, 3, 3, 1, 1, 1, 1, 1, 1),
    "128x64_k63": lab.ConvShape(5, 115, 119, 48, 63, 3, 1, 1, 0, 1, 1, 1, 1),
    "128x32_k31": lab.ConvShape(2, 187, 185, 48, 31, 1, 3, 0, 1, 1, 1, 1, 1),
    "128x128_k94": lab.ConvShape(3, 137, 131, 32, 94, 3, 3, 1, 1, 1, 1, 1, 1),
    "128x128_k255_again": lab.ConvShape(1, 205, 203, 48, 255, 1, 3, 0, 1, 1, 1, 1, 1),
    "256_k255": lab.ConvShape(1, 363, 361, 128, 255, 3, 3, 1, 1, 1, 1, 1, 1),
    "64_k30_halo_layer": lab.ConvShape(3, 22, 21, 64, 30, 3, 3, 2, 2, 1, 1, 2, 2),
    "pipelined_k101": lab.ConvShape(2, 101, 97, 128, 101, 3, 3, 1, 1, 2, 2, 1, 1),
    "pipelined_k130": lab.ConvShape(4, 64, 67, 384, 130, 1, 1, 0, 0, 1, 1, 1, 1),
}


def test_gemm32_byte_stores_on_256_wide_tiles():
    assert "32x32 MFMA tile 256px x 256oc, grid 512x1" in lab.describe("generic", BYTE_CASES["256_k255"])


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(BYTE_CASES))
@pytest.mark.parametrize("off", [0, 3])
def test_gemm32_int8_byte_stores(name, off):
    shape = BYTE_CASES[name]
    x, w, b = lab.make_case_data(shape, seed=35)
    mult, shift = _qparams(shape.k, seed=36)
    expected = oracle.requantize(oracle.conv(shape, x, w, b), mult, shift, 7)
    count, need = shape.output_elements, lab.requant_workspace_bytes(shape)
    bufs = [lab.DeviceBuffer.from_array(a) for a in (x, w, b, mult, shift)]
    yb, ws = lab.DeviceBuffer(count + 16), lab.DeviceBuffer(max(need, 1))
    try:
        yb.fill(0x5A)
        say(f"[gpu] int8 byte stores, {name} at +{off} bytes")
        lab.launch_requant(shape, *bufs[:5], 7, yb.ptr + off, ws, need)
        lab.synchronize()
        raw = yb.download(np.int8, count + 16)
    finally:
        for buf in bufs + [yb, ws]:
            buf.close()
    assert (raw[:off] == 0x5A).all() and (raw[off + count:] == 0x5A).all()
    np.testing.assert_array_equal(raw[off:off + count].reshape(shape.output_shape), expected)


PIPELINED = {
    # the pipelined kernel's requantizing epilogue on each of its tiles: with
    # and without copy waves, channel tails inside a 32-channel block and past
    # one, pixel tails, tiles that store fewer rows than they have
    "128x128_k100": ("128px x 128oc, grid 74x1, 18 k-stages, 4 copy waves",
                     lab.ConvShape(2, 71, 66, 256, 100, 3, 3, 1, 1, 1, 1, 1, 1)),
    "128x128_k384_rows": ("128px x 128oc (96px stored), grid 149x3, 4 k-stages, 4 copy waves",
                          lab.ConvShape(1, 121, 118, 512, 384, 1, 1, 0, 0, 1, 1, 1, 1)),
    "128x128_two_stages": ("128px x 128oc, grid 74x2, 2 k-stages",
                           lab.ConvShape(2, 71, 66, 256, 132, 1, 1, 0, 0, 1, 1, 1, 1)),
    "128x64_k60": ("128px x 64oc, grid 74x1, 3 k-stages",
                   lab.ConvShape(2, 71, 66, 128, 60, 1, 3, 0, 1, 1, 1, 1, 1)),
    "256x64_k36": ("256px x 64oc, grid 193x1, 5 k-stages",
                   lab.ConvShape(1, 222, 222, 128, 36, 5, 1, 2, 0, 1, 1, 1, 1)),
    "256x128_k76": ("256px x 128oc, grid 193x1, 5 k-stages, 8 copy waves",
                    lab.ConvShape(1, 222, 222, 128, 76, 5, 1, 2, 0, 1, 1, 1, 1)),
}


@pytest.mark.parametrize("name", sorted(PIPELINED))
def test_pipelined_kernel_runs_these_layers(name):
    tile, shape = PIPELINED[name]
    assert f"pipelined tile {tile}" in lab.describe("generic", shape)
    assert lab.dispatch(shape) == "generic"


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(PIPELINED))
def test_pipelined_requant_bit_exact(name):
    _, shape = PIPELINED[name]
    x, w, b = lab.make_case_data(shape, seed=51)
    acc = oracle.conv(shape, x, w, b)
    rng = np.random.default_rng(52)
    odd = ((rng.integers(2 ** 29, 2 ** 30, size=shape.k) * 2 + 1).astype(np.int32),
           rng.integers(44, 47, size=shape.k).astype(np.int32))
    # shifts below 33: no channel in the odd-multiplier form's domain
    exact = (rng.integers(100, 200, size=shape.k).astype(np.int32),
             np.full(shape.k, 22, np.int32))
    mixed = (odd[0].copy(), odd[1].copy())
    mixed[0][shape.k - 1], mixed[1][shape.k - 1] = exact[0][0], exact[1][0]
    for form, (mult, shift) in (("odd", odd), ("exact", exact), ("mixed", mixed)):
        say(f"[gpu] pipelined requant {name} {form}")
        got = lab.conv2d_requant(x, w, b, mult, shift, 11, shape)
        exp = oracle.requantize(acc, mult, shift, 11)
        assert len(np.unique(exp)) > 50
        np.testing.assert_array_equal(got, exp, err_msg=form)


# more than 2^20 output channels, C % 128 == 0: past the buffer windows of the
# other forms (a pixel row of this output is 4 MB)
VERY_WIDE = lab.ConvShape(1, 3, 3, 256, (1 << 20) + 4, 1, 1)


def test_very_wide_layers_stay_on_the_pipelined_kernel():
    assert "pipelined tile 128px x 128oc (80px stored), grid 1x8193" in lab.describe("generic", VERY_WIDE)
    assert lab.dispatch(VERY_WIDE) == "generic"
    assert lab.requant_fused(VERY_WIDE) and lab.requant_workspace_bytes(VERY_WIDE) == 0
    assert "pipelined" in lab.describe("splitk", VERY_WIDE)


@pytest.mark.gpu
def test_very_wide_layers_bit_exact():
    shape = VERY_WIDE
    x, w, b = lab.make_case_data(shape, seed=71)
    acc = oracle.conv(shape, x, w, b)
    for kernel in ("generic", "splitk"):
        say(f"[gpu] {kernel} on {shape}")
        assert_bit_exact(run_kernel(kernel, shape, x, w, b), acc, kernel)
    mult, shift = _qparams(shape.k, seed=72)
    say("[gpu] requantized")
    got = lab.conv2d_requant(x, w, b, mult, shift, -1, shape)
    np.testing.assert_array_equal(got, oracle.requantize(acc, mult, shift, -1))


@pytest.mark.gpu
@pytest.mark.parametrize("k", [64, 60, 36, 24, 63])
def test_splitk_64_channel_tiles_bit_exact(k):
    # partial sums in 16-byte stores (whole sectors, ordinary, a tail inside a
    # 32-channel block), in 4-byte stores (N % 4 != 0); a pixel tail; the last
    # split shorter than the others
    shape = lab.ConvShape(1, 17, 13, 384, k, 3, 3, 2, 2, 1, 1, 2, 2)
    assert "splitk pipelined tile 128px x 64oc" in lab.describe("splitk", shape)
    x, w, b = lab.make_case_data(shape, seed=81)
    say(f"[gpu] splitk on {shape}")
    assert_bit_exact(run_kernel("splitk", shape, x, w, b), oracle.conv(shape, x, w, b), f"k{k}")
