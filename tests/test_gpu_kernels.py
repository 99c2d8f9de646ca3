"""Parity of every hand-written HIP kernel against the CPU oracle, called through the C-ABI
device layer (include/dr_hip.h) with plain device pointers.

Tolerances (north star): fp32 layers max relative error <= 1e-4, measured as
max|gpu - oracle| / max|oracle| over the layer; pooling values and max-indices bit-exact.
"""
import ctypes
import os

import numpy as np
import pytest

from conftest import Dev, assert_close, rel_err

pytestmark = pytest.mark.gpu

TOL = 1e-4
RNG = np.random.default_rng(7)


def rnd(*shape, scale=1.0):
    return (RNG.standard_normal(shape) * scale).astype(np.float32)


# (tests that draw from this one leave the inputs of the others as they are)
OWN = np.random.default_rng(8)


def own(*shape, scale=1.0):
    return (OWN.standard_normal(shape) * scale).astype(np.float32)


def ok(lib, rc):
    assert rc == 0, lib.drhip_last_error().decode()


# ---------------------------------------------------------------------------------------------

@pytest.mark.parametrize("W,H,I,O,k,s", [
    (56, 56, 64, 64, 3, 1),      # config 1, direct variant
    (224, 224, 3, 64, 3, 2),     # SqueezeNet conv1
    (17, 13, 5, 7, 3, 1), (20, 18, 4, 20, 5, 1), (33, 31, 3, 9, 3, 2), (16, 16, 2, 3, 7, 3), (9, 9, 1, 1, 1, 2),
    (37, 21, 4, 33, 3, 1), (8, 5, 1, 16, 3, 3), (2, 2, 3, 2, 3, 1),     # I <= 4 with a 3x3 filter: the no-LDS first-layer kernel
    (112, 110, 24, 40, 3, 1), (61, 37, 17, 70, 3, 2), (30, 9, 8, 32, 3, 1),   # 3x3 with raw weights and more than 4 channels: the LDS-tiled kernel
])
def test_conv_direct(lib, dev, oracle, W, H, I, O, k, s):
    x, w, b = np.abs(rnd(I, H, W)), rnd(I, O, k, k, scale=np.sqrt(2.0 / (k * k * I))), rnd(O, scale=0.01)
    want = oracle.conv_direct(x, w, b, (s, s), relu=True)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv2d_direct_f32(dev.put(x), dev.put(w), dev.put(b), out, W, H, I, O, k, k, s, s, 1, None))
    got = dev.get(out, want.shape)
    assert_close(got, want)
    # linear, no bias
    want2 = oracle.conv_direct(x, w, None, (s, s), relu=False)
    ok(lib, lib.drhip_conv2d_direct_f32(dev.put(x), dev.put(w), None, out, W, H, I, O, k, k, s, s, 0, None))
    assert_close(dev.get(out, want2.shape), want2)


@pytest.mark.parametrize("variant", [0, 1, 2, 4, 8, 0x11, 0x14, 0x18])
@pytest.mark.parametrize("W,H,I,O,s", [
    (56, 56, 64, 64, 1),         # config 1, direct variant
    (56, 56, 128, 256, 1),       # config 3's first layer
    (112, 110, 24, 40, 1), (61, 37, 17, 70, 2), (30, 9, 8, 32, 1), (55, 55, 16, 64, 1), (7, 9, 5, 3, 1), (1, 1, 9, 1, 1),
    (2, 3, 33, 65, 2), (28, 28, 40, 48, 2), (3, 1, 6, 2, 1),
])
def test_conv3x3_direct_mfma(lib, dev, oracle, variant, W, H, I, O, s):
    """The implicit-GEMM 3x3 kernel over the prepared filter bank: oracle (same algorithm, direct order), the
    float64 closed form, and the filter bank's layout itself.  Signed inputs, so every padding sample matters."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    n = lib.drhip_conv3x3_direct_filter_floats(I, O)
    chunks, opad = -(-I // 8), -(-O // 32) * 32
    assert n == 9 * chunks * 8 * opad
    F = dev.empty(n)
    ok(lib, lib.drhip_conv3x3_direct_filter_layout_f32(dev.put(w), F, I, O, None))
    if variant == 0:
        expect = np.zeros((9, chunks, opad, 8), np.float32)       # [tap][c/8][o][pos], pos = (c&1)*4 + (c%8)/2
        for c in range(I):
            expect[:, c // 8, :O, (c & 1) * 4 + (c % 8) // 2] = w[c].reshape(O, 9).T
        assert np.array_equal(dev.get(F, expect.shape), expect)
    want = oracle.conv_direct(x, w, b, (s, s), relu=True)
    out = dev.empty(want.size)
    xd, bd = dev.put(x), dev.put(b)
    ok(lib, lib.drhip_conv3x3_direct_mfma_f32(xd, F, bd, out, W, H, I, O, s, 1, variant, None))
    got = dev.get(out, want.shape)
    assert_close(got, want, terms=9 * I)
    assert_close(got, oracle.conv_f64(x, w, b, stride=(s, s), relu=True), terms=9 * I)
    want2 = oracle.conv_direct(x, w, None, (s, s), relu=False)      # linear, no bias: sign-sensitive
    ok(lib, lib.drhip_conv3x3_direct_mfma_f32(xd, F, None, out, W, H, I, O, s, 0, variant, None))
    assert_close(dev.get(out, want2.shape), want2, terms=9 * I)
    if variant == 0:
        assert lib.drhip_conv3x3_direct_mfma_f32(xd, F, None, out, W, H, I, O, 3, 0, 0, None) == -1      # stride 3
        assert lib.drhip_conv3x3_direct_mfma_f32(xd, F, None, out, W, H, I, O, s, 0, 3, None) == -1      # 3 waves


@pytest.mark.parametrize("variant", [0x21, 0x22, 0x24, 0x28, 0x31, 0x34, 0x38])
@pytest.mark.parametrize("W,H,I,O,s", [
    (28, 28, 128, 192, 2), (31, 33, 72, 97, 2), (1, 1, 5, 1, 1), (2, 3, 33, 65, 2), (17, 1, 6, 16, 1), (3, 11, 130, 31, 1), (9, 7, 24, 33, 2), (16, 2, 8, 15, 1)])
def test_conv3x3_direct_tiles_of_16(lib, dev, oracle, variant, W, H, I, O, s):
    """Tiles of 16 pixels: ragged pixels, channels and stages, and the sums for a global average (the same outputs added up tile by
    tile: 16 of them in fp32, so 16 * 2^-24 of the sum of their magnitudes)."""
    x, w, b = own(I, H, W), own(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), own(O, scale=0.01)
    F = dev.empty(lib.drhip_conv3x3_direct_filter_floats(I, O))
    ok(lib, lib.drhip_conv3x3_direct_filter_layout_f32(dev.put(w), F, I, O, None))
    xd, bd = dev.put(x), dev.put(b)
    for relu, bias in ((1, bd), (0, None)):
        want = oracle.conv_direct(x, w, b if bias else None, (s, s), relu=bool(relu))
        out = dev.empty(want.size)
        ok(lib, lib.drhip_conv3x3_direct_mfma_f32(xd, F, bias, out, W, H, I, O, s, relu, variant, None))
        got = dev.get(out, want.shape)
        assert_close(got, want, terms=9 * I)
        assert_close(got, oracle.conv_f64(x, w, b if bias else None, stride=(s, s), relu=bool(relu)), terms=9 * I)
        flat = got.reshape(O, -1).astype(np.float64)
        tiles = -(-flat.shape[1] // 16)
        flat = np.pad(flat, ((0, 0), (0, 16 * tiles - flat.shape[1]))).reshape(O, tiles, 16)
        parts = dev.empty(tiles * O)
        ok(lib, lib.drhip_conv3x3_direct_poolsum_f32(xd, F, bias, parts, W, H, I, O, s, relu, variant, None))
        assert np.all(np.abs(dev.get(parts, (tiles, O)) - flat.sum(2).T) <= 16 * 2.0 ** -24 * np.abs(flat).sum(2).T)


@pytest.mark.parametrize("variant", [0, 0x100, 0x101, 0x110, 0x111, 0x120, 0x121])
@pytest.mark.parametrize("W,H,I,O,kw,kh,sx,sy", [
    (56, 56, 64, 96, 5, 5, 1, 1), (224, 224, 3, 64, 7, 7, 2, 2), (28, 28, 1, 16, 5, 5, 1, 1), (14, 14, 16, 32, 5, 5, 1, 1),
    (33, 9, 17, 33, 3, 3, 2, 2), (7, 5, 5, 3, 7, 3, 1, 1), (1, 1, 1, 1, 1, 1, 1, 1), (19, 21, 48, 70, 1, 5, 3, 2), (40, 17, 4, 129, 3, 5, 2, 1),
    (9, 70, 40, 24, 1, 1, 2, 2)])
def test_conv_split_bank(lib, dev, oracle, variant, W, H, I, O, kw, kh, sx, sy):
    """Any filter and stride on the bf16 matrix cores, operands split into three parts: every tile and wave split, maps
    smaller than a tile, ragged channel counts on both sides, and the image form (at most 4 input channels).  Held to a
    twentieth of the layer bar: the parts carry all 24 bits."""
    if variant and not lib.drhip_conv_bank_usable(W, H, I, O, kw, kh, sx, sy):
        pytest.skip("not covered")
    x, w, b = rnd(I, H, W), rnd(I, O, kh, kw, scale=(2.0 / (I * kw * kh)) ** 0.5), rnd(O, scale=0.1)
    F = dev.empty(lib.drhip_conv_bank_floats(I, O, kw, kh))
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, kw, kh, None))
    Wo, Ho = W // sx, H // sy
    for relu, bias in ((1, b), (0, None)):
        y = dev.empty(O * Ho * Wo)
        ok(lib, lib.drhip_conv_bank_f32(dev.put(x), F, dev.put(bias) if bias is not None else None, y, W, H, I, O, kw, kh, sx, sy, relu, variant, None))
        want = oracle.conv_direct(x, w, bias, stride=(sx, sy), relu=bool(relu))
        got = dev.get(y, want.shape)
        assert_close(got, want, "split bank")
        assert rel_err(got, want) <= TOL / 20


@pytest.mark.parametrize("variant", [0x100, 0x101, 0x110, 0x111, 0x120, 0x121])
@pytest.mark.parametrize("W,H,I,O,k,s", [(28, 28, 1, 16, 5, 1), (14, 14, 16, 32, 5, 1), (27, 9, 17, 33, 5, 1), (1, 1, 3, 70, 7, 1), (33, 40, 4, 129, 5, 2), (18, 5, 40, 9, 3, 3)])
def test_conv_split_bank_with_maxpool(lib, dev, oracle, variant, W, H, I, O, k, s):
    """The same with a 2x2/2 max pooling behind it: the pooling kernel's results bit for bit, on odd maps (where the pooling counts zeros)
    too; an infinity and a NaN reach what they reach without it."""
    x, w, b = own(I, H, W), own(I, O, k, k, scale=(2.0 / (I * k * k)) ** 0.5), own(O, scale=0.1) - 0.1
    F = dev.empty(lib.drhip_conv_bank_floats(I, O, k, k))
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, k, k, None))
    Wo, Ho, bd = W // s, H // s, dev.put(b)
    full, pooled = dev.empty(O * Ho * Wo), dev.empty(O * -(-Ho // 2) * -(-Wo // 2))
    for relu, extremes in ((1, False), (0, False), (0, True)):
        if extremes:
            x[0, H // 2, W // 2], x[I - 1, 0, 0], x[I // 2, H - 1, W - 1] = np.inf, -np.inf, np.nan
        xd = dev.put(x)
        ok(lib, lib.drhip_conv_bank_f32(xd, F, bd, full, W, H, I, O, k, k, s, s, relu, variant, None))
        ok(lib, lib.drhip_conv_bank_maxpool2_f32(xd, F, bd, pooled, W, H, I, O, k, k, s, s, relu, variant, None))
        two = dev.empty(O * -(-Ho // 2) * -(-Wo // 2))
        ok(lib, lib.drhip_pool_f32(full, two, None, Wo, Ho, O, 2, 2, 1, 2, 2, 1, 0, None))
        got, want = (dev.get(p, (O, -(-Ho // 2), -(-Wo // 2))) for p in (pooled, two))
        if extremes:                        # (the four of such a window are worked out again together, in another order of the sums)
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and not np.isnan(got).any()
            f = np.isfinite(want)
            assert not f.any() or np.all(np.abs(got[f] - want[f]) <= TOL / 20 * np.abs(w).sum((0, 2, 3)).max())
        else:
            assert np.array_equal(got, want)


@pytest.mark.parametrize("variant", [0, 0x121, 0x6111, 0x6121, 0x7111, 0x7121])
@pytest.mark.parametrize("W,H,I,O,k,s", [(112, 96, 3, 64, 7, 2), (35, 41, 4, 33, 5, 1), (17, 13, 20, 129, 3, 2), (8, 6, 1, 5, 5, 1), (9, 7, 16, 32, 3, 1), (1, 1, 2, 3, 7, 1), (50, 3, 70, 20, 5, 2)])
def test_conv_split_bank_with_maxpool3(lib, dev, variant, W, H, I, O, k, s):
    """A layer and the 3x3/2 max pooling behind it in one launch: what the two give apart, around its tiles of 4x3 and 4x4 pooled pixels; without ReLU, so
    that what lies beside the map shows, and with samples that have no parts."""
    x, w, b = own(I, H, W), own(I, O, k, k, scale=np.sqrt(2.0 / (k * k * I))), own(O, scale=0.05)
    Wo, Ho = W // s, H // s
    F = dev.empty(lib.drhip_conv_bank_floats(I, O, k, k))
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, k, k, None))
    full, pooled, two, bd = dev.empty(O * Wo * Ho), dev.empty(O * -(-Ho // 2) * -(-Wo // 2)), dev.empty(O * -(-Ho // 2) * -(-Wo // 2)), dev.put(b)
    for relu, extremes in ((1, False), (0, False), (0, True)):
        if extremes:
            x[0, H // 2, W // 2], x[I - 1, 0, 0], x[I // 2, H - 1, W - 1] = np.inf, -np.inf, np.nan
        xd = dev.put(x)
        ok(lib, lib.drhip_conv_bank_f32(xd, F, bd, full, W, H, I, O, k, k, s, s, relu, variant and variant & 0x130 | 1, None))
        ok(lib, lib.drhip_pool_f32(full, two, None, Wo, Ho, O, 3, 3, 1, 2, 2, 1, 0, None))
        ok(lib, lib.drhip_conv_bank_maxpool3s2_f32(xd, F, bd, pooled, W, H, I, O, k, k, s, s, relu, variant, None))
        got, want = (dev.get(p, (O, -(-Ho // 2), -(-Wo // 2))) for p in (pooled, two))
        if extremes:                        # (worked out again in another order of the sums: an error as of two such sums in fp32)
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]) and not np.isnan(got).any()
            f = np.isfinite(want)
            assert not f.any() or np.all(np.abs(got[f] - want[f]) <= TOL / 20 * np.abs(w).sum((0, 2, 3)).max())
        else:
            assert_close(got, want, terms=I * k * k)
            assert np.array_equal(got, want) or variant == 0 or I > 16      # (otherwise the waves may share the steps another way)


@pytest.mark.parametrize("W,H,I,O,sx,sy", [(224, 224, 3, 64, 2, 2), (33, 31, 3, 9, 2, 2), (17, 13, 1, 5, 1, 1), (20, 18, 4, 70, 1, 2),
                                            (8, 5, 2, 16, 3, 1), (2, 2, 3, 2, 1, 1), (9, 9, 4, 33, 2, 2), (64, 48, 3, 32, 1, 1)])
@pytest.mark.parametrize("relu", [1, 0])
def test_first_layer_conv_with_maxpool(lib, dev, oracle, W, H, I, O, sx, sy, relu):
    """3x3 first-layer convolution + 3x3/2 max pooling in one kernel against the two oracle steps.
    Without ReLU the convolution has negative outputs, so the pooling's zero padding is visible."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.05)
    conv = oracle.conv_direct(x, w, b, (sx, sy), relu=bool(relu))
    want = oracle.pool(conv, (3, 3, 1), (2, 2, 1), 0)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv3x3_pool3s2_f32(dev.put(x), dev.put(w), dev.put(b), out, W, H, I, O, sx, sy, relu, None))
    got = dev.get(out, want.shape)
    assert_close(got, want)
    assert_close(got, oracle.pool_f64(oracle.conv_f64(x, w, b, stride=(sx, sy), relu=bool(relu)), (3, 3, 1), (2, 2, 1), 0))
    # no bias
    want2 = oracle.pool(oracle.conv_direct(x, w, None, (sx, sy), relu=bool(relu)), (3, 3, 1), (2, 2, 1), 0)
    ok(lib, lib.drhip_conv3x3_pool3s2_f32(dev.put(x), dev.put(w), None, out, W, H, I, O, sx, sy, relu, None))
    assert_close(dev.get(out, want2.shape), want2)
    assert lib.drhip_conv3x3_pool3s2_f32(dev.put(x), dev.put(w), None, out, W, H, 5, O, sx, sy, relu, None) == -1


@pytest.mark.parametrize("I", [1, 2, 3, 4])
@pytest.mark.parametrize("W,H,O,sx,sy", [(7, 5, 31, 1, 1), (8, 6, 32, 1, 1), (9, 7, 33, 1, 1), (17, 13, 64, 1, 1), (1, 40, 65, 1, 2), (200, 31, 5, 15, 15), (31, 200, 48, 14, 15)])
def test_first_layer_with_maxpool_tiles(lib, dev, oracle, I, W, H, O, sx, sy):
    """Around its tiles of 4x3 pooled pixels and blocks of 32 and 64 channels, with the longest strides; and an infinite weight, which
    spoils the outputs that its tap reaches and no others."""
    x, w, b = own(I, H, W), own(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), own(O, scale=0.05)
    conv = oracle.conv_direct(x, w, b, (sx, sy), relu=True)
    want = oracle.pool(conv, (3, 3, 1), (2, 2, 1), 0)
    out, xd, bd = dev.empty(want.size), dev.put(x), dev.put(b)
    ok(lib, lib.drhip_conv3x3_pool3s2_f32(xd, dev.put(w), bd, out, W, H, I, O, sx, sy, 1, None))
    got = dev.get(out, want.shape)
    assert_close(got, want, terms=9 * I)
    w[I - 1, O - 1, 1, 1] = np.inf                  # (the middle one: never beside the map)
    ok(lib, lib.drhip_conv3x3_pool3s2_f32(xd, dev.put(w), bd, out, W, H, I, O, sx, sy, 1, None))
    spoilt = dev.get(out, want.shape)
    positive = oracle.pool((x[I - 1:, ::sy, ::sx][:, :conv.shape[1], :conv.shape[2]] > 0).astype(np.float32), (3, 3, 1), (2, 2, 1), 0)[0]
    assert np.array_equal(spoilt[:-1], got[:-1]) and np.array_equal(spoilt[-1], np.where(positive > 0, np.float32(np.inf), np.float32(0)))


def test_conv_direct_valu_kernels(lib, dev, oracle):
    """DR_DIRECT_VALU=1: the LDS-tiled / first-layer VALU kernels behind the matrix-core forms."""
    import os
    os.environ["DR_DIRECT_VALU"] = "1"
    try:
        for (W, H, I, O, s) in [(56, 56, 64, 64, 1), (224, 224, 3, 64, 2), (33, 31, 3, 9, 2), (30, 9, 8, 32, 1)]:
            x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
            want = oracle.conv_direct(x, w, b, (s, s), relu=True)
            out = dev.empty(want.size)
            ok(lib, lib.drhip_conv2d_direct_f32(dev.put(x), dev.put(w), dev.put(b), out, W, H, I, O, 3, 3, s, s, 1, None))
            assert_close(dev.get(out, want.shape), want)
    finally:
        os.environ.pop("DR_DIRECT_VALU", None)


def wino_filters(lib, dev, w):
    I, O = w.shape[:2]
    n = lib.drhip_conv3x3_winograd_filter_floats(I, O)
    U = dev.empty(n)
    ok(lib, lib.drhip_winograd_filter_transform_f32(dev.put(w), U, I, O, None))
    return U, n


def wino_workspace(lib, dev, W, H, I, O, variant):
    n = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, variant)
    if not n:
        return None
    ws = dev.put(np.full(n, np.nan, np.float32))          # poison: nothing may be read before it is written
    if variant & 0x800:                                   # joined splits watch the slots for a marker
        ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    return ws


def test_winograd_filter_transform(lib, dev, oracle):
    I, O = 19, 37
    w = rnd(I, O, 3, 3)
    U, n = wino_filters(lib, dev, w)
    chunks, opad = -(-I // 8), -(-O // 32) * 32
    assert n == 16 * chunks * 8 * opad
    got = dev.get(U, (16, chunks, opad, 8))
    want = oracle.wino_filter(w)                          # reference layout [I,16,O]
    # device layout: [xi][c/8][o][pos], channel c%8 at pos (c&1)*4 + (c%8)/2; c and o zero padded
    expect = np.zeros((16, chunks, opad, 8), np.float32)
    for c in range(I):
        expect[:, c // 8, :O, (c & 1) * 4 + (c % 8) // 2] = want[c]
    assert np.allclose(got, expect, rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("variant", [1, 2, 3, 0x11, 0x21, 0x12, 0x33, 0x101, 0x102, 0x103, 0x111, 0x122,
                                     0x401, 0x402, 0x411, 0x432, 0x501, 0x502, 0x503, 0x512])
@pytest.mark.parametrize("W,H,I,O", [
    (56, 56, 64, 64),        # config 1
    (55, 55, 16, 64),        # fire expand3x3: odd size, two stages of 8 channels
    (28, 28, 24, 40),        # I not a multiple of 8, O not a multiple of 32
    (14, 14, 48, 96), (7, 9, 3, 5), (1, 1, 1, 1), (2, 3, 9, 33), (224, 224, 3, 64),
])
def test_winograd_conv(lib, dev, oracle, variant, W, H, I, O):
    x, w, b = np.abs(rnd(I, H, W)), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    want = oracle.conv_winograd(x, w, b, relu=True)
    floor = float(np.abs(b).max())                    # tiny tensors: the output can be what is left of bias against conv sum
    out = dev.empty(want.size)
    xd, bd = dev.put(x), dev.put(b)
    for _ in range(2):                       # twice: a split layer must leave its counters at zero
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, ws, None))
        got = dev.get(out, want.shape)
        assert_close(got, want, floor=floor)
    truth = oracle.conv_f64(x, w, b, relu=True)
    assert_close(got, truth, floor=floor)
    # linear, no bias (pre-activation values, sign-sensitive)
    want2 = oracle.conv_winograd(x, w, None, relu=False)
    ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, None, out, W, H, I, O, 0, variant, ws, None))
    assert_close(dev.get(out, want2.shape), want2)


@pytest.mark.parametrize("variant", [1, 2, 0x11, 0x22, 0x101, 0x112, 0x401, 0x412, 0x502])
@pytest.mark.parametrize("W,H,I,O", [(56, 56, 64, 64), (28, 12, 24, 40), (2, 2, 1, 1), (224, 224, 3, 64)])
def test_winograd_fused_maxpool(lib, dev, oracle, variant, W, H, I, O):
    """Epilogue flag 2: the kernel stores the 2x2/2 maximum of every output tile -- bit for bit what
    the pooling kernel makes of the kernel's own unpooled output."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    xd, bd = dev.put(x), dev.put(b)
    for relu in (1, 0):
        full = dev.empty(O * H * W)
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, full, W, H, I, O, relu, variant, ws, None))
        want = oracle.pool(dev.get(full, (O, H, W)), (2, 2, 1), (2, 2, 1), 0)
        pooled = dev.empty(want.size)
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, pooled, W, H, I, O, relu | 2, variant, ws, None))
        assert np.array_equal(dev.get(pooled, want.shape), want)
        ref = oracle.pool(oracle.conv_winograd(x, w, b, relu=bool(relu)), (2, 2, 1), (2, 2, 1), 0)
        assert_close(dev.get(pooled, want.shape), ref)
    p = dev.empty(64)
    assert lib.drhip_conv3x3_winograd_f32(p, U, None, p, 3, 4, I, O, 2, 1, None, None) == -1      # odd width
    assert lib.drhip_conv3x3_winograd_f32(p, U, None, p, 4, 4, I, O, 4, 1, None, None) == -1      # unknown flag


@pytest.mark.parametrize("I,k,stride", [(3, 7, 2), (4, 5, 1), (20, 5, 1), (17, 3, 3)])
def test_conv_bank_keeps_infinities(lib, dev, I, k, stride):
    """An infinite sample gives what fp32 arithmetic gives, in the filter's reach and nowhere else."""
    W, H, O = 23, 19, 40
    bank_with_infinities(lib, dev, rnd(I, H, W), rnd(I, O, k, k), stride, 0)


@pytest.mark.parametrize("I", [3, 20])
@pytest.mark.parametrize("variant", [0x100, 0x101, 0x110, 0x111, 0x120, 0x121])
def test_conv_bank_keeps_infinities_in_every_tile(lib, dev, I, variant):
    bank_with_infinities(lib, dev, own(I, 19, 23), own(I, 140, 5, 5), 1, variant)


def bank_with_infinities(lib, dev, x, w, stride, variant):
    (I, H, W), O, k = x.shape, w.shape[1], w.shape[2]
    x[1, 9, 12], x[I - 1, 0, 0], x[0, H - 1, W - 1] = np.inf, -np.inf, np.nan
    F = dev.empty(lib.drhip_conv_bank_floats(I, O, k, k))
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, k, k, None))
    Wo, Ho = W // stride, H // stride
    y = dev.empty(O * Ho * Wo)
    ok(lib, lib.drhip_conv_bank_f32(dev.put(x), F, None, y, W, H, I, O, k, k, stride, stride, 0, variant, None))
    got, want = dev.get(y, (O, Ho, Wo)), np.zeros((O, Ho, Wo))
    pad = np.pad(x.astype(np.float64), ((0, 0), (k // 2, k // 2), (k // 2, k // 2)))
    for oy in range(Ho):
        for ox in range(Wo):
            s = pad[:, oy * stride:oy * stride + k, ox * stride:ox * stride + k]
            want[:, oy, ox] = (w.astype(np.float64) * s[:, None]).sum((0, 2, 3))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isinf(want).any()
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    f = np.isfinite(want)
    assert np.abs(got[f] - want[f]).max() <= TOL / 20 * np.abs(want[f]).max()


SPLIT_HALVES, SPLIT_MIXED = 2 << 12 | 2 << 16, 1 << 12 | 4 << 16 | 1 << 20


@pytest.mark.parametrize("variant", [0x100, 0x101, 0x100 | SPLIT_HALVES, 0x101 | SPLIT_HALVES, 0x101 | 3 << 12 | 3 << 16, 0x101 | SPLIT_MIXED,
                                     0x100 | 3 << 12 | 8 << 16 | 1 << 20])
@pytest.mark.parametrize("W,H,I,O", [(33, 17, 16, 33), (31, 40, 17, 70), (61, 63, 64, 128), (32, 2, 33, 65), (224, 20, 3, 64), (75, 1, 48, 1), (320, 6, 40, 96),
                                     (11, 30, 33, 40), (14, 14, 130, 65), (28, 28, 256, 512), (27, 13, 112, 512), (14, 30, 272, 64)])
def test_winograd_split_operands(lib, dev, oracle, variant, W, H, I, O):
    """Winograd on the bf16 matrix cores, operands split into three parts: ragged channels on both sides, a last step without
    channels, panels over up to six rows of tiles and over the end of the map, one-row maps, the pooling epilogue; input channels in
    equal and ragged pieces that are joined inside the launch, two launches on one workspace.
    Held to a twentieth of the layer bar: the parts carry all 24 bits."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.1)
    F = dev.empty(lib.drhip_conv3x3_winograd_split_filter_floats(I, O))
    ok(lib, lib.drhip_winograd_split_filter_transform_f32(dev.put(w), F, I, O, None))
    xd, bd = dev.put(x), dev.put(b)
    n, ws = lib.drhip_conv3x3_winograd_split_workspace_floats(W, H, I, O, variant), None
    if n == 0 and (variant >> 12 or (W < 31 and variant == 0x100)):     # fewer panels or chunks than the variant needs, or a narrow map: refused
        assert lib.drhip_conv3x3_winograd_split_f32(xd, F, None, dev.empty(O * H * W), W, H, I, O, 0, variant, xd, None) == -1
        pytest.skip("refused, as it has to be")
    if n:
        assert lib.drhip_conv3x3_winograd_split_f32(xd, F, None, dev.empty(O * H * W), W, H, I, O, 0, variant, None, None) == -1      # no workspace
        ws = dev.empty(n)
        ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    for relu, bias in ((1, b), (0, None)):
        y = dev.empty(O * H * W)
        ok(lib, lib.drhip_conv3x3_winograd_split_f32(xd, F, bd if bias is not None else None, y, W, H, I, O, relu, variant, ws, None))
        want = oracle.conv_f64(x, w, bias, relu=bool(relu))
        got = dev.get(y, want.shape)
        assert_close(got, want, "split operands")
        assert rel_err(got, want) <= TOL / 20
        pooled = dev.empty(O * (H // 2) * (W // 2))
        rc = lib.drhip_conv3x3_winograd_split_f32(xd, F, bd if bias is not None else None, pooled, W, H, I, O, relu | 2, variant, ws, None)
        assert rc == (-1 if W % 2 or H % 2 else 0)
        if rc == 0:
            mx = oracle.pool(got, (2, 2, 1), (2, 2, 1), 0)
            assert np.array_equal(dev.get(pooled, mx.shape), mx)
    late = ctypes.c_uint(1)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    assert late.value == 0
    assert lib.drhip_conv3x3_winograd_split_f32(xd, F, None, xd, 10, 4, I, O, 0, variant, ws, None) == -1      # more rows of tiles in a panel than LDS has room for


def winograd_replay(x, w):
    """Winograd F(2x2,3x3) step by step in float64: what fp32 arithmetic makes of infinities and NaN, tile by tile."""
    (I, H, W), O = x.shape, w.shape[1]
    th, tw = -(-H // 2), -(-W // 2)
    pad = np.zeros((I, 2 * th + 2, 2 * tw + 2))
    pad[:, 1:H + 1, 1:W + 1] = x
    d = np.stack([[pad[:, r:r + 2 * th:2, c:c + 2 * tw:2] for c in range(4)] for r in range(4)])       # [4][4][I][th][tw]
    rows = lambda a: np.stack([a[0] - a[2], a[1] + a[2], a[2] - a[1], a[3] - a[1]])
    taps = lambda g: np.stack([g[0], .5 * g[0] + .5 * g[1] + .5 * g[2], .5 * g[0] - .5 * g[1] + .5 * g[2], g[2]])
    y = np.zeros((O, 2 * th, 2 * tw))
    with np.errstate(invalid="ignore"):
        u = np.swapaxes(taps(np.swapaxes(taps(w.astype(np.float64).transpose(2, 3, 0, 1)), 0, 1)), 0, 1)    # [4][4][I][O]
        v = np.swapaxes(rows(np.swapaxes(rows(d), 0, 1)), 0, 1)
        m = np.stack([[sum(u[r, s, c][:, None, None] * v[r, s, c] for c in range(I)) for s in range(4)] for r in range(4)])
        half = np.stack([m[0] + m[1] + m[2], m[1] - m[2] + m[3]])                                       # [2][4][O][th][tw]
        for a in range(2):
            y[:, a::2, 0::2] = half[a, 0] + half[a, 1] + half[a, 2]
            y[:, a::2, 1::2] = half[a, 1] - half[a, 2] + half[a, 3]
    return y[:, :H, :W]


def assert_same_extremes(got, want, by_channel=False):
    """NaN where NaN is wanted, the same infinities, the finite rest within a twentieth of the layer bar: of the ordinary and of the huge
    outputs, or of each output channel's largest."""
    assert np.array_equal(np.isnan(got), np.isnan(want)), np.argwhere(np.isnan(got) != np.isnan(want))[:5]
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    finite = np.isfinite(want)
    for part in finite & (np.arange(len(want))[:, None, None, None] == np.arange(len(want))[:, None, None]) if by_channel else (finite & (np.abs(want) < 1e6), finite & (np.abs(want) >= 1e6)):
        if part.any():
            assert np.abs(got[part] - want[part]).max() <= TOL / 20 * np.abs(want[part]).max()


def split_winograd(lib, dev, x, w, variant, flags=0):
    (I, H, W), O = x.shape, w.shape[1]
    F = dev.empty(lib.drhip_conv3x3_winograd_split_filter_floats(I, O))
    ok(lib, lib.drhip_winograd_split_filter_transform_f32(dev.put(w), F, I, O, None))
    n, ws = lib.drhip_conv3x3_winograd_split_workspace_floats(W, H, I, O, variant), None
    if n:
        ws = dev.empty(n)
        ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    shape = (O, H // 2, W // 2) if flags & 2 else (O, H, W)
    y = dev.empty(O * H * W)
    go = lambda xd: ok(lib, lib.drhip_conv3x3_winograd_split_f32(xd, F, None, y, W, H, I, O, flags, variant, ws, None))
    go(dev.put(x))
    return dev.get(y, shape), go


@pytest.mark.parametrize("variant,W,H,I,O", [(v, W, H, I, O) for v in (0x100, 0x101, 0x100 | SPLIT_HALVES, 0x101 | 3 << 12 | 3 << 16)
                                             for W, H, I, O in ((33, 9, 70, 70), (40, 10, 100, 33))]
                         + [(0x101, 33, 9, 272, 33), (0x101 | SPLIT_HALVES, 28, 9, 100, 70), (0x101 | SPLIT_HALVES, 28, 9, 272, 33)])
def test_winograd_split_keeps_infinities(lib, dev, variant, W, H, I, O):
    """Infinite samples, NaN and samples that bf16 rounds to infinity come out as fp32 Winograd has them, at the edges of the
    map too, where the kernel's loads reach into the next row, with the input channels in pieces, from different channels on and on
    narrow maps."""
    x, w = own(I, H, W), own(I, O, 3, 3, scale=0.02)
    x[1, 4, 12], x[0, 0, 0], x[I - 1, H - 1, W - 1], x[I - 2, 3, 0], x[2, 5, W - 1] = np.inf, -np.inf, np.inf, -np.inf, np.inf
    x[3, 2, 26], x[4, 2, 27], x[2, 6, 20] = np.inf, -np.inf, np.nan
    x[5, 7, 5] = x[I - 1, 1, 22] = 3.399e38
    got, _ = split_winograd(lib, dev, x, w, variant)
    want = winograd_replay(x, w)
    assert np.isinf(want).sum() > O and np.isnan(want).any()
    assert_same_extremes(got, want)
    if H % 2 == 0 and W % 2 == 0:           # ReLU and the pooling epilogue: fmaxf passes a NaN over
        pooled, _ = split_winograd(lib, dev, x, w, variant, flags=3)
        act = np.fmax(got, 0)
        assert np.array_equal(pooled, np.fmax(np.fmax(act[:, ::2, ::2], act[:, ::2, 1::2]), np.fmax(act[:, 1::2, ::2], act[:, 1::2, 1::2])))


@pytest.mark.parametrize("variant", [0x100, 0x101 | SPLIT_HALVES])
@pytest.mark.parametrize("infinite", [True, False])
def test_winograd_split_keeps_extreme_weights(lib, dev, variant, infinite):
    """Filters with an infinite or NaN weight, and finite ones that bf16 rounds to infinity, as fp32 Winograd has them."""
    W, H, I, O = 35, 7, 40, 40
    x, w = own(I, H, W, scale=0.01), own(I, O, 3, 3)
    x[:, 3:5, 4:6] = 0
    if infinite:
        w[1, 3, 0, 0], w[I - 1, 7, 2, 2], w[0, 8, 0, 2], w[1, 8, 0, 0], w[0, 39, 1, 2] = np.inf, -np.inf, np.inf, -np.inf, np.nan
    w[1, 11, 0, 0], w[I - 1, 33, 2, 2] = 3.399e38, -np.finfo(np.float32).max
    got, _ = split_winograd(lib, dev, x, w, variant)
    # (the transforms mix the taps of a filter: the rounding of the largest tap is in every output of its channel)
    assert_same_extremes(got, winograd_replay(x, w), by_channel=True)


@pytest.mark.parametrize("I,k,stride,infinite", [(3, 7, 2, True), (4, 5, 1, True), (20, 5, 1, True), (17, 3, 3, True), (3, 7, 2, False), (20, 5, 1, False)])
def test_conv_bank_keeps_extreme_weights(lib, dev, I, k, stride, infinite):
    """Infinite weights, and finite ones that bf16 rounds to infinity, are what they are in fp32."""
    W, H, O = 23, 19, 40
    x, w = np.abs(own(I, H, W, scale=0.01)), own(I, O, k, k)
    x[:, 3, 4] = 0
    if infinite:
        w[1, 3, 1, 1], w[I - 1, 7, 0, 0], w[0, 8, 0, 0], w[1, 8, 1, 1], w[0, 39, 1, 2] = np.inf, -np.inf, np.inf, -np.inf, np.nan
    w[1, 11, 1, 1], w[I - 1, 33, k - 1, 0] = 3.399e38, -np.finfo(np.float32).max
    F = dev.empty(lib.drhip_conv_bank_floats(I, O, k, k))
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, k, k, None))
    Wo, Ho = W // stride, H // stride
    y = dev.empty(O * Ho * Wo)
    ok(lib, lib.drhip_conv_bank_f32(dev.put(x), F, None, y, W, H, I, O, k, k, stride, stride, 0, 0, None))
    got, want = dev.get(y, (O, Ho, Wo)), np.zeros((O, Ho, Wo))
    for oy in range(Ho):
        for ox in range(Wo):
            ys, xs = np.arange(k) + oy * stride - k // 2, np.arange(k) + ox * stride - k // 2
            j, i = (ys >= 0) & (ys < H), (xs >= 0) & (xs < W)
            with np.errstate(invalid="ignore"):         # (a weight over the edge of the map is not multiplied by anything)
                want[:, oy, ox] = (w.astype(np.float64)[:, :, j][:, :, :, i] * x[:, ys[j]][:, :, xs[i]][:, None]).sum((0, 2, 3))
    assert_same_extremes(got, want)


PAIR = 0x200


def pair_winograd(lib, dev, x, w, variant, flags=0, bias=None):
    """One launch of the kernel of two f16 parts."""
    (I, H, W), O = x.shape, w.shape[1]
    F = dev.empty(lib.drhip_conv3x3_winograd_pair_filter_floats(I, O))
    ok(lib, lib.drhip_winograd_pair_filter_transform_f32(dev.put(w), F, I, O, None))
    n, ws = lib.drhip_conv3x3_winograd_split_workspace_floats(W, H, I, O, variant | PAIR), None
    if n:
        ws = dev.empty(n)
        ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    shape = (O, H // 2, W // 2) if flags & 2 else (O, H, W)
    y, xd = dev.empty(int(np.prod(shape))), dev.put(x)
    for _ in range(2):                      # (twice on one workspace)
        ok(lib, lib.drhip_conv3x3_winograd_split_f32(xd, F, dev.put(bias) if bias is not None else None, y, W, H, I, O, flags, variant | PAIR, ws, None))
    return dev.get(y, shape)


@pytest.mark.parametrize("variant,W,H,I,O", [
    (0x100, 33, 17, 16, 33), (0x101, 31, 40, 17, 70), (0x100, 61, 63, 64, 128), (0x101, 61, 63, 65, 128), (0x100, 32, 2, 33, 65), (0x101, 75, 1, 48, 1),
    (0x100, 224, 20, 3, 64), (0x101, 11, 30, 33, 40), (0x101, 320, 6, 200, 96), (0x101, 28, 28, 256, 512), (0x100 | SPLIT_HALVES, 61, 63, 64, 128),
    (0x101 | SPLIT_HALVES, 28, 28, 256, 512), (0x101 | 3 << 12 | 3 << 16, 27, 14, 112, 200), (0x101 | SPLIT_MIXED, 64, 36, 100, 70),
    (0x100 | 3 << 20 | 1 << 12 | 2 << 16, 64, 36, 130, 70), (0x100 | 4 << 20 | 1 << 12 | 3 << 16, 64, 36, 130, 70),
    (0x100 | 4 << 20 | 1 << 12 | 4 << 16, 63, 36, 200, 70), (0x100 | 3 << 12 | 3 << 16, 61, 20, 79, 65)])
def test_winograd_pair_operands(lib, dev, oracle, variant, W, H, I, O):
    """Winograd on the f16 matrix cores, operands split into two parts: ragged channels, single steps, narrow and one-row maps, pieces, panels that begin
    at different channels, the pooling epilogue.  Held to a twentieth of the layer bar, like three parts."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.1)
    for flags, bias in ((1, b), (0, None)):
        want = oracle.conv_f64(x, w, bias, relu=bool(flags))
        got = pair_winograd(lib, dev, x, w, variant, flags, bias)
        assert_close(got, want, "two parts")
        assert rel_err(got, want) <= TOL / 20
        if W % 2 == 0 and H % 2 == 0:
            assert np.array_equal(pair_winograd(lib, dev, x, w, variant, flags | 2, bias), oracle.pool(got, (2, 2, 1), (2, 2, 1), 0))


@pytest.mark.parametrize("W,H,I,O", [(61, 63, 64, 128), (40, 30, 96, 64), (57, 44, 128, 70), (33, 31, 256, 96), (30, 28, 512, 64)])
def test_winograd_pair_is_as_exact_as_three_parts(lib, dev, oracle, W, H, I, O):
    """From 64 channels on, rms against 64 bits on rectified samples: two parts lose 2^-24 of a product and round the accumulator half as often."""
    x, w = np.maximum(own(I, H, W), 0), own(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I)))
    want = oracle.conv_f64(x, w)
    rms = lambda y: float(np.sqrt(np.mean((y.astype(np.float64) - want) ** 2)))
    assert rms(pair_winograd(lib, dev, x, w, 0x101)) <= rms(split_winograd(lib, dev, x, w, 0x101)[0])


@pytest.mark.parametrize("variant", [0x100, 0x101, 0x101 | SPLIT_HALVES])
@pytest.mark.parametrize("kind", ["rising", "late", "leap", "late leap", "dark", "tiny", "denormal", "huge", "weights", "zero"])
def test_winograd_pair_scales(lib, dev, oracle, kind, variant):
    """Every column of tiles has a scale of its own that follows its largest sample: channels that get larger from step to step, that are zero at first,
    or that leap beyond what the scale has room for, maps of which one side is 2^-30 of the other, samples of any size, output channels of any size."""
    W, H, I, O = 70, 6, 100, 40
    x, w = own(I, H, W), own(I, O, 3, 3, scale=0.1)
    if kind == "rising":                    # (weights that make up for it: what is lost in a channel would show)
        up = np.exp2(np.arange(I) // 4).astype(np.float32)
        x, w = x * up[:, None, None], np.maximum(np.abs(w), 0.05) * np.sign(w)
    elif kind == "late":
        x[:40] = 0
        x[40:90, :, 30:] = 0
        x[40] *= np.float32(2.0 ** -40)
    elif kind in ("leap", "late leap"):     # from one step to the next by more than the scale leaves room for
        x[:40] *= np.float32(2.0 ** -70 if kind == "leap" else 0.0)
        x[40:] *= np.float32(2.0 ** 70)
    elif kind == "dark":
        x[:, :, 35:] *= np.float32(2.0 ** -30)
    elif kind in ("tiny", "denormal", "huge"):
        x = (x * {"tiny": 2.0 ** -100, "denormal": 2.0 ** -140, "huge": 2.0 ** 120}[kind]).astype(np.float32)
        w = w * np.float32(2.0 ** (-20 if kind == "huge" else 20))
    elif kind == "weights":
        w = w * np.exp2(np.arange(O) * 4.0 - 80)[:, None, None].astype(np.float32)
    else:
        x[:] = 0
    want, got = oracle.conv_f64(x, w), pair_winograd(lib, dev, x, w, variant)
    if kind == "dark":                      # (the transforms mix neighbouring tiles' samples: the dark side begins a tile further on)
        assert rel_err(got[:, :, 38:], want[:, :, 38:], floor=0.0) <= TOL / 20
        got, want = got[:, :, :34], want[:, :, :34]
    if kind == "weights":
        for o in range(O):
            assert rel_err(got[o], want[o], floor=0.0) <= TOL / 20, o
    elif kind == "zero":
        assert np.array_equal(got, np.zeros_like(got))
    else:
        assert rel_err(got, want, floor=0.0) <= TOL / 20


@pytest.mark.parametrize("variant,W,H,I,O", [(0x100, 33, 9, 70, 70), (0x100, 40, 10, 70, 70), (0x101, 40, 10, 100, 33), (0x101 | SPLIT_HALVES, 28, 9, 272, 33)])
def test_winograd_pair_keeps_infinities(lib, dev, variant, W, H, I, O):
    """Infinite, NaN and the largest finite samples come out as fp32 Winograd has them, at the edges of the map too."""
    x, w = own(I, H, W), own(I, O, 3, 3, scale=0.02)
    x[1, 4, 12], x[0, 0, 0], x[I - 1, H - 1, W - 1], x[I - 2, 3, 0], x[2, 5, W - 1] = np.inf, -np.inf, np.inf, -np.inf, np.inf
    x[3, 2, 26], x[4, 2, 27], x[2, 6, 20] = np.inf, -np.inf, np.nan
    x[5, 7, 5] = x[I - 1, 1, 22] = 3.399e38
    got, want = pair_winograd(lib, dev, x, w, variant), winograd_replay(x, w)
    assert np.isinf(want).sum() > O and np.isnan(want).any()
    assert_same_extremes(got, want)


@pytest.mark.parametrize("variant", [0x100, 0x101, 0x100 | PAIR, 0x101 | PAIR])
@pytest.mark.parametrize("W,H,I,O", [(40, 10, 70, 33), (36, 17, 64, 65), (64, 1, 64, 70), (72, 34, 65, 128)])
def test_winograd_stores_pairs_of_tiles(lib, dev, oracle, variant, W, H, I, O):
    """Rows of two neighbouring tiles are stored together where they lie on 8 bytes, one tile at a time elsewhere: the same bits, on odd heights, ragged
    channels and part of a panel, with an infinity and a NaN among the samples, and nothing behind the outputs is written."""
    x, w, b = own(I, H, W), own(I, O, 3, 3, scale=0.05), own(O)
    xs = [x, x.copy()]
    xs[1][3, H // 2, 5], xs[1][I - 1, 0, W - 2] = np.inf, np.nan
    kind = "pair" if variant & PAIR else "split"
    F = dev.empty(getattr(lib, "drhip_conv3x3_winograd_%s_filter_floats" % kind)(I, O))
    ok(lib, getattr(lib, "drhip_winograd_%s_filter_transform_f32" % kind)(dev.put(w), F, I, O, None))
    for x in xs:
        for flags in (0, 1, 3):
            if flags & 2 and (W | H) & 1:
                continue
            shape = (O, H // 2, W // 2) if flags & 2 else (O, H, W)
            n, outs = int(np.prod(shape)), []
            for first in (0, 2, 1):                     # on 16 bytes, on 8, on 4
                y = dev.put(np.full(n + 8, 7, np.float32))
                ok(lib, lib.drhip_conv3x3_winograd_split_f32(dev.put(x), F, dev.put(b), ctypes.c_void_p((y.value if hasattr(y, "value") else y) + 4 * first), W, H, I, O, flags, variant, None, None))
                got = dev.get(y, (n + 8,))
                assert np.all(got[:first] == 7) and np.all(got[first + n:] == 7)
                outs.append(got[first:first + n])
            assert np.array_equal(outs[0], outs[2], equal_nan=True) and np.array_equal(outs[1], outs[2], equal_nan=True)


@pytest.mark.parametrize("I,O", [(64, 32), (65, 33), (200, 300), (17, 64), (1, 1), (257, 97)])
def test_a_pair_bank_knows_whether_it_holds_its_weights(lib, dev, I, O):
    """The device tells it of all weights as the host does: at either end of the channels, in chunks that end early, for the first and the last tap, whatever the sign,
    and has the scales that the largest weights ask for."""
    def both(w):
        F, holds = dev.put(np.full(lib.drhip_conv3x3_winograd_pair_filter_floats(I, O), np.nan, np.float32)), ctypes.c_int(-1)
        ok(lib, lib.drhip_winograd_pair_filter_transform_f32(dev.put(w), F, I, O, None))
        ok(lib, lib.drhip_winograd_pair_holds(F, I, O, ctypes.byref(holds), None))
        assert holds.value == lib.drhip_winograd_pair_fits(np.ascontiguousarray(w).ctypes.data_as(ctypes.c_void_p), I, O, 9)
        at = -(-I // 16) * -(-O // 32) * 8192
        scale = dev.get(F, (at + -(-O // 32) * 32,))[at:at + O]
        if np.isfinite(w).all() and (np.abs(w).max(axis=(0, 2, 3)) > 0).all():
            assert np.array_equal(scale, np.exp2(np.floor(np.log2(np.abs(w).max(axis=(0, 2, 3)))) - 13).astype(np.float32))
        return holds.value

    w0 = own(I, O, 3, 3)
    w0[:, :, 1, 1] = np.copysign(np.maximum(np.abs(w0[:, :, 1, 1]), 0.01), w0[:, :, 1, 1])
    assert both(w0) == 1
    for c in {0, I - 1, I // 2}:
        for o in {0, O - 1, O // 2}:
            for value, alone in ((np.inf, 0), (-np.nan, 0), (2.0 ** 101, 0)):
                w = w0.copy()
                w[c, o, 2 * (c & 1), 2 * (o & 1)] = value
                assert both(w) == alone
            for value in (0.0, 2.0 ** -16):
                w = w0.copy()
                w[c, o] = value
                assert both(w) == (I == 1)          # (the only filter of its output channel is the largest)
    assert both(w0 * np.float32(2.0 ** -99 * 2.0 ** -10)) == 0
    w = w0.copy()
    w[:, O // 2] = 0
    assert both(w) == 1


@pytest.mark.parametrize("operand,power", [(o, p) for o in ("samples", "weights") for p in (-146, -136, -126, -112, -60, 60, 100, 116, 124)])
def test_split_kernels_hold_operands_of_any_size(lib, dev, oracle, operand, power):
    """Samples and weights down to the smallest fp32 number keep all their bits, and what is too large for three parts once it is scaled, the
    results included, is worked out in fp32."""
    W, H, I, O = 23, 9, 20, 40
    other = 2.0 ** (20 if power < 0 else -20)                       # results that fp32 has 24 bits for
    scaled = lambda a, on: (a.astype(np.float64) * (2.0 ** power if on else other)).astype(np.float32)
    x = scaled(own(I, H, W), operand == "samples")
    for k in (3, 5):
        w = scaled(own(I, O, k, k), operand == "weights")
        F, y = dev.empty(lib.drhip_conv_bank_floats(I, O, k, k)), dev.empty(O * H * W)
        ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, k, k, None))
        ok(lib, lib.drhip_conv_bank_f32(dev.put(x), F, None, y, W, H, I, O, k, k, 1, 1, 0, 0, None))
        want = oracle.conv_f64(x, w)
        assert rel_err(dev.get(y, want.shape), want, floor=0.0) <= TOL / 20, k
        if k == 3 and (operand == "samples" or power >= -126):      # (fp32 has no bits left for the transform of smaller filters)
            for variant in (0x101, 0x101 | SPLIT_HALVES):
                assert rel_err(split_winograd(lib, dev, x, w, variant)[0], want, floor=0.0) <= TOL / 20, hex(variant)


def kernel_us(lib, go, arg, repeats=5):
    """Shortest execution time of the kernels that go(arg) launches."""
    best = 1e30
    for _ in range(repeats):
        ms, count = (ctypes.c_float * 64)(), ctypes.c_int()
        ok(lib, lib.drhip_timing_begin())
        go(arg)
        ok(lib, lib.drhip_timing_end(ms, 64, ctypes.byref(count)))
        assert count.value
        best = min(best, 1e3 * sum(ms[:count.value]))
    return best


def test_a_sample_that_is_nan_does_not_hold_a_launch_up(lib, dev):
    """What the split-operand kernels do about outputs that came out as NaN is work for whole waves, and none where a sample is NaN: such
    a launch takes a multiple of its time, not milliseconds."""
    W, H, I, O = 56, 56, 64, 96
    x, w = own(I, H, W), own(I, O, 5, 5, scale=0.05)
    bad = x.copy()
    bad[10, 20, 30] = np.nan
    bad[11, 40, 9] = np.inf
    F, y = dev.empty(lib.drhip_conv_bank_floats(I, O, 5, 5)), dev.empty(O * H * W)
    ok(lib, lib.drhip_conv_bank_layout_f32(dev.put(w), F, I, O, 5, 5, None))
    bank = lambda xd: ok(lib, lib.drhip_conv_bank_f32(xd, F, None, y, W, H, I, O, 5, 5, 1, 1, 0, 0, None))
    _, wino = split_winograd(lib, dev, x, own(I, O, 3, 3, scale=0.05), 0x101)
    for what, go in (("bank", bank), ("winograd", wino)):
        good, worse, none = [kernel_us(lib, go, dev.put(a)) for a in (x, bad, np.full_like(x, np.nan))]
        print("%s: %.1f us, with a NaN and an infinity %.1f us, all NaN %.1f us" % (what, good, worse, none))
        assert worse <= 40 * good and none <= 20 * good     # (by one lane each: 160 times)


@pytest.mark.parametrize("nA,sA,sB", [(1, 1, 2), (1, 2, 1), (1, 2, 2), (2, 1, 2), (0, 1, 2), (1, 4, 3), (1, 1, 4), (1, 3, 1)])
def test_winograd_split_stays_inside_its_workspace(lib, dev, oracle, nA, sA, sB):
    """Whole panels in front of cut ones, behind them, and pieces of two sizes: the result, every slot left with its marker, and
    nothing written behind the workspace."""
    W, H, I, O = 64, 36, 100, 70
    variant = (0x101 if max(sA, sB) > 2 else 0x100) | nA << 20 | sA << 12 | sB << 16
    x, w = own(I, H, W), own(I, O, 3, 3, scale=0.05)
    n, guard = lib.drhip_conv3x3_winograd_split_workspace_floats(W, H, I, O, variant), 1 << 16
    F, ws, y, xd = dev.empty(lib.drhip_conv3x3_winograd_split_filter_floats(I, O)), dev.empty(n + guard), dev.empty(O * H * W), dev.put(x)
    ok(lib, lib.drhip_winograd_split_filter_transform_f32(dev.put(w), F, I, O, None))
    ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    want = oracle.conv_f64(x, w)
    for _ in range(2):
        ok(lib, lib.drhip_conv3x3_winograd_split_f32(xd, F, None, y, W, H, I, O, 0, variant, ws, None))
        assert rel_err(dev.get(y, want.shape), want) <= TOL / 20
        left = dev.get(ws, (n + guard,))
        assert np.all(left[:n].view(np.uint32) == 0xffa5c3e1) and np.all(left[n:] == -777)


@pytest.mark.parametrize("W,H,I,O", [(257, 129, 113, 65), (21, 48, 400, 512), (33, 31, 256, 512)])
def test_winograd_split_picked(lib, dev, oracle, W, H, I, O):
    """The variant that the rule picks: a round of whole panels and halves behind it, narrow and wide maps in pieces, panels
    that begin at different channels."""
    variant = lib.drhip_conv3x3_winograd_split_pick_variant(W, H, I, O)
    n = lib.drhip_conv3x3_winograd_split_workspace_floats(W, H, I, O, variant)
    assert variant >> 12 and n
    x, w = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I)))
    F, ws, y, xd = dev.empty(lib.drhip_conv3x3_winograd_split_filter_floats(I, O)), dev.empty(n), dev.empty(O * H * W), dev.put(x)
    ok(lib, lib.drhip_winograd_split_filter_transform_f32(dev.put(w), F, I, O, None))
    ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    want = oracle.conv_f64(x, w, None, relu=False)
    for _ in range(3):
        ok(lib, lib.drhip_conv3x3_winograd_split_f32(xd, F, None, y, W, H, I, O, 0, variant, ws, None))
        assert rel_err(dev.get(y, want.shape), want) <= TOL / 20


@pytest.mark.parametrize("variant", [0x811, 0x812, 0x821, 0x831, 0xc11, 0xc12, 0xc21, 0xc22, 0xc31])
@pytest.mark.parametrize("W,H,I,O", [
    (56, 56, 64, 64), (14, 14, 64, 96), (28, 20, 32, 40), (13, 9, 16, 33), (2, 2, 128, 3), (14, 14, 512, 512),
])
def test_winograd_joined_splits(lib, dev, oracle, variant, W, H, I, O):
    """Variant bit 0x800: the splits of a panel add their partial tiles up inside the one launch.  Same sums in the
    same order as the two-kernel form, so the results must be bit-identical to it; the workspace must be left
    holding the marker again; several launches in a row; the pooling epilogue."""
    chunks = -(-I // 8)
    per_split = -(-chunks // min(1 << ((variant >> 4) & 0xf), chunks))
    splits = -(-chunks // per_split)                      # what the launcher makes of the request: no empty split
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    xd, bd = dev.put(x), dev.put(b)
    out = dev.empty(O * H * W)
    n = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, variant)
    nt, two_sets = variant & 0xf, bool(variant & 0x400)
    groups = -(-(-(-W // 2) * -(-H // 2)) // 32) * -(-O // (32 * nt)) * splits
    resident = groups <= 256 * (1 if two_sets else {1: 3, 2: 2}[nt])     # MI355X: 256 CUs
    if splits * per_split != chunks or splits & (splits - 1) or not resident:     # unequal splits, or more workgroups than fit at once: refused
        assert n > 0
        assert lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, dev.empty(n), None) == -1
        return
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    plain = variant & ~0x800
    ws2 = wino_workspace(lib, dev, W, H, I, O, plain)
    ref = dev.empty(O * H * W)
    ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, ref, W, H, I, O, 1, plain, ws2, None))
    want = dev.get(ref, (O, H, W))
    assert_close(want, oracle.conv_winograd(x, w, b, relu=True), floor=float(np.abs(b).max()))
    for _ in range(3):
        ok(lib, lib.drhip_fill_f32(out, 7.0, O * H * W, None))
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, ws, None))
        assert np.array_equal(dev.get(out, want.shape), want)
        assert np.all(dev.get(ws, (n,)).view(np.uint32) == 0xffa5c3e1)
    if W % 2 == 0 and H % 2 == 0:
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, ref, W, H, I, O, 2, plain, ws2, None))
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 2, variant, ws, None))
        assert np.array_equal(dev.get(out, (O, H // 2, W // 2)), dev.get(ref, (O, H // 2, W // 2)))
    late = ctypes.c_uint(123)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    assert late.value == 0


def test_winograd_joined_refused_when_not_resident(lib, dev):
    """A joined split needs every workgroup of the launch resident at once; a layer with more panels is refused."""
    p = dev.empty(64)
    n = lib.drhip_conv3x3_winograd_workspace_floats(224, 224, 16, 64, 0x811)
    assert n > 0
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 224, 224, 16, 64, 0, 0x811, p, None) == -1
    assert b"resident" in lib.drhip_last_error()
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 8, 8, 16, 16, 0, 0x801, p, None) == -1     # joined, but unsplit
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 8, 8, 16, 16, 0, 0x911, p, None) == -1     # 16-tile blocks


@pytest.mark.parametrize("variant", [0x1801, 0x1802])
@pytest.mark.parametrize("W,H,I,O", [
    (112, 112, 128, 128),    # 49 panels per XCD: one cut into 16, 16 halved, 32 whole
    (112, 112, 64, 128),     # 8 stages: the finest cut is 8
    (56, 56, 64, 64), (28, 20, 32, 40), (13, 9, 16, 33), (2, 2, 128, 3), (14, 14, 512, 512),
    (28, 28, 24, 40),        # 3 stages: nothing to halve, the launch stays unsplit
    (7, 9, 3, 5),
])
def test_winograd_tiered_splits(lib, dev, oracle, variant, W, H, I, O):
    """Variant bits 0x1800: the panels of an XCD go out in tiers of whole, halved, quartered ... panels whose pieces
    add their partial tiles up inside the launch.  Against the oracle; repeated launches bit-identical; the
    workspace left holding the marker; the pooling epilogue equal to the pooled unpooled output."""
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    xd, bd = dev.put(x), dev.put(b)
    out = dev.empty(O * H * W)
    n = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, variant)
    chunks = -(-I // 8)
    assert (n > 0) == (chunks % 2 == 0)
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    want = oracle.conv_winograd(x, w, b, relu=True)
    first = None
    for _ in range(3):
        ok(lib, lib.drhip_fill_f32(out, 7.0, O * H * W, None))
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, ws, None))
        got = dev.get(out, want.shape)
        assert_close(got, want, floor=float(np.abs(b).max()))
        first = got if first is None else first
        assert np.array_equal(got, first)
        if n:
            assert np.all(dev.get(ws, (n,)).view(np.uint32) == 0xffa5c3e1)
    assert_close(first, oracle.conv_f64(x, w, b, relu=True), floor=float(np.abs(b).max()))
    if W % 2 == 0 and H % 2 == 0:
        pooled = dev.empty(O * H * W // 4)
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, pooled, W, H, I, O, 1 | 2, variant, ws, None))
        assert np.array_equal(dev.get(pooled, (O, H // 2, W // 2)), oracle.pool(first, (2, 2, 1), (2, 2, 1), 0))
    late = ctypes.c_uint(123)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    assert late.value == 0
    if n:       # the pieces wait for each other through the workspace: none offered, refused
        assert lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, None, None) == -1


@pytest.mark.parametrize("W,H,I,O", [
    (8, 8, 64, 32),          # one panel: its XCD has 31 helpers for it
    (9, 7, 67, 40), (13, 9, 130, 33), (2, 2, 128, 300),     # ragged tiles, channels and outputs
    (64, 40, 128, 224),      # 140 panels, two of an XCD's 18 for most of its 14 helpers
    (52, 52, 250, 256),      # 176: three each
    (56, 56, 256, 256),      # 200: four, the last XCD has none of its own in part
])
def test_winograd_helpers(lib, dev, oracle, W, H, I, O):
    """Variant 0x2c01: CUs without a panel take the last stages of the others' panels.  As for the tiered splits."""
    variant = 0x2c01
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    xd, bd = dev.put(x), dev.put(b)
    out = dev.empty(O * H * W)
    n = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, variant)
    assert n == -(-(-(-W // 2) * -(-H // 2)) // 32) * -(-O // 32) * 4096
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    want = oracle.conv_winograd(x, w, b, relu=True)
    first = None
    for _ in range(3):
        ok(lib, lib.drhip_fill_f32(out, 7.0, O * H * W, None))
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, ws, None))
        got = dev.get(out, want.shape)
        assert_close(got, want, floor=float(np.abs(b).max()))
        first = got if first is None else first
        assert np.array_equal(got, first)
        assert np.all(dev.get(ws, (n,)).view(np.uint32) == 0xffa5c3e1)
    assert_close(first, oracle.conv_f64(x, w, b, relu=True), floor=float(np.abs(b).max()))
    if W % 2 == 0 and H % 2 == 0:
        pooled = dev.empty(O * H * W // 4)
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, bd, pooled, W, H, I, O, 1 | 2, variant, ws, None))
        assert np.array_equal(dev.get(pooled, (O, H // 2, W // 2)), oracle.pool(first, (2, 2, 1), (2, 2, 1), 0))
    ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, None, out, W, H, I, O, 0, variant, ws, None))
    assert_close(dev.get(out, want.shape), oracle.conv_winograd(x, w, None, relu=False))
    late = ctypes.c_uint(123)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    assert late.value == 0
    assert lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, W, H, I, O, 1, variant, None, None) == -1
    # too short to share, or more panels than one round of the CUs: refused
    for shape in ((W, H, 24, O), (112, 112, 256, 256)):
        assert lib.drhip_conv3x3_winograd_workspace_floats(*shape, variant) == 0
        assert lib.drhip_conv3x3_winograd_f32(xd, U, bd, out, *shape, 1, variant, ws, None) == -1


@pytest.mark.parametrize("variant", [0x2c01, 0xc11, 0x821, 0x1801])
def test_winograd_joins_keep_infinities(lib, dev, variant):
    """Infinities and NaN in the share of the one, of the other and of both whose sums are joined (with helpers the first 64 channels are the panel's
    own): what fp32 Winograd makes of them, also of a NaN that looks like the marker of a tile that has not arrived, and the next launch sees nothing
    of it.  (Not in the columns at the edge, whose samples the kernel multiplies by zero for their neighbours.)"""
    W, H, I, O = 13, 9, 128, 33
    x, w = own(I, H, W), own(I, O, 3, 3, scale=0.02)
    spoilt = x.copy()
    spoilt[3, 4, 4], spoilt[100, 4, 4], spoilt[5, 1, 7], spoilt[127, 6, 9], spoilt[70, 7, 3] = np.inf, -np.inf, np.inf, np.inf, np.nan
    spoilt.view(np.uint32)[[9, 90, 126], 2, 10] = 0xffa5c3e1
    U, _ = wino_filters(lib, dev, w)
    n, y = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, variant), dev.empty(O * H * W)
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    for a in (x, spoilt, x, spoilt):
        ok(lib, lib.drhip_conv3x3_winograd_f32(dev.put(a), U, None, y, W, H, I, O, 0, variant, ws, None))
        with np.errstate(invalid="ignore"):
            got, want = dev.get(y, (O, H, W)), winograd_replay(a, w)
        assert np.isnan(want).any() == np.isinf(want).any() == (a is spoilt)
        assert_same_extremes(got, want)
        assert np.all(dev.get(ws, (n,)).view(np.uint32) == 0xffa5c3e1)
    late = ctypes.c_uint(123)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    assert late.value == 0


def test_winograd_tiered_refused_combinations(lib, dev):
    p = dev.empty(64)
    # not joined, 16-tile blocks, two wave sets, split bits, 128 channels; helpers with one wave set, 64 channels, split bits, not joined, in tiers; an unknown bit
    for variant in (0x1001, 0x1901, 0x1c01, 0x1811, 0x1803, 0x2801, 0x2c02, 0x2c11, 0x2001, 0x3c01, 0x4801, 0x4c01):
        assert lib.drhip_conv3x3_winograd_workspace_floats(8, 8, 16, 16, variant) == 0
        assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 8, 8, 16, 16, 0, variant, p, None) == -1, hex(variant)


def test_winograd_auto_variant_vgg_shapes(lib, dev, oracle):
    assert lib.drhip_conv3x3_winograd_pick_variant(112, 112, 128, 128) == 0x1801      # (MI355X: 32 CUs per XCD)
    assert lib.drhip_conv3x3_winograd_pick_variant(14, 14, 512, 512) == 0x831
    assert lib.drhip_conv3x3_winograd_pick_variant(224, 224, 3, 64) == 1           # an image layer: 32-channel blocks
    assert lib.drhip_conv3x3_winograd_pick_variant(224, 224, 64, 64) == 2
    for (W, I, O) in [(224, 3, 64), (224, 64, 64), (112, 128, 128), (56, 128, 256), (28, 256, 512), (14, 512, 512)]:
        x, w, b = np.abs(rnd(I, W, W)), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
        U, _ = wino_filters(lib, dev, w)
        variant = lib.drhip_conv3x3_winograd_pick_variant(W, W, I, O)
        ws = wino_workspace(lib, dev, W, W, I, O, variant)
        want = oracle.conv_winograd(x, w, b, relu=True)
        out = dev.empty(want.size)
        ok(lib, lib.drhip_conv3x3_winograd_f32(dev.put(x), U, dev.put(b), out, W, W, I, O, 1, variant, ws, None))
        assert_close(dev.get(out, want.shape), want)
        # variant 0 without a workspace falls back to an unsplit configuration
        ok(lib, lib.drhip_conv3x3_winograd_f32(dev.put(x), U, dev.put(b), out, W, W, I, O, 1, 0, None, None))
        assert_close(dev.get(out, want.shape), want)
        dev.close()


@pytest.mark.parametrize("W,H,I,O,split,whole", [
    (34, 32, 128, 256, 0x101, 0x101), (20, 123, 124, 117, 0x101, 0x101),       # the 16-tile form, which joined halves beat and halves in two launches do not
    (36, 36, 256, 96, 0x421, 0x401), (28, 28, 512, 512, 0x411, 0x401), (48, 48, 256, 256, 0x401, 0x401), (112, 112, 128, 128, 1, 1)])
def test_winograd_variant_0_joins_nothing(lib, dev, W, H, I, O, split, whole):
    """Variant 0 takes the best form without joins, with a workspace (that of the picked variant is enough) or without: the same bits."""
    U, _ = wino_filters(lib, dev, own(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))))
    xd, y = dev.put(own(I, H, W)), dev.empty(O * H * W)
    n = lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, lib.drhip_conv3x3_winograd_pick_variant(W, H, I, O))
    assert lib.drhip_conv3x3_winograd_workspace_floats(W, H, I, O, split) <= n
    ws = dev.empty(max(n, 1))

    def run(variant, workspace):
        ok(lib, lib.drhip_conv3x3_winograd_f32(xd, U, None, y, W, H, I, O, 0, variant, workspace, None))
        return dev.get(y, (O, H, W))

    assert np.array_equal(run(0, ws), run(split, ws)) and np.array_equal(run(0, None), run(whole, None))


def test_winograd_rejects_bad_arguments(lib, dev):
    p = dev.empty(64)
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 0, 4, 1, 1, 0, 0, None, None) == -1
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 4, 4, 1, 1, 0, 9, None, None) == -1
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 4, 4, 1, 1, 0, 4, None, None) == -1      # panel codes are 1..3
    assert lib.drhip_conv3x3_winograd_f32(None, p, None, p, 4, 4, 1, 1, 0, 0, None, None) == -1
    assert lib.drhip_conv3x3_winograd_f32(p, p, None, p, 4, 4, 32, 1, 0, 0x11, None, None) == -1    # split without workspace
    assert b"workspace" in lib.drhip_last_error()


@pytest.mark.parametrize("variant", [0, 1, 2, 4, 8, 0x101, 0x102, 0x108, 0x110])
@pytest.mark.parametrize("P,I,O", [(3025, 128, 16), (3025, 16, 64), (196, 512, 1000), (196, 512, 64), (784, 256, 32), (50, 7, 5), (1, 1, 1), (33, 9, 65), (70, 24, 40)])
def test_conv1x1(lib, dev, oracle, variant, P, I, O):
    x, w, b = np.abs(rnd(I, 1, P)), rnd(I, O, 1, 1, scale=np.sqrt(2.0 / I)), rnd(O, scale=0.01)
    want = oracle.conv1x1(x, w, b, relu=True)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv1x1_f32(dev.put(x), dev.put(w), dev.put(b), out, P, I, O, 1, variant, None))
    assert_close(dev.get(out, want.shape), want)
    want2 = oracle.conv1x1(x, w, None, relu=False)
    ok(lib, lib.drhip_conv1x1_f32(dev.put(x), dev.put(w), None, out, P, I, O, 0, variant, None))
    assert_close(dev.get(out, want2.shape), want2)


@pytest.mark.parametrize("W,H,C,k,s", [(56, 56, 256, 2, 2), (112, 112, 64, 3, 2), (55, 55, 7, 3, 2), (14, 14, 1000, 14, 14), (9, 7, 3, 2, 3), (5, 5, 2, 5, 1),
                                         (13, 13, 5, 8, 8), (20, 17, 3, 9, 4), (30, 30, 2, 16, 16)])   # >= 64 samples: one wavefront per output
def test_pool_bit_exact(lib, dev, oracle, W, H, C, k, s):
    x = rnd(C, H, W)                     # signed values: the zero padding is observable
    x[:, ::3, ::2] = x[0, 0, 0]          # ties: the first maximum in scan order must win
    for kind in (0, 1):
        want, warg = oracle.pool(x, (k, k, 1), (s, s, 1), kind, want_argmax=True) if kind == 0 else (oracle.pool(x, (k, k, 1), (s, s, 1), kind), None)
        out = dev.empty(want.size)
        arg = dev.empty(want.size, np.int32) if kind == 0 else None
        ok(lib, lib.drhip_pool_f32(dev.put(x), out, arg, W, H, C, k, k, 1, s, s, 1, kind, None))
        got = dev.get(out, want.shape)
        if kind == 0:
            assert np.array_equal(got, want)                                   # values bit-exact
            assert np.array_equal(dev.get(arg, want.shape, np.int32), warg)    # max-indices bit-exact
        else:
            assert rel_err(got, want) <= 1e-6


def test_pool_depth_window(lib, dev, oracle):
    x = rnd(6, 5, 4)
    want = oracle.pool(x, (2, 2, 2), (2, 2, 2), 0)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_pool_f32(dev.put(x), out, None, 4, 5, 6, 2, 2, 2, 2, 2, 2, 0, None))
    assert np.array_equal(dev.get(out, want.shape), want)


@pytest.mark.parametrize("C,H,W,N,relu", [(512, 7, 7, 4096, 1), (4096, 1, 1, 1000, 0), (16, 3, 5, 10, 1), (3, 2, 2, 7, 0), (64, 1, 1, 130, 1), (1, 1, 1, 1, 0)])
def test_fc(lib, dev, oracle, C, H, W, N, relu):
    K = C * H * W
    x, Wt, b = np.abs(rnd(C, H, W)), rnd(K, N, scale=np.sqrt(2.0 / K)), rnd(N, scale=0.01)
    want = oracle.fc(x, Wt, b, relu=bool(relu)).reshape(-1)
    truth = oracle.fc_f64(x, Wt, b, relu=bool(relu)).reshape(-1)
    raw, perm = dev.put(Wt), dev.empty(K * N)
    ok(lib, lib.drhip_fc_permute_rows_f32(raw, perm, W, H, C, N, None))
    nparts = lib.drhip_fc_scratch_floats(K, N)
    parts = dev.empty(nparts) if nparts else None
    y = dev.empty(N)
    xd, bd = dev.put(x), dev.put(b)
    first = None
    for _ in range(2):                     # the scratch needs no reset between calls
        ok(lib, lib.drhip_fc_f32(xd, perm, bd, y, parts, K, N, relu, None))
        got = dev.get(y, (N,))
        assert_close(got, want, terms=K)
        assert_close(got, truth, terms=K)
        assert first is None or np.array_equal(first, got)      # fixed summation order
        first = got


@pytest.mark.parametrize("Win,Hin,I,O", [(56, 56, 128, 32), (28, 28, 256, 48), (55, 27, 20, 7), (9, 6, 3, 17), (2, 2, 1, 1), (1, 1, 5, 3)])
def test_conv1x1_with_pooled_input(lib, dev, oracle, Win, Hin, I, O):
    """3x3/2 max pooling taken while the 1x1 layer loads its input: the same values as the pooling kernel
    followed by the 1x1 GEMM (to rounding: the channel sum may be dealt to a different number of waves),
    and the oracle's pool -> conv1x1 within the layer bar.
    Signed inputs: windows hanging over the border must see 0.0, not -inf and not the edge sample."""
    x, w, b = rnd(I, Hin, Win), rnd(I, O, 1, 1, scale=np.sqrt(2.0 / I)), rnd(O, scale=0.01)
    Wp, Hp = -(-Win // 2), -(-Hin // 2)
    pooled = oracle.pool(x, (3, 3, 1), (2, 2, 1), 0)
    assert pooled.shape == (I, Hp, Wp)
    xd, wd, bd = dev.put(x), dev.put(w), dev.put(b)
    for relu in (1, 0):
        want = oracle.conv1x1(pooled, w, b, relu=bool(relu))
        out = dev.empty(want.size)
        ok(lib, lib.drhip_conv1x1_pooled3s2_f32(xd, wd, bd, out, Win, Hin, I, O, relu, None))
        got = dev.get(out, want.shape)
        assert_close(got, want, "pooled-input 1x1 %dx%dx%d->%d" % (Win, Hin, I, O))
        # against the two kernels it replaces
        mid, two = dev.empty(pooled.size), dev.empty(want.size)
        ok(lib, lib.drhip_pool_f32(xd, mid, None, Win, Hin, I, 3, 3, 1, 2, 2, 1, 0, None))
        assert np.array_equal(dev.get(mid, pooled.shape), pooled)
        ok(lib, lib.drhip_conv1x1_f32(mid, wd, bd, two, Wp * Hp, I, O, relu, 0, None))
        assert_close(got, dev.get(two, want.shape), "pooled-input 1x1 vs pool + 1x1 kernels")
    assert lib.drhip_conv1x1_pooled3s2_f32(xd, wd, bd, None, Win, Hin, I, O, 0, None) == -1


class DeferredVec(ctypes.Structure):
    """drhip_deferred_vec (include/dr_hip.h)."""
    _fields_ = [("partials", ctypes.c_void_p), ("bias", ctypes.c_void_p), ("slices", ctypes.c_int), ("n", ctypes.c_int), ("relu", ctypes.c_int), ("finished", ctypes.c_void_p),
                ("divisor", ctypes.c_float)]


@pytest.mark.parametrize("N2", [1000, 2500])        # softmax with the vector in registers / re-read from memory
def test_fc_chain_without_finishing_kernels(lib, dev, oracle, N2):
    """FC -> FC -> softmax where each consumer sums the producer's split-K partials itself: every
    result equals the one of the three separate calls bit for bit."""
    K, N1 = 1024, 2048
    x, W1, b1 = np.abs(rnd(K)), rnd(K, N1, scale=np.sqrt(2.0 / K)), rnd(N1, scale=0.01)
    W2, b2 = rnd(N1, N2, scale=np.sqrt(2.0 / N1)), rnd(N2, scale=0.01)
    xd, W1d, b1d, W2d, b2d = dev.put(x), dev.put(W1), dev.put(b1), dev.put(W2), dev.put(b2)
    s1, s2 = lib.drhip_fc_slices(K, N1), lib.drhip_fc_slices(N1, N2)
    assert s1 > 1 and s2 > 1 and lib.drhip_fc_scratch_floats(K, N1) == s1 * N1
    p1, p2 = dev.empty(s1 * N1), dev.empty(s2 * N2)
    y1, y2, prob = dev.empty(N1), dev.empty(N2), dev.empty(N2)
    # plain chain
    ok(lib, lib.drhip_fc_f32(xd, W1d, b1d, y1, p1, K, N1, 1, None))
    ok(lib, lib.drhip_fc_f32(y1, W2d, b2d, y2, p2, N1, N2, 0, None))
    ok(lib, lib.drhip_softmax_f32(y2, prob, N2, None))
    want1, want2, wantp = dev.get(y1, (N1,)), dev.get(y2, (N2,)), dev.get(prob, (N2,))
    assert_close(want2, oracle.fc(oracle.fc(x.reshape(K, 1, 1), W1, b1, relu=True), W2, b2, relu=False).reshape(-1))
    # deferred chain: y1 and y2 are never written
    q1, q2, prob2 = dev.empty(s1 * N1), dev.empty(s2 * N2), dev.empty(N2)
    ok(lib, lib.drhip_fc_ex_f32(xd, None, W1d, b1d, None, q1, K, N1, 1, 1, None))
    d1 = DeferredVec(q1.value, b1d.value, s1, N1, 1, None)
    y2b = dev.empty(N2)
    ok(lib, lib.drhip_fc_ex_f32(None, ctypes.byref(d1), W2d, b2d, y2b, q2, N1, N2, 0, 0, None))
    assert np.array_equal(dev.get(y2b, (N2,)), want2)
    ok(lib, lib.drhip_fc_ex_f32(None, ctypes.byref(d1), W2d, b2d, None, q2, N1, N2, 0, 1, None))
    d2 = DeferredVec(q2.value, b2d.value, s2, N2, 0, None)
    ok(lib, lib.drhip_softmax_ex_f32(None, ctypes.byref(d2), prob2, N2, None))
    assert np.array_equal(dev.get(prob2, (N2,)), wantp)
    # ... and with the consumers also storing the finished vectors (producers whose output is wanted too)
    fin1, fin2 = dev.put(np.full(N1, -7.0, np.float32)), dev.put(np.full(N2, -7.0, np.float32))
    d1f = DeferredVec(q1.value, b1d.value, s1, N1, 1, fin1.value)
    ok(lib, lib.drhip_fc_ex_f32(None, ctypes.byref(d1f), W2d, b2d, None, q2, N1, N2, 0, 1, None))
    assert np.array_equal(dev.get(fin1, (N1,)), want1)
    d2f = DeferredVec(q2.value, b2d.value, s2, N2, 0, fin2.value)
    ok(lib, lib.drhip_softmax_ex_f32(None, ctypes.byref(d2f), prob2, N2, None))
    assert np.array_equal(dev.get(prob2, (N2,)), wantp) and np.array_equal(dev.get(fin2, (N2,)), want2)
    d2bad = DeferredVec(q2.value, b2d.value, s2, N2, 0, prob2.value)
    assert lib.drhip_softmax_ex_f32(None, ctypes.byref(d2bad), prob2, N2, None) == -1
    # argument checks
    bad = DeferredVec(q1.value, b1d.value, s1, N1 + 1, 1, None)
    assert lib.drhip_fc_ex_f32(None, ctypes.byref(bad), W2d, b2d, y2b, q2, N1, N2, 0, 0, None) == -1
    assert lib.drhip_fc_ex_f32(xd, None, W1d, b1d, None, None, 64, 8, 0, 1, None) == -1        # unsplit layers cannot defer


@pytest.mark.parametrize("P,I,O,relu", [(196, 512, 1000, 1), (196, 64, 40, 0), (33, 9, 65, 1), (1, 1, 1, 0), (70, 24, 31, 1)])
def test_conv1x1_with_global_average(lib, dev, oracle, P, I, O, relu):
    """1x1 convolution whose epilogue leaves per-tile pixel sums; the softmax in front of which the
    pooled vector is needed adds the tiles and divides (drhip_deferred_vec.divisor)."""
    x, w, b = rnd(I, 1, P), rnd(I, O, 1, 1, scale=np.sqrt(2.0 / I)), rnd(O, scale=0.05)
    conv = oracle.conv1x1(x, w, b, relu=bool(relu))                      # [O, 1, P]
    pooled = oracle.pool(conv, (P, 1, 1), (P, 1, 1), 1).reshape(-1)       # global average
    slices = lib.drhip_conv1x1_poolsum_slices(P)
    assert slices == (P + 31) // 32
    parts = dev.empty(slices * O)
    ok(lib, lib.drhip_conv1x1_poolsum_f32(dev.put(x), dev.put(w), dev.put(b), parts, P, I, O, relu, None))
    got = dev.get(parts, (slices, O)).astype(np.float64).sum(axis=0) / P
    assert_close(got, pooled)
    fin, prob = dev.empty(O), dev.empty(O)
    d = DeferredVec(parts.value, None, slices, O, 0, fin.value, float(P))
    ok(lib, lib.drhip_softmax_ex_f32(None, ctypes.byref(d), prob, O, None))
    assert_close(dev.get(fin, (O,)), pooled)
    assert_close(dev.get(prob, (O,)), oracle.softmax(pooled))


@pytest.mark.parametrize("C,H,W", [(3, 224, 224), (1, 5, 7), (4, 17, 33), (64, 56, 56), (1, 1, 2)])
def test_normalize(lib, dev, oracle, C, H, W):
    x = (np.random.default_rng(C + H).random((C, H, W), dtype=np.float32) * 255.0).astype(np.float32)
    n = x.size
    scratch = dev.empty(lib.drhip_normalize_scratch_floats(n))
    xd, y = dev.put(x), dev.empty(n)
    for kind, tm, td in [(0, 3.0, 1.0), (1, 0.0, 2.0), (2, 0.0, 1.0), (2, 0.5, 1.5)]:
        first = None
        for _ in range(2):                   # the scratch needs no reset between calls; fixed summation order
            ok(lib, lib.drhip_normalize_f32(xd, y, n, kind, tm, td, scratch, None))
            got = dev.get(y, x.shape)
            assert first is None or np.array_equal(first, got)
            first = got
        assert_close(got, oracle.normalize(x, kind, tm, td))
        assert_close(got, oracle.normalize_f64(x, kind, tm, td))
    assert lib.drhip_normalize_f32(xd, y, n, 3, 0.0, 1.0, scratch, None) == -1
    assert lib.drhip_normalize_f32(xd, y, 0, 2, 0.0, 1.0, scratch, None) == -1


@pytest.mark.parametrize("n", [1, 3, 5, 1023, 1027, 1024 * 256 * 4 + 2, 1024 * 256 * 16 + 1024 * 128 + 3])
def test_normalize_merges_what_workgroups_leave(lib, dev, oracle, n):
    """The deviation out of sums about the workgroups' own means, which lie far apart here: one workgroup, ragged ends, all of its elements
    in registers and more than those."""
    x = (OWN.random(n, dtype=np.float32) + 100.0 * np.sin(np.arange(n) / 4096.0)).astype(np.float32)
    xd, y, scratch = dev.put(x), dev.empty(n), dev.empty(lib.drhip_normalize_scratch_floats(n))
    for kind, tm, td in [(1, 0.0, 2.0), (2, 0.5, 1.5)] if n > 1 else [(0, 3.0, 1.0)]:
        ok(lib, lib.drhip_normalize_f32(xd, y, n, kind, tm, td, scratch, None))
        want = oracle.normalize_f64(x.reshape(1, 1, n), kind, tm, td).reshape(-1)
        # (sums of n terms in a tree of at least 256 lanes: n / 2^18 terms one after the other, each step half a unit of 2^-23)
        assert np.abs(dev.get(y, (n,)) - want).max() <= (16 + n / 2 ** 18) * 2.0 ** -23 * max(np.abs(want).max(), np.abs(x).max() * td / max(x.std(), 1e-3))


def test_softmax(lib, dev, oracle):
    for n, scale in [(1000, 3.0), (10, 1.0), (5000, 5.0), (1, 1.0), (2048, 2.0), (2049, 2.0), (257, 1.0)]:
        x = rnd(n, scale=scale)
        y = dev.empty(n)
        ok(lib, lib.drhip_softmax_f32(dev.put(x), y, n, None))
        got = dev.get(y, (n,))
        assert_close(got, oracle.softmax(x))
        assert_close(got, oracle.softmax_f64(x))
        assert abs(float(got.sum()) - 1) < 1e-5 and int(got.argmax()) == int(x.argmax())
    # logits that overflow exp() unshifted still give a distribution here
    big = np.array([100.0, 101.0, 99.0], np.float32)
    y = dev.empty(3)
    ok(lib, lib.drhip_softmax_f32(dev.put(big), y, 3, None))
    assert_close(dev.get(y, (3,)), oracle.softmax_f64(big))


@pytest.mark.parametrize("env", [{}, {"DR_SPIN_US": "0"}, {"DR_UPLOAD_KERNEL": "0"}])
def test_staged_transfers_carry_every_byte(lib, dev, env):
    """Uploads through the pinned area (by kernel and by the DMA engine: odd destination offsets and sizes
    take the latter) and downloads through the flagged copy kernel, many times over with new contents and
    sizes each time: a flag seen before its data, or data left in the area from the call before, would show."""
    import os
    os.environ.update(env)
    try:
        h = ctypes.c_void_p()
        ok(lib, lib.drhip_staging_create(ctypes.byref(h), 1 << 20))
    finally:
        for k in env:
            os.environ.pop(k, None)
    assert lib.drhip_staging_upload_capacity(h) == 1 << 20 and lib.drhip_staging_download_capacity(h) == 65536
    rng = np.random.default_rng(11)
    buf = dev.empty(1 << 18)
    vp = ctypes.c_void_p
    try:
        for it in range(300):
            n = int(rng.choice([1, 3, 4, 250, 1000, 4096, 16383, 16384, 75001, 131072]))     # (from 256 KiB on an upload goes in two pieces)
            off = int(rng.integers(0, 64)) * int(rng.choice([1, 4]))          # floats; some 16-byte aligned, some not
            a = rng.standard_normal(n).astype(np.float32) + it
            ok(lib, lib.drhip_upload_staged(h, buf, 4 * off, a.ctypes.data_as(vp), a.nbytes, None))
            a_copy = a.copy()
            a[...] = np.nan                                                    # the caller's array is free again
            if a.nbytes <= 65536:
                back = np.full(n, -1.0, np.float32)
                ok(lib, lib.drhip_download_staged(h, back.ctypes.data_as(vp), buf, 4 * off, back.nbytes, None))
            else:                                                              # (beyond the download area: the plain blocking copy)
                back = dev.get(buf, (off + n,))[off:]
            assert np.array_equal(back, a_copy), (it, n, off)
        # many uploads in a row with no download in between (the two pinned areas are reused while earlier uploads
        # may still be in flight), the caller's array overwritten after every call
        n, rows = 4096, 24
        src = np.empty(n, np.float32)
        want = np.empty((rows, n), np.float32)
        for k in range(rows):
            src[...] = rng.standard_normal(n).astype(np.float32) + 100 * k
            want[k] = src
            ok(lib, lib.drhip_upload_staged(h, buf, 4 * k * n, src.ctypes.data_as(vp), src.nbytes, None))
            src[...] = np.nan
        for k in range(rows):
            back = np.full(n, -1.0, np.float32)
            ok(lib, lib.drhip_download_staged(h, back.ctypes.data_as(vp), buf, 4 * k * n, back.nbytes, None))
            assert np.array_equal(back, want[k]), k
        # bytes that are not whole floats go through the DMA engine both ways
        raw = rng.integers(0, 256, 1001, dtype=np.uint8)
        ok(lib, lib.drhip_upload_staged(h, buf, 3, raw.ctypes.data_as(vp), raw.nbytes, None))
        got = np.zeros_like(raw)
        ok(lib, lib.drhip_download_staged(h, got.ctypes.data_as(vp), buf, 3, got.nbytes, None))
        assert np.array_equal(got, raw)
        assert lib.drhip_download_staged(h, got.ctypes.data_as(vp), buf, 0, 65537, None) == -1
        assert lib.drhip_upload_staged(h, buf, 0, raw.ctypes.data_as(vp), (1 << 20) + 1, None) == -1
    finally:
        lib.drhip_staging_destroy(h)


@pytest.mark.parametrize("pixels,channels", [(1, 3), (5, 2), (1023, 3), (1025, 4), (50176, 3), (65537, 2), (4097, 1), (700, 7), (9, 64), (400001, 3), (115210, 3), (307201, 3)])
@pytest.mark.parametrize("env", [{}, {"DR_UPLOAD_KERNEL": "0"}])
def test_interleaved_upload_and_joint_download(lib, dev, pixels, channels, env):
    """[pixels][channels] on the host -> [channels][pixels] on the device: by kernel in one, two, three and eight pieces, at the
    edges of its 512-pixel blocks, beyond 4 MiB and with many channels (host), each twice; then several arrays back
    in one trip, and in several where they do not fit the download area."""
    import os
    os.environ.update(env)
    try:
        h = ctypes.c_void_p()
        ok(lib, lib.drhip_staging_create(ctypes.byref(h), 4 * pixels * channels))
    finally:
        for k in env:
            os.environ.pop(k, None)
    vp = ctypes.c_void_p
    try:
        rng = np.random.default_rng(pixels)
        buf = dev.empty(pixels * channels)
        for _ in range(2):
            a = rng.standard_normal((pixels, channels)).astype(np.float32)
            want = a.T.copy()
            ok(lib, lib.drhip_timing_begin())
            ok(lib, lib.drhip_upload_staged_interleaved(h, buf, a.ctypes.data_as(vp), pixels, channels, None))
            launches, ms = ctypes.c_int(), (ctypes.c_float * 8)()
            ok(lib, lib.drhip_timing_end(ms, 8, ctypes.byref(launches)))
            assert (launches.value > 0) == (not env and a.nbytes <= 4 << 20)      # by kernel up to 4 MiB, whatever the channels
            a[...] = np.nan                                                    # the caller's array is free again
            lengths = [min(pixels, 9000), 1, min(pixels, 17)] if channels > 1 else [pixels]
            backs = [np.full(n, -1.0, np.float32) for n in lengths]
            addr = buf.value if isinstance(buf, vp) else buf
            srcs = (vp * len(lengths))(*[addr + 4 * k * pixels * (channels > k) for k in range(len(lengths))])
            dsts = (vp * len(lengths))(*[b.ctypes.data for b in backs])
            ok(lib, lib.drhip_download_staged_many(h, len(lengths), dsts, srcs, (ctypes.c_size_t * len(lengths))(*lengths), None))
            for k, b in enumerate(backs):
                assert np.array_equal(b, want[k * (channels > k)][:lengths[k]]), k
            assert np.array_equal(dev.get(buf, want.shape), want)
    finally:
        lib.drhip_staging_destroy(h)


def test_copy3d_and_scalar(lib, dev, oracle):
    x = rnd(6, 9, 11)
    out = dev.empty(3 * 4 * 5)
    ok(lib, lib.drhip_copy3d_f32(dev.put(x), 11, 9, 2, 3, 1, out, 5, 4, 0, 0, 0, 5, 4, 3, None))
    assert np.array_equal(dev.get(out, (3, 4, 5)), x[1:4, 3:7, 2:7])
    assert lib.drhip_copy3d_f32(dev.put(x), 11, 9, 8, 0, 0, out, 5, 4, 0, 0, 0, 5, 4, 3, None) == -1   # box leaves the source
    for op, s in [(0, 1.5), (1, 123.68), (2, 0.5), (3, 4.0), (7, 2.0)]:
        y = dev.empty(x.size)
        ok(lib, lib.drhip_scalar_op_f32(dev.put(x), y, x.size, op, s, None))
        assert np.array_equal(dev.get(y, x.shape), oracle.scalar_op(x, op, s))


# ---------------------------------------------------------------------------------------------
# Seeded sweeps over ragged shapes: sizes that are no multiple of any tile, panel, stage or vector
# width the kernels use, single rows / columns / channels included.

def _sweep(seed, count, draw):
    """`count` seeded draws; DR_SWEEP_SCALE=n in the environment multiplies the count for a one-off wider run."""
    rng = np.random.default_rng(seed)
    return [draw(rng) for _ in range(count * int(os.environ.get("DR_SWEEP_SCALE", "1")))]


@pytest.mark.parametrize("W,H,I,O,variant", _sweep(11, 40, lambda r: (
    int(r.integers(1, 41)), int(r.integers(1, 41)), int(r.integers(1, 41)), int(r.integers(1, 71)),
    int(r.choice([0, 1, 2, 3, 0x11, 0x12, 0x21, 0x31, 0x101, 0x102, 0x103, 0x111, 0x121,
                  0x401, 0x402, 0x411, 0x422, 0x501, 0x502, 0x503, 0x511, 0x521]))))
    + [(1, 37, 9, 31, 0x11), (37, 1, 8, 32, 1), (3, 3, 64, 33, 0x21), (40, 2, 17, 1, 2)])
def test_winograd_sweep(lib, dev, oracle, W, H, I, O, variant):
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    U, _ = wino_filters(lib, dev, w)
    ws = wino_workspace(lib, dev, W, H, I, O, variant)
    relu = (W + H + I + O) & 1
    want = oracle.conv_winograd(x, w, b, relu=bool(relu))
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv3x3_winograd_f32(dev.put(x), U, dev.put(b), out, W, H, I, O, relu, variant, ws, None))
    got = dev.get(out, want.shape)
    assert_close(got, want)
    assert_close(got, oracle.conv_f64(x, w, b, relu=bool(relu)))


@pytest.mark.parametrize("W,H,I,O,kw,kh,sx,sy", _sweep(12, 20, lambda r: (
    int(r.integers(1, 40)), int(r.integers(1, 40)), int(r.integers(1, 20)), int(r.integers(1, 40)),
    int(r.choice([1, 3, 5, 7])), int(r.choice([1, 3, 5])), int(r.integers(1, 4)), int(r.integers(1, 4)))))
def test_conv_direct_sweep(lib, dev, oracle, W, H, I, O, kw, kh, sx, sy):
    if W // sx == 0 or H // sy == 0:
        pytest.skip("empty output")
    x, w, b = rnd(I, H, W), rnd(I, O, kh, kw, scale=np.sqrt(2.0 / (kh * kw * I))), rnd(O, scale=0.01)
    want = oracle.conv_direct(x, w, b, (sx, sy), relu=False)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv2d_direct_f32(dev.put(x), dev.put(w), dev.put(b), out, W, H, I, O, kw, kh, sx, sy, 0, None))
    got = dev.get(out, want.shape)
    assert_close(got, want)
    assert_close(got, oracle.conv_f64(x, w, b, stride=(sx, sy)))


@pytest.mark.parametrize("W,H,I,O,s,variant", _sweep(16, 32, lambda r: (
    int(r.integers(1, 41)), int(r.integers(1, 41)), int(r.integers(1, 41)), int(r.integers(1, 71)), int(r.integers(1, 3)),
    int(r.choice([0, 1, 2, 4, 8, 0x11, 0x12, 0x14, 0x18]))))
    + [(1, 40, 9, 31, 1, 0x12), (40, 1, 8, 33, 2, 4), (3, 3, 64, 65, 1, 8), (2, 2, 7, 1, 2, 0x11)])
def test_conv3x3_direct_mfma_sweep(lib, dev, oracle, W, H, I, O, s, variant):
    if W // s == 0 or H // s == 0:
        pytest.skip("empty output")
    x, w, b = rnd(I, H, W), rnd(I, O, 3, 3, scale=np.sqrt(2.0 / (9 * I))), rnd(O, scale=0.01)
    F = dev.empty(lib.drhip_conv3x3_direct_filter_floats(I, O))
    ok(lib, lib.drhip_conv3x3_direct_filter_layout_f32(dev.put(w), F, I, O, None))
    relu = (W + H + I + O) & 1
    want = oracle.conv_direct(x, w, b, (s, s), relu=bool(relu))
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv3x3_direct_mfma_f32(dev.put(x), F, dev.put(b), out, W, H, I, O, s, relu, variant, None))
    got = dev.get(out, want.shape)
    assert_close(got, want, terms=9 * I)
    assert_close(got, oracle.conv_f64(x, w, b, stride=(s, s), relu=bool(relu)), terms=9 * I)


@pytest.mark.parametrize("Win,Hin,I,O", _sweep(17, 20, lambda r: (
    int(r.integers(1, 60)), int(r.integers(1, 60)), int(r.integers(1, 140)), int(r.integers(1, 70)))))
def test_conv1x1_with_pooled_input_sweep(lib, dev, oracle, Win, Hin, I, O):
    x, w, b = rnd(I, Hin, Win), rnd(I, O, 1, 1, scale=np.sqrt(2.0 / I)), rnd(O, scale=0.01)
    pooled = oracle.pool(x, (3, 3, 1), (2, 2, 1), 0)
    relu = (Win + Hin + I + O) & 1
    want = oracle.conv1x1(pooled, w, b, relu=bool(relu))
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv1x1_pooled3s2_f32(dev.put(x), dev.put(w), dev.put(b), out, Win, Hin, I, O, relu, None))
    assert_close(dev.get(out, want.shape), want, terms=I)


@pytest.mark.parametrize("P,I,O,variant", _sweep(13, 20, lambda r: (
    int(r.integers(1, 400)), int(r.integers(1, 100)), int(r.integers(1, 100)), int(r.choice([0, 1, 2, 4, 8, 0x101, 0x104, 0x110])))))
def test_conv1x1_sweep(lib, dev, oracle, P, I, O, variant):
    x, w, b = rnd(I, 1, P), rnd(I, O, 1, 1, scale=np.sqrt(2.0 / I)), rnd(O, scale=0.01)
    want = oracle.conv1x1(x, w, b, relu=False)
    out = dev.empty(want.size)
    ok(lib, lib.drhip_conv1x1_f32(dev.put(x), dev.put(w), dev.put(b), out, P, I, O, 0, variant, None))
    assert_close(dev.get(out, want.shape), want)


@pytest.mark.parametrize("W,H,C,kx,ky,kz,sx,sy,sz", _sweep(14, 24, lambda r: (
    int(r.integers(1, 30)), int(r.integers(1, 30)), int(r.integers(1, 9)),
    int(r.integers(1, 12)), int(r.integers(1, 12)), int(r.integers(1, 3)),
    int(r.integers(1, 6)), int(r.integers(1, 6)), int(r.integers(1, 3)))))
def test_pool_sweep(lib, dev, oracle, W, H, C, kx, ky, kz, sx, sy, sz):
    x = rnd(C, H, W)
    x[:, ::2, ::3] = x.flat[0]
    for kind in (0, 1):
        want = oracle.pool(x, (kx, ky, kz), (sx, sy, sz), kind)
        out = dev.empty(want.size)
        ok(lib, lib.drhip_pool_f32(dev.put(x), out, None, W, H, C, kx, ky, kz, sx, sy, sz, kind, None))
        got = dev.get(out, want.shape)
        if kind == 0:
            assert np.array_equal(got, want)
        else:
            assert rel_err(got, want) <= 1e-6


@pytest.mark.parametrize("C,H,W,N", _sweep(15, 16, lambda r: (
    int(r.integers(1, 70)), int(r.integers(1, 6)), int(r.integers(1, 6)), int(r.integers(1, 600)))))
def test_fc_sweep(lib, dev, oracle, C, H, W, N):
    K = C * H * W
    x, Wt, b = rnd(C, H, W), rnd(K, N, scale=np.sqrt(2.0 / K)), rnd(N, scale=0.01)
    want = oracle.fc(x, Wt, b, relu=False).reshape(-1)
    perm = dev.empty(K * N)
    ok(lib, lib.drhip_fc_permute_rows_f32(dev.put(Wt), perm, W, H, C, N, None))
    n = lib.drhip_fc_scratch_floats(K, N)
    y = dev.empty(N)
    ok(lib, lib.drhip_fc_f32(dev.put(x), perm, dev.put(b), y, dev.empty(n) if n else None, K, N, 0, None))
    got = dev.get(y, (N,))
    assert_close(got, want, terms=K)
    assert_close(got, oracle.fc_f64(x, Wt, b).reshape(-1), terms=K)


@pytest.mark.parametrize("K,N", [(7, 10), (15, 1000), (48, 98), (191, 300), (1000, 10), (8240, 10)])
def test_fc_last_rows(lib, dev, K, N):
    """Rows left over behind whole turns, eight at a time: against float64 (an fp32 sum of K products, so eps sqrt(K) of the sum of their
    amounts), and an infinite weight in the last row, whose place stands in for rows that do not exist, stays an infinity."""
    x, Wt = np.abs(rnd(K)) + np.float32(0.1), rnd(K, N, scale=np.sqrt(2.0 / K))
    n = lib.drhip_fc_scratch_floats(K, N)
    for inf in (False, True):
        if inf:
            Wt[K - 1, 0] = np.inf
        y = dev.empty(N)
        ok(lib, lib.drhip_fc_f32(dev.put(x), dev.put(Wt), None, y, dev.empty(n) if n else None, K, N, 0, None))
        got = dev.get(y, (N,)).astype(np.float64)
        assert not inf or got[0] == np.inf
        x64, w64 = x.astype(np.float64), Wt.astype(np.float64)[:, 1:]
        assert (np.abs(got[1:] - x64 @ w64) <= 2.0 ** -23 * np.sqrt(K) * (x64 @ np.abs(w64))).all()


def test_mfma_clock_probe(lib, gpu):
    """The measurement aid of bench.py: shader clock under a stream of fp32 MFMAs, from the two clock counters a wave
    can read.  Somewhere between idle clocks and the 2.4 GHz of the data sheet."""
    mhz, us = ctypes.c_float(0), ctypes.c_float(0)
    lib.drhip_mfma_clock_probe.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_float), ctypes.c_void_p]
    ok(lib, lib.drhip_mfma_clock_probe(100, 3, ctypes.byref(mhz), ctypes.byref(us), None))
    assert 500.0 < mhz.value < 2600.0 and us.value > 5.0, (mhz.value, us.value)
    assert lib.drhip_mfma_clock_probe(0, 1, ctypes.byref(mhz), None, None) == -1
