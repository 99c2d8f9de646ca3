"""Joined Winograd launches whose workgroups do not wait for each other (DR_WINO_JOIN_SPINS): what they leave behind.  (The kernels count
such waits over the life of the process, and other tests want that count to be zero: this file comes behind theirs.)
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MARKER = 0xffa5c3e1


def ok(lib, rc):
    assert rc == 0, lib.drhip_last_error().decode()


@pytest.mark.parametrize("spins", [1, 4, 16])
@pytest.mark.parametrize("kind,variant,W,H,I,O", [
    ("fp32", 0x2c01, 56, 56, 256, 256), ("fp32", 0x2c01, 34, 31, 200, 70),      # helpers: of four panels each, of one
    ("fp32", 0xc11, 28, 28, 256, 512), ("fp32", 0x831, 14, 14, 512, 512), ("fp32", 0xc22, 14, 14, 128, 96),     # joined halves, eighths, quarters
    ("fp32", 0x1801, 112, 112, 128, 128),       # tiers
    ("split", 0x101 | 2 << 12 | 2 << 16, 28, 28, 256, 512), ("split", 0x101 | 4 << 12 | 4 << 16, 27, 13, 256, 130), ("split", 0x100 | 2 << 12 | 2 << 16, 64, 36, 96, 70),
    ("split", 0x101 | 3 << 12 | 3 << 16, 88, 72, 256, 128),     # 39 pieces for the 32 CUs of an XCD: some wait for others that have not begun
    # two f16 parts: quarters with two wave sets, thirds and halves with one, whole panels in front of quarters, thirds and halves, and pieces of two kinds
    ("pair", 0x301 | 4 << 12 | 4 << 16, 27, 13, 256, 130), ("pair", 0x300 | 3 << 12 | 3 << 16, 73, 28, 400, 130), ("pair", 0x300 | 2 << 12 | 2 << 16, 64, 36, 96, 70),
    ("pair", 0x300 | 4 << 20 | 1 << 12 | 4 << 16, 64, 36, 256, 70), ("pair", 0x300 | 4 << 20 | 1 << 12 | 3 << 16, 63, 36, 200, 70),
    ("pair", 0x300 | 3 << 20 | 1 << 12 | 2 << 16, 64, 36, 130, 70), ("pair", 0x301 | 2 << 20 | 2 << 12 | 3 << 16, 64, 36, 130, 70),
])
def test_tiles_that_come_too_late_are_gone_with_the_launch(lib, dev, monkeypatch, kind, variant, W, H, I, O, spins):
    """A workgroup that does not wait for its partners gives NaN for what is missing, and their tiles, which come later, are not
    there for the next launch: every launch leaves the marker in every slot, and gives what is right where it gives numbers.  Another
    launch that takes whole CUs runs beside them, so that workgroups begin at different times."""
    rng = np.random.default_rng(W * I + variant)
    draw = lambda *shape: rng.standard_normal(shape).astype(np.float32)
    w, out = draw(I, O, 3, 3), dev.empty(O * H * W)
    split = kind != "fp32"
    named = {"fp32": "", "split": "split_", "pair": "pair_"}[kind]
    U = dev.empty(getattr(lib, "drhip_conv3x3_winograd_%sfilter_floats" % named)(I, O))
    ok(lib, getattr(lib, "drhip_winograd_%sfilter_transform_f32" % named)(dev.put(w), U, I, O, None))
    n = (lib.drhip_conv3x3_winograd_split_workspace_floats if split else lib.drhip_conv3x3_winograd_workspace_floats)(W, H, I, O, variant)
    assert n
    ws = dev.empty(n)
    ok(lib, lib.drhip_conv3x3_winograd_workspace_prepare_f32(ws, n, None))
    conv = lib.drhip_conv3x3_winograd_split_f32 if split else lib.drhip_conv3x3_winograd_f32
    inputs = [dev.put(draw(I, H, W)) for _ in range(3)]

    R = (112, 112, 64, 128)         # the rival: unsplit, 128 KiB of LDS
    rivalU, rivalOut = dev.empty(lib.drhip_conv3x3_winograd_split_filter_floats(*R[2:])), dev.empty(R[0] * R[1] * R[3])
    rivalIn = dev.put(draw(R[2], R[1], R[0]))
    ok(lib, lib.drhip_winograd_split_filter_transform_f32(dev.put(draw(R[2], R[3], 3, 3)), rivalU, *R[2:], None))
    streams = [ctypes.c_void_p(), ctypes.c_void_p()]
    for st in streams:
        ok(lib, lib.drhip_stream_create(ctypes.byref(st)))

    def run(x):
        for _ in range(3):
            ok(lib, lib.drhip_conv3x3_winograd_split_f32(rivalIn, rivalU, None, rivalOut, *R, 0, 0x101, None, streams[1]))
        ok(lib, conv(x, U, None, out, W, H, I, O, 0, variant, ws, streams[0]))
        for st in streams:
            ok(lib, lib.drhip_stream_sync(st))
        return dev.get(out, (O, H, W))

    def left_behind():
        return int(np.count_nonzero(dev.get(ws, (n,), np.uint32) != MARKER))

    want = [run(x) for x in inputs]
    assert all(np.isfinite(y).all() for y in want) and left_behind() == 0
    late = ctypes.c_uint(0)
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    before, missing = late.value, 0
    monkeypatch.setenv("DR_WINO_JOIN_SPINS", str(spins))
    for _ in range(4):
        for x, y in zip(inputs, want):
            got = run(x)
            assert left_behind() == 0
            known = ~np.isnan(got)
            missing += int(np.count_nonzero(~known))
            assert np.array_equal(got[known], y[known])
    ok(lib, lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)))
    print("%s %#x: %d outputs missing, %d waits given up" % (kind, variant, missing, late.value - before))
    assert late.value > before or missing == 0          # (no output is missing that was not counted)
    monkeypatch.delenv("DR_WINO_JOIN_SPINS")
    for x, y in zip(inputs, want):                      # launches that wait again, and see their tiles off
        assert np.array_equal(run(x), y) and left_behind() == 0
    for st in streams:
        ok(lib, lib.drhip_stream_destroy(st))
