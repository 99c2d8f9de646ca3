"""End-to-end parity through the deepRacin C graph API (dR_NewGraph ... dR_downloadArray) on the GPU.

Every benchmark configuration is built from seeded synthetic tensors, run through libdeepracin.so and
compared with the CPU oracle evaluating the same layer list.  Bars (north star): per-layer max
relative error <= 1e-4 (max|gpu-oracle| / max|oracle| of that layer), final logits max abs error
<= 1e-3 with identical argmax, pooling bit-exact given equal inputs.
"""
import ctypes
import os

import numpy as np
import pytest

import deepracin_amd as dr
from deepracin_amd import configs
from conftest import GOLDEN, assert_close, rel_err, spec_terms

pytestmark = pytest.mark.gpu

LAYER_TOL = 1e-4
LOGIT_TOL = 1e-3


class _Handler(ctypes.Structure):
    _fields_ = [("outputFor", ctypes.c_void_p), ("size", ctypes.c_int), ("numberOfDependencies", ctypes.c_int),
                ("bufptr", ctypes.POINTER(ctypes.c_void_p)), ("buf", ctypes.c_void_p)]


class _NodeHead(ctypes.Structure):
    _fields_ = [("oshape", dr.Shape3), ("layerID", ctypes.c_int32), ("previous_layers", ctypes.c_void_p),
                ("next_layers", ctypes.c_void_p), ("clKernel", ctypes.c_void_p), ("outputBuf", ctypes.POINTER(_Handler))]


def node_output(graph, node):
    """Download a node's buffer via the public struct layout (include/dR_types.h) as [C][H][W]."""
    head = ctypes.cast(node.ptr, ctypes.POINTER(_NodeHead)).contents
    s = head.oshape
    flat = np.empty(s.s0 * s.s1 * s.s2, np.float32)
    graph.lib.dR_downloadArray(graph.ptr, b"", head.outputBuf.contents.bufptr, 0, flat.nbytes, flat.ctypes.data_as(ctypes.c_void_p))
    return flat.reshape(s.s2, s.s1, s.s0)


def run_config(name, outputs=None, env_vars=None, **kw):
    spec, feeds, outs = configs.CONFIGS[name](**kw)
    outs = outputs(spec, outs) if callable(outputs) else (outputs or outs)
    old = {k: os.environ.get(k) for k in (env_vars or {})}
    os.environ.update(env_vars or {})
    try:
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, outs)
            dr.prepare(g)
            for i, a in feeds.items():
                configs.feed_chw(nodes[i], a)
            assert g.lib.dR_apply(g.ptr)
            got = {i: node_output(g, nodes[i]) for i in outs}
            # a second pass over the same buffers must reproduce the first bit for bit
            assert g.lib.dR_apply(g.ptr)
            again = {i: node_output(g, nodes[i]) for i in outs}
    finally:
        for k, v in old.items():
            if v is None:
                os.environ.pop(k, None)
            else:
                os.environ[k] = v
    for i in outs:
        assert np.array_equal(got[i], again[i]), "node %d differs between two applies" % i
    return spec, feeds, got


def all_compute_nodes(spec, outs):
    return [i for i, n in enumerate(spec) if n["op"] != "feed"]


def check_layers(oracle, spec, feeds, got, force_direct=False):
    """Two comparisons with the oracle.  End to end (the oracle's own chain of layers): norm-wise 1e-4 per
    node.  Layer by layer (the oracle evaluates every node on the tensors the GPU produced for its
    inputs): norm-wise 1e-4 and element-wise |gpu-oracle| <= 1e-4*|oracle| + 1e-6*max|oracle| -- applied
    to the nodes all of whose inputs are feeds or downloaded tensors."""
    want = oracle.run_spec(spec, feeds, force_direct=force_direct)
    for i, g in got.items():
        assert g.shape == want[i].shape, "node %d shape %s vs %s" % (i, g.shape, want[i].shape)
        e = rel_err(g, want[i])
        assert e <= LAYER_TOL, "node %d (%s): rel err %.3g" % (i, spec[i]["op"], e)
    step = oracle.run_spec(spec, feeds, force_direct=force_direct, inputs_from=got)
    for i, g in got.items():
        ins = spec[i].get("ins", [spec[i]["in"]] if "in" in spec[i] else [])
        if all(j in got or spec[j]["op"] == "feed" for j in ins):
            assert_close(g, step[i], "node %d (%s) on the GPU's own inputs" % (i, spec[i]["op"]), LAYER_TOL, spec_terms(spec[i]))
    return want


def test_config1_conv3x3_winograd_and_direct(oracle, gpu):
    spec, feeds, got = run_config("conv3x3")
    check_layers(oracle, spec, feeds, got)
    spec, feeds, got_d = run_config("conv3x3", env_vars={"DR_CONV3X3": "direct"})
    check_layers(oracle, spec, feeds, got_d, force_direct=True)
    truth = oracle.run_spec(spec, feeds, f64=True)[1]
    assert rel_err(got[1], truth) <= LAYER_TOL and rel_err(got_d[1], truth) <= LAYER_TOL


def test_config2_fire_module(oracle, gpu):
    # default: only the concat is an output -> producers write straight into the concat buffer
    spec, feeds, got = run_config("fire")
    want = check_layers(oracle, spec, feeds, got)
    assert got[4].shape == (128, 55, 55)
    # every node an output -> nothing is fused, the concat copies; same numbers
    spec, feeds, got_all = run_config("fire", outputs=all_compute_nodes)
    check_layers(oracle, spec, feeds, got_all)
    # default run: the 1x1 expand rides along in the 3x3 expand's Winograd launch (centre taps), so its
    # channels round differently at the 1e-6 level; with that fusion off the runs agree bit for bit
    assert np.array_equal(got_all[4][64:], got[4][64:]) and rel_err(got[4], got_all[4]) <= 1e-5
    _, _, apart = run_config("fire", env_vars={"DR_FUSE_EXPAND": "0"})
    assert np.array_equal(got_all[4], apart[4])
    assert np.array_equal(got_all[4][:64], got_all[2]) and np.array_equal(got_all[4][64:], got_all[3])
    assert rel_err(got[4], oracle.run_spec(spec, feeds, f64=True)[4]) <= LAYER_TOL
    del want


def test_config3_vgg_conv3_block(oracle, gpu):
    spec, feeds, got = run_config("vgg_conv3", outputs=all_compute_nodes)
    want = check_layers(oracle, spec, feeds, got)
    assert got[4].shape == (256, 28, 28)
    # pooling is bit-exact given the same input: pool the GPU's own conv output on the CPU
    assert np.array_equal(got[4], oracle.pool(got[3], (2, 2, 1), (2, 2, 1), 0))
    del want


def test_maxpool_fused_into_convolution(oracle, gpu):
    """With only the final tensor requested, the last convolution of the block stores the pooled
    tensor itself (no pooling launch); the numbers equal the unfused run bit for bit."""
    spec, feeds, fused = run_config("vgg_conv3")
    _, _, plain = run_config("vgg_conv3", env_vars={"DR_FUSE_POOL": "0"})
    assert np.array_equal(fused[4], plain[4]) and fused[4].shape == (256, 28, 28)
    want = oracle.run_spec(spec, feeds)
    assert_close(fused[4], want[4], "fused pool")
    # the pooling node of the fused run launches nothing
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [4])
        dr.prepare(g)
        configs.feed_chw(nodes[0], feeds[0])
        dr.graph_config(g).profilingGPU = 1
        assert g.lib.dR_apply(g.ptr)
        assert dr.node_struct(nodes[4]).drLastKernelMs == 0.0 and dr.node_struct(nodes[3]).drLastKernelMs > 0.0


@pytest.mark.parametrize("W,H,I,O,relu", [(224, 224, 3, 64, True), (2, 2, 1, 1, False), (34, 18, 4, 33, False), (98, 66, 2, 70, True), (124, 70, 4, 33, False), (99, 66, 3, 33, False), (98, 66, 5, 33, True)])
def test_average_pooling_behind_an_image_layer(oracle, gpu, W, H, I, O, relu):
    """A 3x3 layer over an image and a 2x2/2 average pooling in one launch: the two kernels' numbers (DR_FUSE_POOL=0); small and odd maps
    and layers of five channels stay apart."""
    st = configs._Streams(95)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O, relu=relu), {"op": "pool", "in": 1, "window": (2, 2, 1), "stride": (2, 2, 1), "kind": 1}]
    x = configs.image_input(st, W, H, I)
    want, res, launches = oracle.run_spec(spec, {0: x}), {}, {}
    for mode in ("1", "0"):
        os.environ["DR_FUSE_POOL"] = mode
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [2])
                dr.prepare(g)
                configs.feed_chw(nodes[0], x)
                assert g.lib.dR_apply(g.ptr)
                res[mode] = configs.fetch_chw(g)[0].copy()
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                launches[mode] = g.lib.drhip_timing_count()
        finally:
            os.environ.pop("DR_FUSE_POOL", None)
    fused = bool(dr.load_library().drhip_conv3x3_image_avgpool2_usable(W, H, I, O, dr.load_library().drhip_conv3x3_winograd_pick_variant(W, H, I, O)))
    assert launches["0"] - launches["1"] == fused and fused == (W % 2 == 0 and I <= 4 and W > 40)      # (small maps: the 16-tile kernel)
    assert np.array_equal(res["1"], res["0"])
    assert_close(res["1"], want[2], terms=9 * I)


@pytest.mark.parametrize("W,H,I,O,k,reader,fused", [(200, 200, 3, 64, 7, "", True), (47, 33, 3, 20, 7, "", True), (64, 63, 16, 33, 5, "", True), (33, 47, 64, 64, 5, "", False), (260, 260, 3, 160, 7, "", False),
                                                  (200, 200, 3, 64, 7, "1x1", True), (96, 96, 3, 24, 7, "1x1", False)])
def test_maxpool_of_three_behind_other_filters(oracle, gpu, W, H, I, O, k, reader, fused):
    """A layer of other filters by stride 2 and the 3x3/2 pooling behind it, in one launch where that is the faster way, and apart (DR_FUSE_POOL=0); in front of a
    1x1 layer, which otherwise takes the pooling on load, a launch more or less makes no difference in the count."""
    st = configs._Streams(97)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, k, I, O, stride=2), {"op": "pool", "in": 1, "window": (3, 3, 1), "stride": (2, 2, 1), "kind": 0}]
    if reader:
        spec.append(configs._conv(st, 2, 1, O, 16))
    x = configs.image_input(st, W, H, I)
    want, res, launches, variant = oracle.run_spec(spec, {0: x}), {}, {}, 0
    lib = dr.load_library()
    assert (lib.drhip_conv_bank_maxpool3s2_pick_variant(W, H, I, O, k, k, 2, 2, 1 if reader else 0) != 0) == fused
    for mode in ("1", "0"):
        os.environ["DR_FUSE_POOL"] = mode
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [len(spec) - 1])
                dr.prepare(g)
                configs.feed_chw(nodes[0], x)
                assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)
                res[mode] = configs.fetch_chw(g)[0].copy()
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                launches[mode] = g.lib.drhip_timing_count()
        finally:
            os.environ.pop("DR_FUSE_POOL", None)
    assert launches["0"] - launches["1"] == (1 if fused and not reader else 0), launches
    for got in res.values():
        assert_close(got, want[-1], terms=I * k * k)


def test_maxpool_taken_on_load_by_the_1x1_layer_behind_it(oracle, gpu):
    """SqueezeNet's pool3 / pool5 pattern: fire module -> 3x3/2 max pool -> squeeze 1x1.  With only the last
    tensor requested the squeeze layer pools while it loads (no pooling launch, no pooled tensor); with
    DR_FUSE_POOLIN=0 the two kernels run.  Same values to rounding (the channel sum is dealt to a different
    number of waves), and the layer bar against the oracle either way."""
    spec, feeds, outs = configs.fire_module(seed=21, size=27, cin=24, squeeze=8, expand=16)
    st = configs._Streams(22)
    spec.append(configs._maxpool(outs[0], 3, 2)); pool = len(spec) - 1
    spec.append(configs._conv(st, pool, 1, 32, 12)); sq = len(spec) - 1
    want = oracle.run_spec(spec, feeds)
    res = {}
    for flag in ("1", "0"):
        os.environ["DR_FUSE_POOLIN"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [sq])
                dr.prepare(g)
                for i, a in feeds.items():
                    configs.feed_chw(nodes[i], a)
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                pool_ms = dr.node_struct(nodes[pool]).drLastKernelMs
                dr.graph_config(g).profilingGPU = 0
                assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)       # recorded, then replayed
                res[flag] = (configs.fetch_chw(g)[0], pool_ms)
        finally:
            os.environ.pop("DR_FUSE_POOLIN", None)
    assert res["1"][1] == 0.0 and res["0"][1] > 0.0, "the pooling node must launch nothing when fused"
    assert res["1"][0].shape == (12, 14, 14)
    assert_close(res["1"][0], want[sq], "squeeze behind pool, fused")
    assert_close(res["0"][0], want[sq], "squeeze behind pool, unfused")
    assert rel_err(res["1"][0], res["0"][0]) <= 1e-5
    # the pooled tensor requested as an output: nothing is fused, and it is there
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [pool, sq])
        dr.prepare(g)
        for i, a in feeds.items():
            configs.feed_chw(nodes[i], a)
        assert g.lib.dR_apply(g.ptr)
        got_pool, got_sq = configs.fetch_chw(g)
    assert_close(got_pool, want[pool], "pool as output")
    assert_close(got_sq, want[sq], "squeeze, pool as output")


FIRE_CHAINS = [
    # w, h, input channels, modules (squeeze, expand, 'p' with a 3x3/2 max pooling behind it), relu, bias, squeeze layers computed in other launches
    (1, 1, 3, [(1, 32, ""), (1, 32, "")], True, True, 1),                       # one pixel
    (13, 9, 20, [(16, 64, ""), (16, 64, "p"), (32, 128, "")], True, True, 2),
    (56, 56, 24, [(16, 64, ""), (16, 64, "p"), (32, 128, ""), (32, 128, "p"), (48, 192, "")], True, True, 4),   # SqueezeNet's maps
    (14, 14, 64, [(48, 192, ""), (64, 256, ""), (64, 256, "")], True, True, 2),
    (17, 2, 40, [(64, 32, "p"), (50, 96, ""), (7, 32, "p"), (33, 64, "")], False, False, 2),        # ragged channels, nothing clipped at 0; pooled behind a plain tensor: apart
    (113, 75, 16, [(16, 64, ""), (16, 64, "p"), (24, 32, "")], True, False, 2),
    (85, 23, 16, [(12, 32, ""), (12, 64, "")], True, True, 1),                  # last module stored in rows: widths that no block of them divides
    (59, 7, 8, [(40, 32, ""), (33, 96, "")], True, True, 1),
    (9, 11, 8, [(65, 32, ""), (16, 48, ""), (64, 64, ""), (64, 32, "p")], True, True, 1),           # 65 and 48 are not covered: kernels of their own
]


@pytest.mark.parametrize("chain", FIRE_CHAINS, ids=lambda c: "%dx%d" % c[:2])
def test_fire_modules_in_a_chain(oracle, gpu, chain):
    """The expand layers of a module and the next module's squeeze layer in one launch, against the oracle and against
    kernels of their own (DR_FUSE_FIRE=0)."""
    w, h, cin, modules, relu, bias, hidden = chain
    st = configs._Streams(77)
    spec = [{"op": "feed", "shape": (w, h, cin)}]
    cur, squeezes, tail = 0, [], None
    for squeeze, expand, pool in modules:
        spec.append(configs._conv(st, cur, 1, cin, squeeze, relu=relu, bias=bias)); s = len(spec) - 1
        squeezes.append(s)
        spec.append(configs._conv(st, s, 1, squeeze, expand, relu=relu, bias=bias))
        spec.append(configs._conv(st, s, 3, squeeze, expand, relu=relu, bias=bias))
        spec.append({"op": "concat", "ins": [s + 1, s + 2], "dim": 2}); cur, cin = s + 3, 2 * expand
        if pool:
            spec.append(configs._maxpool(cur, 3, 2)); cur = len(spec) - 1
    feeds = {0: configs.image_input(st, w, h, spec[0]["shape"][2], 2.0) - np.float32(1)}
    want = oracle.run_spec(spec, feeds)[cur]
    res = {}
    for flag in ("1", "0"):
        os.environ["DR_FUSE_FIRE"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [cur])
                dr.prepare(g)
                configs.feed_chw(nodes[0], feeds[0])
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                silent = sum(dr.node_struct(nodes[i]).drLastKernelMs == 0.0 for i in squeezes)
                dr.graph_config(g).profilingGPU = 0
                first = configs.fetch_chw(g)[0]
                assert g.lib.dR_apply(g.ptr)
                res[flag] = configs.fetch_chw(g)[0]
                assert np.array_equal(first, res[flag])
        finally:
            os.environ.pop("DR_FUSE_FIRE", None)
        assert silent == (hidden if flag == "1" else 0)
        # (every layer rounds like a sum of at most 10 * 64 or 2 * 256 products; a chain of n of them carries n times that)
        assert_close(res[flag], want, "chain, DR_FUSE_FIRE=%s" % flag, terms=1024 * len(modules) ** 2)
    # another order of the same sums
    assert rel_err(res["1"], res["0"]) <= 2e-6 * len(modules)


@pytest.mark.parametrize("w,h,cin,first,squeeze,expand,classes,bias", [
    (91, 74, 3, 64, 16, 64, 1000, True),        # SqueezeNet's ends around one module; odd maps
    (18, 14, 4, 20, 33, 32, 17, False),         # ragged channels, one block of pooled pixels and a bit
    (132, 260, 2, 64, 64, 256, 10, True),       # 33 x 65 pixels: tiles of 32 in front of the average
    (132, 260, 2, 64, 64, 256, 333, True),      # the same pixel by pixel
    (24, 10, 1, 8, 8, 32, 5, True),             # one input channel: the squeeze layer stays a kernel of its own
], ids=lambda v: str(v))
def test_fire_chain_with_both_ends(oracle, gpu, w, h, cin, first, squeeze, expand, classes, bias):
    """First layer, pooling and squeeze layer in one launch in front of a module, and behind it a 1x1 layer with a global average
    that reads the module's outputs pixel by pixel: against the oracle, and against the kernels apart."""
    st = configs._Streams(78)
    spec = [{"op": "feed", "shape": (w, h, cin)}, configs._conv(st, 0, 3, cin, first, stride=2, bias=bias), configs._maxpool(1, 3, 2),
            configs._conv(st, 2, 1, first, squeeze, bias=bias), configs._conv(st, 3, 1, squeeze, expand, bias=bias), configs._conv(st, 3, 3, squeeze, expand, bias=bias),
            {"op": "concat", "ins": [4, 5], "dim": 2}, configs._conv(st, 6, 1, 2 * expand, classes, bias=bias)]
    wp, hp = -(-(w // 2) // 2), -(-(h // 2) // 2)
    spec += [{"op": "pool", "in": 7, "window": (wp, hp, 1), "stride": (wp, hp, 1), "kind": 1}, {"op": "softmax", "in": 8}]
    feeds = {0: configs.image_input(st, w, h, cin, 2.0) - np.float32(1)}
    want = oracle.run_spec(spec, feeds)
    res = {}
    for flag in ("1", "0"):
        os.environ["DR_FUSE_FIRE"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [9, 8])
                dr.prepare(g)
                configs.feed_chw(nodes[0], feeds[0])
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                silent = dr.node_struct(nodes[3]).drLastKernelMs == 0.0
                dr.graph_config(g).profilingGPU = 0
                assert g.lib.dR_apply(g.ptr)
                res[flag] = configs.fetch_chw(g)
        finally:
            os.environ.pop("DR_FUSE_FIRE", None)
        assert silent == (flag == "1" and cin > 1)
        assert_close(res[flag][1].reshape(-1), want[8].reshape(-1), "average, DR_FUSE_FIRE=%s" % flag, terms=4096)
        assert np.abs(res[flag][0].reshape(-1) - want[9].reshape(-1)).max() <= 1e-5
    # another order of the same sums
    assert rel_err(res["1"][1], res["0"][1]) <= 5e-6


@pytest.mark.parametrize("w,h,cin,first,k,stride", [(65, 47, 3, 64, 7, 2), (30, 34, 8, 64, 5, 1), (60, 52, 16, 32, 3, 2), (41, 37, 4, 24, 5, 2)])
def test_fire_module_behind_a_pooled_layer_of_other_filters(oracle, gpu, w, h, cin, first, k, stride):
    """A layer on the split filter bank with a 2x2 pooling in its launch, then two modules: the squeeze layer behind the pooling is
    a launch of its own, in front of a chain."""
    st = configs._Streams(79)
    spec = [{"op": "feed", "shape": (w, h, cin)}, configs._conv(st, 0, k, cin, first, stride=stride), configs._maxpool(1, 2, 2)]
    channels = first
    for squeeze, expand in ((16, 32), (20, 64)):
        s = len(spec)
        spec += [configs._conv(st, s - 1, 1, channels, squeeze), configs._conv(st, s, 1, squeeze, expand), configs._conv(st, s, 3, squeeze, expand),
                 {"op": "concat", "ins": [s + 1, s + 2], "dim": 2}]
        channels = 2 * expand
    x = configs.image_input(st, w, h, cin, 2.0) - np.float32(1)
    want = oracle.run_spec(spec, {0: x})
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [len(spec) - 1])
        dr.prepare(g)
        configs.feed_chw(nodes[0], x)
        assert g.lib.dR_apply(g.ptr)
        assert rel_err(configs.fetch_chw(g)[0], want[-1]) <= LAYER_TOL


@pytest.mark.parametrize("K,N,front,logits", [(1, 1, 0, True), (1024, 32, 0, False), (32, 1024, 40, True), (333, 98, 900, True), (128, 10, 1568, True), (5, 700, 0, True)],
                         ids=lambda v: str(v))
def test_small_layer_in_the_softmax(oracle, gpu, K, N, front, logits):
    """A small fully connected layer in the launch of the softmax behind it, on a plain or an unfinished input, and outputs that go to the
    host from that launch: against the oracle, the kernels apart (DR_FUSE_FC=0) and dR_apply with a download."""
    st = configs._Streams(81)
    spec = [{"op": "feed", "shape": (front or K, 1, 1)}]
    if front:
        spec.append(configs._fc(st, 0, front, K, True))
    spec.append(configs._fc(st, len(spec) - 1, K, N, False)); fc = len(spec) - 1
    spec.append({"op": "softmax", "in": fc})
    outs = [fc, fc + 1] if logits else [fc + 1]
    x = configs.image_input(st, front or K, 1, 1)
    want = oracle.run_spec(spec, {0: x})
    for flag in ("1", "0"):
        os.environ["DR_FUSE_FC"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, outs)
                dr.prepare(g)
                for k in (0, 1, 2):             # (another input in between: what comes back is this pass's)
                    configs.feed_chw(nodes[0], x if k != 1 else 1 - x)
                    got = dr.apply(g)
                assert g.lib.dR_apply(g.ptr)
                again = dr.download_outputs(g)
                dr.graph_config(g).profilingGPU = 1         # (apart: a profiled pass is waited for)
                slow = dr.apply(g)
                ms = dr.node_struct(nodes[fc]).drLastKernelMs
        finally:
            os.environ.pop("DR_FUSE_FC", None)
        assert (ms == 0.0) == (flag == "1")
        for u, v, w, i in zip(got, again, slow, outs):
            assert np.array_equal(u, v) and np.array_equal(u, w)
            # (a sum of K products that are themselves rounded sums)
            assert_close(np.reshape(u, -1), want[i].reshape(-1), "node %d" % i, terms=max(K, front) * (4 if front else 1), floor=0.01)


def test_outputs_on_their_way_to_the_host(gpu):
    """Outputs that the last kernel pushes: fetched late, twice, behind another pass, another download, a new image, and by one call."""
    st = configs._Streams(99)
    spec = [{"op": "feed", "shape": (9, 7, 3)}, configs._fc(st, 0, 189, 40, False), {"op": "softmax", "in": 1}]
    a, b = configs.image_input(st, 9, 7, 3), configs.image_input(st, 9, 7, 3)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [1, 2])
        dr.prepare(g)
        want = {}
        for name, x in (("a", a), ("b", b)):
            configs.feed_chw(nodes[0], x)
            assert g.lib.dR_apply(g.ptr)
            want[name] = [o.copy() for o in dr.download_outputs(g)]
        same = lambda got, name: all(np.array_equal(u, v) for u, v in zip(got, want[name])) and len(got) == 2
        configs.feed_chw(nodes[0], a)
        assert g.lib.dR_applyAhead(g.ptr)
        configs.feed_chw(nodes[0], b)                       # (behind the pass)
        assert same(dr.download_outputs(g), "a") and same(dr.download_outputs(g), "a")
        assert g.lib.dR_applyAhead(g.ptr)
        assert np.array_equal(np.squeeze(configs.fetch_chw(g)[1]), want["b"][1])        # one by one, through the same area
        assert same(dr.download_outputs(g), "b")
        configs.feed_chw(nodes[0], a)
        assert g.lib.dR_applyAhead(g.ptr)
        configs.feed_chw(nodes[0], b)
        assert g.lib.dR_apply(g.ptr) and same(dr.download_outputs(g), "b")              # an ordinary pass behind it
        configs.feed_chw(nodes[0], a)
        assert same(dr.apply(g), "a")
        flats = [np.empty(40, np.float32) for _ in range(2)]
        hosts = (ctypes.c_void_p * 2)(*[f.ctypes.data for f in flats])
        configs.feed_chw(nodes[0], b)
        assert g.lib.dR_applyAndDownload(g.ptr, hosts, 2) == 2 and same(flats, "b")
        configs.feed_chw(nodes[0], a)
        assert g.lib.dR_applyAndDownload(g.ptr, hosts, 1) == 1 and np.array_equal(flats[0], want["a"][0]) and np.array_equal(flats[1], want["b"][1])
        assert g.lib.dR_applyAhead(g.ptr)                   # (and nobody fetches them)


@pytest.mark.parametrize("W,H,I,O,split", [(30, 30, 24, 32, True), (33, 47, 36, 50, True), (7, 5, 9, 3, True), (90, 62, 70, 300, True), (20, 20, 64, 64, False), (41, 40, 80, 70, False)])
def test_strided_layers_by_either_kernel(oracle, gpu, W, H, I, O, split):
    """3x3/2 layers on both sides of the rule that chooses their kernel, and by the general one (DR_DIRECT_VALU=1)."""
    st = configs._Streams(91)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O, stride=2)]
    x = configs.image_input(st, W, H, I)
    want = oracle.conv_f64(x, spec[1]["w"], spec[1]["b"], stride=(2, 2), relu=True)
    for flag in ("0", "1"):
        os.environ["DR_DIRECT_VALU"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [1])
                dr.prepare(g)
                configs.feed_chw(nodes[0], x)
                assert g.lib.dR_apply(g.ptr)
                got = configs.fetch_chw(g)[0]
                line = ctypes.string_at(ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_void_p)(dr.node_struct(nodes[1]).printLayer)(nodes[1].ptr)).decode()
                assert ("split-operand" in line) == (split and flag == "0")
        finally:
            os.environ.pop("DR_DIRECT_VALU", None)
        assert_close(got, want, "DR_DIRECT_VALU=" + flag, terms=9 * I)


@pytest.mark.parametrize("case", ["means", "ragged", "mixed", "shared"])
def test_scalar_operations_in_front_of_a_concat(oracle, gpu, case):
    """Slices, scalar operations and the concat they fill in one launch (DR_FUSE_SCALAR=0: kernels apart): the same numbers."""
    w, h, c = (23, 17, 5) if case != "ragged" else (1, 1, 3)
    spec = [{"op": "feed", "shape": (w, h, c)}]
    def ew(src, kind, value):
        spec.append({"op": "scalar", "in": src, "kind": kind, "value": value})
        return len(spec) - 1
    def part(origin, shape):
        spec.append({"op": "slice", "in": 0, "origin": origin, "shape": shape})
        return len(spec) - 1
    if case == "mixed":                         # two channels, a box that has to be copied, and a tensor that is no slice
        base = ew(0, 2, 3.0)
        spec.append({"op": "slice", "in": base, "origin": (0, 0, 1), "shape": (w, h, 2)})
        ins = [ew(len(spec) - 1, 0, 1.5), ew(base, 1, 0.25)]
    elif case == "shared":                      # a slice with another reader stays
        one = part((0, 0, 2), (w, h, 1))
        ins = [ew(one, 3, 7.0), ew(one, 7, 2.0), ew(part((0, 0, 0), (w, h, 1)), 2, -1.0)]
    else:
        ins = [ew(part((0, 0, k), (w, h, 1)), 1, 10.0 * k) for k in (2, 0, 1)]
    spec.append({"op": "concat", "ins": ins, "dim": 2}); cat = len(spec) - 1
    if case == "mixed":
        spec.append({"op": "slice", "in": 0, "origin": (1, 2, 0), "shape": (5, 4, 2)}); box = len(spec) - 1
        a, b = ew(box, 1, 4.0), ew(box, 0, 4.0)
        spec.append({"op": "concat", "ins": [a, b], "dim": 2})
    outs = [cat] if case != "mixed" else [cat, len(spec) - 1]
    feeds = {0: configs.image_input(configs._Streams(79), w, h, c, 255.0)}
    want = oracle.run_spec(spec, feeds)
    for flag in ("1", "0"):
        os.environ["DR_FUSE_SCALAR"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, outs)
                dr.prepare(g)
                configs.feed_chw(nodes[0], feeds[0])
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                assert (dr.node_struct(nodes[ins[0]]).drLastKernelMs == 0.0) == (flag == "1")
                dr.graph_config(g).profilingGPU = 0
                assert g.lib.dR_apply(g.ptr)
                got = configs.fetch_chw(g)
        finally:
            os.environ.pop("DR_FUSE_SCALAR", None)
        for x, i in zip(got, outs):
            assert np.array_equal(x, want[i]) or np.abs(x - want[i]).max() <= 2.0 ** -23 * np.abs(want[i]).max()     # (a division's last bit)


def test_fc_chain_fused(oracle, gpu):
    """FC -> FC -> softmax: the finishing kernels of the two GEMVs disappear into their consumers
    (3 launches instead of 5) and the probabilities do not change by a bit."""
    rng = np.random.default_rng(5)
    spec = [{"op": "feed", "shape": (4, 4, 64)},
            {"op": "fc", "in": 0, "w": (rng.standard_normal((1024, 2048)) * 0.04).astype(np.float32), "b": (rng.standard_normal(2048) * 0.01).astype(np.float32), "relu": True},
            {"op": "fc", "in": 1, "w": (rng.standard_normal((2048, 1000)) * 0.03).astype(np.float32), "b": (rng.standard_normal(1000) * 0.01).astype(np.float32), "relu": False},
            {"op": "softmax", "in": 2}]
    x = rng.random((64, 4, 4), dtype=np.float32)
    res, launches = {}, {}
    for mode in ("1", "0"):
        os.environ["DR_FUSE_FC"] = mode
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [3])
                dr.prepare(g)
                configs.feed_chw(nodes[0], x)
                assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)          # captured pass, then its replay
                res[mode] = configs.fetch_chw(g)[0].copy()
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                launches[mode] = g.lib.drhip_timing_count()
                assert np.array_equal(configs.fetch_chw(g)[0], res[mode])
        finally:
            os.environ.pop("DR_FUSE_FC", None)
    assert launches == {"1": 3, "0": 5}
    assert np.array_equal(res["1"], res["0"])
    want = oracle.run_spec(spec, {0: x})
    assert rel_err(res["1"], want[3]) <= LAYER_TOL and int(res["1"].argmax()) == int(want[3].argmax())
    # Both GEMV outputs wanted by the caller as well: still 3 launches, the consumers store the
    # finished vectors into the producers' output buffers on the way.
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [1, 2, 3])
        dr.prepare(g)
        configs.feed_chw(nodes[0], x)
        assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)
        outs = [a.copy() for a in configs.fetch_chw(g)]
        dr.graph_config(g).profilingGPU = 1
        assert g.lib.dR_apply(g.ptr) and g.lib.drhip_timing_count() == 3
    assert np.array_equal(outs[2], res["0"])
    for k in range(3):
        assert_close(outs[k], want[k + 1], "fc chain %d" % k)


def test_conv_global_average_softmax_fused(oracle, gpu):
    """1x1 conv -> global average pooling -> softmax (SqueezeNet's tail): the pooling kernel and the
    convolution's tensor disappear; the pooled tensor, an output here, is stored by the softmax."""
    rng = np.random.default_rng(9)
    for tail in ("softmax", "fc"):
        spec = [{"op": "feed", "shape": (13, 11, 24)},
                {"op": "conv", "in": 0, "w": (rng.standard_normal((24, 70, 1, 1)) * 0.3).astype(np.float32), "b": (rng.standard_normal(70) * 0.05).astype(np.float32), "stride": (1, 1), "relu": True},
                {"op": "pool", "in": 1, "window": (13, 11, 1), "stride": (13, 11, 1), "kind": 1}]
        if tail == "softmax":
            spec.append({"op": "softmax", "in": 2})
        else:
            spec.append({"op": "fc", "in": 2, "w": (rng.standard_normal((70, 300)) * 0.2).astype(np.float32), "b": (rng.standard_normal(300) * 0.05).astype(np.float32), "relu": False})
        x = rng.random((24, 11, 13), dtype=np.float32)
        want = oracle.run_spec(spec, {0: x})
        res, launches = {}, {}
        for mode in ("1", "0"):
            os.environ["DR_FUSE_AVGPOOL"] = mode
            try:
                with dr.Environment() as env:
                    g = env.create_graph()
                    nodes = configs.build_graph(g, spec, [2, 3])
                    dr.prepare(g)
                    configs.feed_chw(nodes[0], x)
                    assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)
                    res[mode] = [a.copy() for a in configs.fetch_chw(g)]
                    dr.graph_config(g).profilingGPU = 1
                    assert g.lib.dR_apply(g.ptr)
                    launches[mode] = g.lib.drhip_timing_count()
            finally:
                os.environ.pop("DR_FUSE_AVGPOOL", None)
        assert launches["0"] - launches["1"] == 1, launches
        for k in range(2):
            assert rel_err(res["1"][k], want[2 + k]) <= LAYER_TOL and rel_err(res["1"][k], res["0"][k]) <= 1e-5


@pytest.mark.parametrize("W,H,I,O,tail", [(29, 23, 64, 70, "fc"), (5, 2, 60, 33, "fc"), (20, 20, 96, 9, "softmax"), (86, 94, 64, 32, "fc"), (92, 90, 64, 32, "fc")])
def test_global_average_behind_a_strided_layer(oracle, gpu, W, H, I, O, tail):
    """A 3x3/2 layer that leaves its pixel sums to the reader of the average behind it, up to 64 tiles of pixels, and the kernels apart
    (DR_FUSE_AVGPOOL=0)."""
    st = configs._Streams(93)
    Wo, Ho = W // 2, H // 2
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O, stride=2), {"op": "pool", "in": 1, "window": (Wo, Ho, 1), "stride": (Wo, Ho, 1), "kind": 1}]
    spec.append(configs._fc(st, 2, O, 300, False) if tail == "fc" else {"op": "softmax", "in": 2})
    x = configs.image_input(st, W, H, I)
    want, res, launches = oracle.run_spec(spec, {0: x}), {}, {}
    for mode in ("1", "0"):
        os.environ["DR_FUSE_AVGPOOL"] = mode
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, [2, 3])
                dr.prepare(g)
                configs.feed_chw(nodes[0], x)
                assert g.lib.dR_apply(g.ptr) and g.lib.dR_apply(g.ptr)
                res[mode] = [a.copy() for a in configs.fetch_chw(g)]
                dr.graph_config(g).profilingGPU = 1
                assert g.lib.dR_apply(g.ptr)
                launches[mode] = g.lib.drhip_timing_count()
        finally:
            os.environ.pop("DR_FUSE_AVGPOOL", None)
    assert launches["0"] - launches["1"] == (1 if Wo * Ho <= 64 * 32 else 0), launches
    for k in range(2):
        assert rel_err(res["1"][k], want[2 + k]) <= LAYER_TOL and rel_err(res["1"][k], res["0"][k]) <= 1e-5


def test_squeezenet_with_normalization_node(oracle, gpu):
    """Config 4 with its per-image normalisation moved into the graph: raw U[0,255) image in, a
    Normalization node (mean 0, deviation 1) in front of conv1."""
    spec, feeds, got = run_config("squeezenet", size=96, normalise_in_graph=True)
    assert spec[1]["op"] == "norm" and float(feeds[0].max()) > 100.0
    want = oracle.run_spec(spec, feeds)
    for i in got:
        assert_close(got[i], want[i], "node %d" % i)
    assert int(got[len(spec) - 1].argmax()) == int(want[-1].argmax())
    # the node alone, as an output
    _, _, only = run_config("squeezenet", outputs=[1], size=96, normalise_in_graph=True)
    assert_close(only[1], want[1], "normalization node")
    assert abs(float(only[1].astype(np.float64).mean())) < 1e-4 and abs(float(only[1].astype(np.float64).std()) - 1.0) < 1e-4


def test_normalization_behind_an_odd_volume_producer_in_a_concat(oracle, gpu):
    """feed 5x5x3 -> {1x1 conv (75 floats), Normalization} -> channel concat: a fused concat would put the
    Normalization node 300 bytes into the buffer, where its 16-byte accesses cannot go; the graph is valid
    in the reference (src/dR_nodes_transform.c:238-281) and must run here in either input order."""
    rng = np.random.default_rng(5)
    w = rng.standard_normal((3, 3, 1, 1)).astype(np.float32)
    x = rng.standard_normal((3, 5, 5)).astype(np.float32)
    for ins in ([1, 2], [2, 1]):
        spec = [{"op": "feed", "shape": (5, 5, 3)},
                {"op": "conv", "in": 0, "w": w, "b": None, "stride": (1, 1), "relu": False},
                {"op": "norm", "in": 0, "kind": 2, "mean": 0.0, "dev": 1.0},
                {"op": "concat", "ins": ins, "dim": 2}]
        want = oracle.run_spec(spec, {0: x})
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, [3])
            dr.prepare(g)
            configs.feed_chw(nodes[0], x)
            assert g.lib.dR_apply(g.ptr)
            got = configs.fetch_chw(g)[0]
            assert not g.lib.dR_prepare(g.ptr)               # one prepare per graph; refused, the plan stands
            assert g.lib.dR_apply(g.ptr)
            assert np.array_equal(configs.fetch_chw(g)[0], got)
        assert_close(got, want[3], "concat %s" % ins)


def test_layer_wider_than_the_packed_argument_fields(oracle, gpu):
    """A 3x3 layer on a 70000 x 2 map (a width beyond the 16-bit fields the matrix-core kernels carry their shapes
    in) runs on the general direct kernel and gives the oracle's values, with a pooling behind it unfused."""
    rng = np.random.default_rng(6)
    W, H = 70000, 2
    w = (rng.standard_normal((1, 2, 3, 3)) * 0.3).astype(np.float32)
    b = (rng.standard_normal(2) * 0.1).astype(np.float32)
    x = rng.standard_normal((1, H, W)).astype(np.float32)
    spec = [{"op": "feed", "shape": (W, H, 1)},
            {"op": "conv", "in": 0, "w": w, "b": b, "stride": (1, 1), "relu": True},
            {"op": "pool", "in": 1, "window": (3, 3, 1), "stride": (2, 2, 1), "kind": 0}]
    want = oracle.run_spec(spec, {0: x})
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [2])
        dr.prepare(g)
        configs.feed_chw(nodes[0], x)
        assert g.lib.dR_apply(g.ptr)
        got = configs.fetch_chw(g)[0]
    assert_close(got, want[2], "pool behind a 70000-wide 3x3 layer", terms=9)


def test_config4_squeezenet(oracle, gpu):
    spec, feeds, got = run_config("squeezenet", outputs=all_compute_nodes)
    want = check_layers(oracle, spec, feeds, got)
    probs, logits = got[len(spec) - 1].reshape(-1), got[len(spec) - 2].reshape(-1)
    wl = want[len(spec) - 2].reshape(-1)
    assert np.abs(logits - wl).max() <= LOGIT_TOL
    assert int(logits.argmax()) == int(wl.argmax()) and int(probs.argmax()) == int(want[-1].argmax())
    assert abs(float(probs.sum()) - 1) < 1e-4
    # fused-concat production run gives the same final numbers as the all-outputs run (the two fusions
    # that change a summation order switched off)
    _, _, prod = run_config("squeezenet", env_vars={"DR_FUSE_EXPAND": "0", "DR_FUSE_AVGPOOL": "0", "DR_FUSE_POOLIN": "0"})
    assert np.array_equal(prod[len(spec) - 1], got[len(spec) - 1])
    # and with the expand pairs of the 8 fire modules fused into single Winograd launches
    _, _, fused = run_config("squeezenet")
    assert rel_err(fused[len(spec) - 1], got[len(spec) - 1]) <= LAYER_TOL
    assert np.abs(fused[len(spec) - 2] - got[len(spec) - 2]).max() <= LOGIT_TOL
    assert int(fused[len(spec) - 1].argmax()) == int(got[len(spec) - 1].argmax())


def test_config5_vgg16(oracle, gpu):
    spec, feeds, got = run_config("vgg16", outputs=all_compute_nodes)
    want = check_layers(oracle, spec, feeds, got)
    logits, wl = got[len(spec) - 2].reshape(-1), want[len(spec) - 2].reshape(-1)
    assert np.abs(logits - wl).max() <= LOGIT_TOL
    assert int(logits.argmax()) == int(wl.argmax())
    probs = got[len(spec) - 1].reshape(-1)
    assert int(probs.argmax()) == int(want[-1].argmax()) and abs(float(probs.sum()) - 1) < 1e-4


@pytest.mark.parametrize("name,cls", [("tiger", 292), ("puzzle", 611)])
def test_stored_squeezenet_known_answer(oracle, gpu, name, cls):
    """The reference's only known answers: its stored SqueezeNet v1.1 on its two example images
    (examples/squeezenet-v1.1/squeezenet_deployed.c:199-207), loaded with dR_loadGraph."""
    img = np.load(os.path.join(GOLDEN, "%s_224_rgb_u8.npy" % name))
    chw = np.ascontiguousarray(img.transpose(2, 0, 1).astype(np.float32))
    with dr.Environment() as env:
        g = env.create_graph()
        nodes, feeds = dr.load_graph(g, os.path.join(GOLDEN, "squeezenet_whole"))
        assert len(nodes) == 48 and feeds[0].shape == [224, 224, 3]
        dr.mark_as_output(nodes[-1])
        dr.mark_as_output(nodes[-2])
        dr.prepare(g)
        configs.feed_chw(feeds[0], chw)
        assert g.lib.dR_apply(g.ptr)
        probs, pooled = [a.reshape(-1) for a in configs.fetch_chw(g)]
    want = oracle.run_graph_dir(os.path.join(GOLDEN, "squeezenet_whole"), chw)
    assert int(probs.argmax()) == cls
    assert np.abs(pooled - want[-2].reshape(-1)).max() <= LOGIT_TOL
    assert rel_err(probs, want[-1].reshape(-1)) <= LAYER_TOL


def test_python_frontend_hwc_roundtrip(oracle, gpu):
    """The wrapper's layout rules: HWC in, HWIO weights, HWC out (reference python wrapper :444-497,:559-562)."""
    rng = np.random.default_rng(3)
    x = rng.random((10, 12, 5), dtype=np.float32)                     # H, W, C
    w = (rng.standard_normal((3, 3, 5, 6)) * 0.2).astype(np.float32)  # H, W, I, O
    b = (rng.standard_normal(6) * 0.1).astype(np.float32)
    with dr.Environment() as env:
        g = env.create_graph("HWC")
        f = dr.feed_node(g, [10, 12, 5])
        c = dr.Conv2d(f, (3, 3, 5, 6), (1, 1, 1, 1), "relu", w, b)
        p = dr.Pooling(c, "max", (1, 2, 2, 1), (1, 2, 2, 1))
        dr.mark_as_output(p)
        dr.prepare(g)
        dr.feed_data(f, x)
        out = dr.apply(g)[0]
    want = oracle.pool(oracle.conv_winograd(x.transpose(2, 0, 1), w.transpose(2, 3, 0, 1), b, relu=True), (2, 2, 1), (2, 2, 1), 0)
    assert out.shape == (5, 6, 6)
    assert rel_err(out, want.transpose(1, 2, 0)) <= LAYER_TOL


def test_feed_and_download_through_pinned_staging(oracle, gpu):
    """dR_feedData goes through the graph's pinned staging area and does not wait for the bus: the caller's
    array must have been read when the call returns (it is overwritten right after each call here), feeds
    with an offset and back-to-back feeds must land where and in the order they were made, and
    DR_STAGING=0 (plain blocking copies) must give the same bytes."""
    spec, feeds, outs = configs.CONFIGS["conv3x3"](seed=5)
    x = feeds[0]
    want = oracle.run_spec(spec, feeds)[outs[0]]
    res = {}
    for flag in ("1", "0"):
        os.environ["DR_STAGING"] = flag
        try:
            with dr.Environment() as env:
                g = env.create_graph()
                nodes = configs.build_graph(g, spec, outs)
                dr.prepare(g)
                assert bool(dr.graph_struct(g).drStaging) == (flag == "1")
                lib, feed = g.lib, nodes[0]
                scratch = np.empty_like(x)
                fp = scratch.ctypes.data_as(dr.POINTER(dr.c_float))
                outs_seen = []
                for rep in range(3):
                    # garbage first, then the real image in two halves from ONE reused host array
                    scratch[...] = -1e30
                    lib.dR_feedData(g.ptr, feed.ptr, fp, 0, x.size)
                    half = x.size // 2
                    flat = scratch.reshape(-1)
                    flat[:half] = x.reshape(-1)[:half] * (rep + 1)
                    lib.dR_feedData(g.ptr, feed.ptr, fp, 0, half)
                    flat[:x.size - half] = x.reshape(-1)[half:] * (rep + 1)          # overwrites what was just fed
                    lib.dR_feedData(g.ptr, feed.ptr, fp, half, x.size - half)
                    scratch[...] = 7e30                                               # and again before the pass runs
                    assert lib.dR_apply(g.ptr)
                    outs_seen.append(configs.fetch_chw(g)[0])
                res[flag] = outs_seen
        finally:
            os.environ.pop("DR_STAGING", None)
    for rep in range(3):
        assert np.array_equal(res["1"][rep], res["0"][rep])
    assert_close(res["1"][0], want, "pass fed through the staging area")
    assert not np.array_equal(res["1"][0], res["1"][1])              # the scaled images really arrived


def test_linearity_at_full_size(gpu):
    """Size-independent property at VGG scale: a bias-free linear conv commutes with scaling and adds."""
    rng = np.random.default_rng(5)
    I, O, S = 128, 256, 56
    w = (rng.standard_normal((I, O, 3, 3)) * np.sqrt(2.0 / (9 * I))).astype(np.float32)
    spec = [{"op": "feed", "shape": (S, S, I)}, {"op": "conv", "in": 0, "w": w, "b": None, "stride": (1, 1), "relu": False}]
    a, b = rng.random((I, S, S), dtype=np.float32), rng.random((I, S, S), dtype=np.float32)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [1])
        dr.prepare(g)
        res = []
        for inp in (a, b, a + 2 * b):
            configs.feed_chw(nodes[0], inp)
            assert g.lib.dR_apply(g.ptr)
            res.append(configs.fetch_chw(g)[0])
    assert rel_err(res[2], res[0] + 2 * res[1]) <= LAYER_TOL


def _run_many(spec, outs, inputs, graph_mode, branches=False):
    old = os.environ.get("DR_HIPGRAPH")
    os.environ["DR_HIPGRAPH"] = "1" if graph_mode else "0"
    os.environ["DR_BRANCHES"] = "1" if branches else "0"
    try:
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, outs)
            dr.prepare(g)
            res = []
            for x in inputs:
                configs.feed_chw(nodes[0], x)          # eager blocking copy between the replays
                assert g.lib.dR_apply(g.ptr)
                res.append([a.copy() for a in configs.fetch_chw(g)])   # blocking download = sync
            tail = dr.graph_struct(g)
            used_graph = bool(tail.drGraphExec)
            _run_many.groups = tail.drBranchGroups
    finally:
        os.environ.pop("DR_BRANCHES", None)
        if old is None:
            os.environ.pop("DR_HIPGRAPH", None)
        else:
            os.environ["DR_HIPGRAPH"] = old
    return res, used_graph


@pytest.mark.parametrize("name", ["squeezenet", "vgg_conv3"])
def test_launch_graph_replays_equal_node_by_node(gpu, name):
    """dR_apply replays a captured hipGraph after the first pass.  Every replay -- with blocking copies
    and synchronisations of the program in between -- must equal the node-by-node result bit for bit."""
    spec, feeds, outs = configs.CONFIGS[name](seed=9)
    rng = np.random.default_rng(10)
    inputs = [feeds[0]] + [rng.random(feeds[0].shape, dtype=np.float32) for _ in range(4)] + [feeds[0]]
    eager, g0 = _run_many(spec, outs, inputs, graph_mode=False)
    replay, g1 = _run_many(spec, outs, inputs, graph_mode=True)
    assert not g0 and g1, "graph mode flags: eager run used a graph=%s, graph run used a graph=%s" % (g0, g1)
    assert _run_many.groups == 0
    if name == "squeezenet":
        # opt-in: the two expand convolutions of each of the 8 fire modules forked onto side streams
        forked, g2 = _run_many(spec, outs, inputs, graph_mode=True, branches=True)
        assert g2 and _run_many.groups == 8
        for a, b in zip(eager, forked):
            for x, y in zip(a, b):
                assert np.array_equal(x, y)
    for k, (a, b) in enumerate(zip(eager, replay)):
        for x, y in zip(a, b):
            assert np.array_equal(x, y), "replay %d differs from the node-by-node pass" % k
    assert np.array_equal(replay[0][0], replay[-1][0])


# ---------------------------------------------------------------------------------------------
# Random topologies: the buffer planner (live intervals, fused concats, pooled convolutions, joint
# expand launches, deferred GEMV reductions) must give the oracle's values whatever the graph looks
# like and whichever subset of nodes the caller reads.

def _random_spec(seed):
    rng = np.random.default_rng(seed)
    W, H, C = int(rng.integers(5, 30)), int(rng.integers(5, 30)), int(rng.integers(1, 9))
    spec = [{"op": "feed", "shape": (W, H, C)}]
    shapes = [(W, H, C)]

    def conv(src, k, cout, stride=1, relu=True):
        cin = shapes[src][2]
        w = (rng.standard_normal((cin, cout, k, k)) * np.sqrt(2.0 / (k * k * cin))).astype(np.float32)
        b = (rng.standard_normal(cout) * 0.05).astype(np.float32) if rng.random() < 0.8 else None
        spec.append({"op": "conv", "in": src, "w": w, "b": b, "stride": (stride, stride), "relu": relu})
        shapes.append((shapes[src][0] // stride, shapes[src][1] // stride, cout))
        return len(spec) - 1

    cur = 0
    for _ in range(int(rng.integers(3, 8))):
        w_, h_, c_ = shapes[cur]
        kind = rng.choice(["conv3", "conv1", "conv5", "pool2", "pool3", "fire", "branch3", "slice", "scalar", "norm"])
        if kind == "conv3":
            cur = conv(cur, 3, int(rng.integers(1, 40)), relu=bool(rng.integers(0, 2)))
        elif kind == "conv1":
            cur = conv(cur, 1, int(rng.integers(1, 40)))
        elif kind == "conv5" and min(w_, h_) >= 4:
            cur = conv(cur, 5, int(rng.integers(1, 12)), stride=int(rng.integers(1, 3)))
        elif kind in ("pool2", "pool3") and min(w_, h_) >= 2:
            k, s = (2, 2) if kind == "pool2" else (3, 2)
            spec.append({"op": "pool", "in": cur, "window": (k, k, 1), "stride": (s, s, 1), "kind": int(rng.integers(0, 2))})
            shapes.append((-(-w_ // s), -(-h_ // s), c_)); cur = len(spec) - 1
        elif kind == "fire":
            s = conv(cur, 1, int(rng.integers(1, 12)))
            e = int(rng.integers(1, 40))
            if e % 4 == 0:                           # what the launches of whole fire modules cover
                e = 32 if e % 8 == 0 else 64
            a, b = conv(s, 1, e), conv(s, 3, e)
            spec.append({"op": "concat", "ins": [a, b], "dim": 2}); shapes.append((w_, h_, 2 * e)); cur = len(spec) - 1
        elif kind == "branch3":                      # three producers, one of them read twice
            a, b = conv(cur, 3, int(rng.integers(1, 10))), conv(cur, 1, int(rng.integers(1, 10)))
            ins = [a, b, cur] if rng.random() < 0.5 else [b, a, a]
            spec.append({"op": "concat", "ins": ins, "dim": 2})
            shapes.append((w_, h_, sum(shapes[i][2] for i in ins))); cur = len(spec) - 1
        elif kind == "slice" and c_ >= 2:
            z0 = int(rng.integers(0, c_ - 1)); cz = int(rng.integers(1, c_ - z0 + 1))
            x0 = int(rng.integers(0, w_)); cw = int(rng.integers(1, w_ - x0 + 1))
            spec.append({"op": "slice", "in": cur, "origin": (x0, 0, z0), "shape": (cw, h_, cz)})
            shapes.append((cw, h_, cz)); cur = len(spec) - 1
        elif kind == "scalar":
            spec.append({"op": "scalar", "in": cur, "kind": int(rng.integers(0, 3)), "value": float(rng.uniform(0.5, 2.0))})
            shapes.append(shapes[cur]); cur = len(spec) - 1
        elif kind == "norm" and w_ * h_ * c_ > 1:
            spec.append({"op": "norm", "in": cur, "kind": int(rng.integers(0, 3)), "mean": 0.25, "dev": 1.5})
            shapes.append(shapes[cur]); cur = len(spec) - 1
    if rng.random() < 0.6:                           # classifier tail
        w_, h_, c_ = shapes[cur]
        for n_out, relu in ((int(rng.integers(200, 700)), True), (int(rng.integers(2, 300)), False)):
            k = shapes[cur][0] * shapes[cur][1] * shapes[cur][2]
            spec.append({"op": "fc", "in": cur, "w": (rng.standard_normal((k, n_out)) * np.sqrt(2.0 / k)).astype(np.float32),
                         "b": (rng.standard_normal(n_out) * 0.05).astype(np.float32), "relu": relu})
            shapes.append((n_out, 1, 1)); cur = len(spec) - 1
        spec.append({"op": "softmax", "in": cur}); shapes.append(shapes[cur]); cur = len(spec) - 1
    x = rng.random((C, H, W), dtype=np.float32) + np.float32(0.1)
    compute = [i for i in range(1, len(spec))]
    some = sorted(set([cur] + [int(i) for i in rng.choice(compute, size=min(2, len(compute)), replace=False)]))
    return spec, x, some


@pytest.mark.parametrize("seed", range(48 * int(os.environ.get("DR_SWEEP_SCALE", "1"))))    # (a one-off wider run: DR_SWEEP_SCALE=n)
def test_random_topologies(oracle, gpu, seed):
    spec, x, some = _random_spec(1000 + seed)
    want = oracle.run_spec(spec, {0: x})
    if not all(np.isfinite(a).all() for a in want if a is not None):
        pytest.skip("degenerate draw: a Normalization node met a constant tensor (deviation 0)")
    for outs in (some, [i for i in range(1, len(spec))]):
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, outs)
            dr.prepare(g)
            configs.feed_chw(nodes[0], x)
            for rep in range(2):                         # the captured pass, then a replay
                assert g.lib.dR_apply(g.ptr)
                got = configs.fetch_chw(g)
                for i, a in zip(outs, got):
                    assert a.shape == want[i].shape, (seed, i, spec[i]["op"], a.shape, want[i].shape)
                    if rel_err(a, want[i]) > LAYER_TOL:
                        k = int(np.abs(a - want[i]).argmax())
                        raise AssertionError("seed %d, %d outputs, pass %d: node %d (%s) of %s: element %d of %d is %r, the oracle has %r; "
                                             "%d elements differ by more than 1e-4 of the largest" % (
                                                 seed, len(outs), rep, i, spec[i]["op"], [s["op"] for s in spec], k, a.size, a.reshape(-1)[k],
                                                 want[i].reshape(-1)[k], int((np.abs(a - want[i]) > 1e-4 * np.abs(want[i]).max()).sum())))
                if len(outs) == len(spec) - 1:           # every tensor downloaded: judge each layer on the GPU's own inputs
                    step = oracle.run_spec(spec, {0: x}, inputs_from=dict(zip(outs, got)))
                    for i, a in zip(outs, got):
                        assert_close(a, step[i], "seed %d node %d (%s) of %s" % (seed, i, spec[i]["op"], [s["op"] for s in spec]),
                                     terms=spec_terms(spec[i]))


def _branches_spec(kind):
    """Graphs whose memory a launch touches beyond its own node's inputs and output, beside independent nodes that are planned into
    the same places: a pooled layer that averages, one pooled on load, a small layer inside its softmax."""
    st = configs._Streams(80)
    conv, pool = configs._conv, configs._maxpool
    if kind == "average":           # node 4 writes the average of node 5 where node 1 was, which node 3 in front of it reads
        spec = [{"op": "feed", "shape": (124, 70, 3)}, conv(st, 0, 1, 3, 16), {"op": "scalar", "in": 0, "kind": 2, "value": 0.5}, conv(st, 1, 1, 16, 9), conv(st, 2, 3, 3, 33),
                {"op": "pool", "in": 4, "window": (2, 2, 1), "stride": (2, 2, 1), "kind": 1}, conv(st, 3, 1, 9, 7), conv(st, 5, 1, 33, 5)]
    elif kind == "on load":         # node 6 writes where node 1 was, which node 3 in front of it pools on load
        spec = [{"op": "feed", "shape": (37, 29, 8)}, conv(st, 0, 5, 8, 16), pool(1, 3, 2), conv(st, 2, 1, 16, 24), conv(st, 0, 1, 8, 16), conv(st, 4, 3, 16, 12),
                conv(st, 5, 1, 12, 16), conv(st, 3, 1, 24, 6), conv(st, 6, 1, 16, 4)]
    elif kind == "joins":           # both leave partial tiles in the graph's one region for them
        spec = [{"op": "feed", "shape": (33, 31, 256)}, conv(st, 0, 3, 256, 512), conv(st, 0, 3, 256, 256)]
    else:                           # node 6 writes where node 1 was, which the softmax in front of it reads for the layer that it computes
        fc = lambda src, k, n: {"op": "fc", "in": src, "w": (st.next().standard_normal((k, n)) * k ** -0.5).astype(np.float32), "b": None, "relu": True}
        spec = [{"op": "feed", "shape": (60, 1, 1)}, fc(0, 60, 60), fc(1, 60, 20), {"op": "softmax", "in": 2}, fc(0, 60, 50), fc(4, 50, 60), fc(5, 60, 60), fc(6, 60, 30), {"op": "softmax", "in": 7}]
    read = {n["in"] for n in spec[1:]}
    return spec, [i for i in range(1, len(spec)) if i not in read]


@pytest.mark.parametrize("kind", ["average", "on load", "softmax", "joins"])
def test_branches_keep_off_memory_that_fusions_touch(oracle, gpu, kind):
    """Independent nodes on side streams (DR_BRANCHES=1): every replay as node by node."""
    spec, outs = _branches_spec(kind)
    rng = np.random.default_rng(4)
    w, h, c = spec[0]["shape"]
    inputs = [rng.standard_normal((c, h, w)).astype(np.float32) for _ in range(4)]
    eager, _ = _run_many(spec, outs, inputs, graph_mode=False)
    forked, used = _run_many(spec, outs, inputs, graph_mode=True, branches=True)
    assert used and (kind != "joins" or _run_many.groups == 0)
    want = oracle.run_spec(spec, {0: inputs[0]})
    for i, a in zip(outs, eager[0]):
        assert rel_err(a, want[i]) <= LAYER_TOL
    for a, b in zip(eager, forked):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


def test_joined_layers_share_one_region(oracle, gpu):
    """Halves, quarters, helpers and pieces of one graph, one behind the other, leave the region as they found it: every pass gives the same bits, and
    those of the layers in graphs of their own."""
    st = configs._Streams(81)
    conv = configs._conv
    spec = [{"op": "feed", "shape": (48, 48, 256)}, conv(st, 0, 3, 256, 256), conv(st, 1, 3, 256, 256), {"op": "pool", "in": 2, "window": (2, 2, 1), "stride": (2, 2, 1), "kind": 0},
            conv(st, 3, 3, 256, 512), conv(st, 4, 3, 512, 512), {"op": "pool", "in": 5, "window": (2, 2, 1), "stride": (2, 2, 1), "kind": 0}, conv(st, 6, 3, 512, 512)]
    x = np.random.default_rng(6).standard_normal((256, 48, 48)).astype(np.float32)
    (first, second, third), _ = _run_many(spec, [3, 4, 6, 7], [x, 2 * x, x], graph_mode=False)
    for a, b in zip(first, third):
        assert np.array_equal(a, b)
    got, src = first, x
    for layers, a in (((1, 2, 3), got[0]), ((4,), got[1]), ((5, 6), got[2]), ((7,), got[3])):
        own = [{"op": "feed", "shape": src.shape[::-1]}] + [dict(spec[i], **{"in": k}) for k, i in enumerate(layers)]
        alone, _ = _run_many(own, [len(own) - 1], [src], graph_mode=False)
        assert np.array_equal(alone[0][0], a), layers
        want = oracle.run_spec(own, {0: src})[-1]
        assert rel_err(a, want) <= LAYER_TOL
        src = a


def _kernels(nodes):
    """What the convolutions say that they run."""
    fn = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_void_p)
    texts = [ctypes.string_at(fn(dr.node_struct(n).printLayer)(n.ptr)).decode() for n in nodes if n.desc == "Conv2D"]
    return [next(l for l in t.splitlines() if "Kernel:" in l) for t in texts]


@pytest.mark.parametrize("replay", [False, True])
@pytest.mark.parametrize("what", ["infinite", "nan", "far below"])
@pytest.mark.parametrize("W,H,I,O", [(64, 66, 64, 256), (56, 56, 256, 256), (73, 28, 400, 476)])       # whole panels, halves behind which helpers join, thirds
def test_refilled_weights_that_two_parts_cannot_hold(oracle, gpu, monkeypatch, W, H, I, O, what, replay):
    """dR_Conv2d_setVariables and dR_fillBuffers on a prepared graph: weights that the first ones' bank has no room for are computed as a graph that was
    prepared with them computes them, and so are the next ones; the other layer stays as it is."""
    monkeypatch.setenv("DR_HIPGRAPH", "1" if replay else "0")
    st = configs._Streams(83)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O, relu=False), configs._conv(st, 0, 3, I, O, relu=False)]
    x = np.random.default_rng(7).standard_normal((I, H, W)).astype(np.float32)
    w0, b = spec[2]["w"], spec[2]["b"]
    w1 = np.ascontiguousarray(w0[:, ::-1]).copy()
    w1[3, 5, 1, 1] = {"infinite": np.inf, "nan": np.nan, "far below": 1.0}[what]
    if what == "far below":                         # (and samples that make up for it)
        w1[3] *= np.float32(2.0 ** -24)
    xs = x.copy()
    xs[3] *= np.float32(2.0 ** 24 if what == "far below" else 1.0)

    def run(g, nodes, a):
        configs.feed_chw(nodes[0], a)
        assert g.lib.dR_apply(g.ptr)
        return [y.copy() for y in configs.fetch_chw(g)]

    def refill(g, node, w):
        g.lib.dR_Conv2d_setVariables(node.ptr, dr._fptr(w), dr._fptr(b))
        assert g.lib.dR_fillBuffers(ctypes.c_void_p(g.ptr)) == 1

    with dr.Environment() as env:
        g, own = env.create_graph(), env.create_graph()
        nodes = configs.build_graph(g, spec, [1, 2])
        dr.prepare(g)
        before = _kernels(nodes)
        assert all("f16" in k for k in before)
        first = [run(g, nodes, a) for a in (x, xs, x)]
        refill(g, nodes[2], w1)
        got = [run(g, nodes, a) for a in (x, xs, x)]
        assert _kernels(nodes)[0] == before[0]
        there = configs.build_graph(own, spec[:2] + [dict(spec[2], w=w1)], [1, 2])
        dr.prepare(own)
        for a, old, now in zip((x, xs, x), first, got):
            alone = run(own, there, a)
            assert np.array_equal(now[0], old[0]) and np.array_equal(now[1], alone[1], equal_nan=True)
            if what == "far below":
                assert rel_err(now[1], oracle.conv_f64(a, w1, b, relu=False)) <= LAYER_TOL / 20
            else:
                assert np.isfinite(now[1][:5]).all() and not np.isfinite(now[1][5]).all()
        assert _kernels(nodes) == _kernels(there) and "f16" not in _kernels(nodes)[1]
        refill(g, nodes[2], w0)                     # weights that would fit again
        again = [run(g, nodes, a) for a in (x, xs, x)]
        for old, now in zip(first, again):
            assert np.array_equal(now[0], old[0]) and rel_err(now[1], old[1]) <= LAYER_TOL / 20
        assert all(np.array_equal(a, b) for a, b in zip(again[0], again[2]))


@pytest.mark.parametrize("what,kernel", [("fit", "f16"), ("zero filter", None), ("tiny filter", None)])
@pytest.mark.parametrize("W,H,I,O,other", [(56, 56, 256, 256, "Winograd F(2x2,3x3) MFMA"), (112, 112, 128, 128, "split-operand bf16 MFMA"), (33, 31, 256, 512, "split-operand bf16 MFMA")])
def test_samples_behind_filters_of_nothing_are_no_measure(oracle, gpu, W, H, I, O, other, what, kernel):
    """The samples of a column of tiles share a scale in the two-part kernel, which follows the largest.  Where that is of a channel whose filters are zero, or next
    to it, the outputs are made of the others, which the scale would leave few bits: such a layer is prepared in a form that holds all of them."""
    st = configs._Streams(87)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O)]
    x = np.random.default_rng(9).random((I, H, W), dtype=np.float32)
    if what != "fit":
        spec[1]["w"][7] *= np.float32(0.0 if what == "zero filter" else 2.0 ** -24)
        x[7] *= np.float32(2.0 ** 24)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [1])
        dr.prepare(g)
        assert (kernel or other) in _kernels(nodes)[0]
        configs.feed_chw(nodes[0], x)
        for _ in range(2):
            assert g.lib.dR_apply(g.ptr)
        got = configs.fetch_chw(g)[0]
    assert rel_err(got, oracle.conv_f64(x, spec[1]["w"], spec[1]["b"], relu=True)) <= LAYER_TOL / 20


@pytest.mark.parametrize("W,H,I,O,other", [(56, 56, 256, 256, "Winograd F(2x2,3x3) MFMA"), (33, 31, 256, 512, "split-operand bf16 MFMA")])
def test_two_parts_can_be_declined(oracle, gpu, monkeypatch, W, H, I, O, other):
    """DR_WINO_PAIR=0 in front of dR_prepare: the forms that hold all bits of an operand.  A flat map under one box filter shows them: three parts are exact to
    2^-22 there."""
    st = configs._Streams(89)
    spec = [{"op": "feed", "shape": (W, H, I)}, configs._conv(st, 0, 3, I, O, relu=False, bias=False)]
    x = np.full((I, H, W), 0.7310586, np.float32)
    spec[1]["w"][:] = np.float32(1 / 9)
    want = oracle.conv_f64(x, spec[1]["w"])
    for env_var, kernel in (("0", other), ("1", "f16"), (None, "f16")):
        monkeypatch.delenv("DR_WINO_PAIR", raising=False) if env_var is None else monkeypatch.setenv("DR_WINO_PAIR", env_var)
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, [1])
            dr.prepare(g)
            assert kernel in _kernels(nodes)[0]
            configs.feed_chw(nodes[0], x)
            assert g.lib.dR_apply(g.ptr)
            got = configs.fetch_chw(g)[0]
        assert rel_err(got, want) <= LAYER_TOL / 20 and ("bf16" not in kernel or rel_err(got, want) <= 2.0 ** -21)


@pytest.mark.parametrize("W,H,S,E,kernel", [(56, 56, 64, 256, "Winograd F(2x2,3x3) MFMA"), (112, 112, 64, 128, "split-operand bf16 MFMA"), (33, 31, 256, 256, "split-operand bf16 MFMA")])
def test_expand_pairs_keep_three_parts(oracle, gpu, W, H, S, E, kernel):
    """The 3x3 layer of a pair that is one launch has the kernel that the planner prices, also with weights that two parts could hold."""
    st = configs._Streams(85)
    spec = [{"op": "feed", "shape": (W, H, S)}, configs._conv(st, 0, 1, S, E), configs._conv(st, 0, 3, S, E), {"op": "concat", "ins": [1, 2], "dim": 2}]
    spec[1]["w"] = spec[1]["w"] + np.copysign(np.float32(0.01), spec[1]["w"])
    x = np.random.default_rng(8).standard_normal((S, H, W)).astype(np.float32)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, [3])
        assert g.lib.drhip_conv3x3_winograd_pair_pick_variant(W, H, S, 2 * E)
        for n in (1, 2):
            w = spec[n]["w"]
            assert g.lib.drhip_winograd_pair_fits(w.ctypes.data_as(ctypes.c_void_p), S, E, w.shape[2] * w.shape[3])
        dr.prepare(g)
        assert kernel in _kernels(nodes)[1]
        configs.feed_chw(nodes[0], x)
        assert g.lib.dR_apply(g.ptr)
        got = configs.fetch_chw(g)[0]
    assert rel_err(got, oracle.run_spec(spec, {0: x})[3]) <= LAYER_TOL


@pytest.mark.parametrize("W,H,I,O,helpers", [(33, 31, 256, 512, False), (56, 56, 256, 256, True), (48, 48, 128, 256, True)])
def test_joined_layers_of_two_graphs_on_two_streams(lib, gpu, W, H, I, O, helpers):
    """Pieces of a split-operand layer, and panels and their helpers, wait for each other inside the launch.  Two graphs with such a layer, each on its
    own stream, run at the same time: every pass as if it were alone, and no piece waited in vain."""
    rng = np.random.default_rng(3)
    split = lib.drhip_conv3x3_winograd_split_pick_variant(W, H, I, O)
    assert split == 0 and lib.drhip_conv3x3_winograd_pick_variant(W, H, I, O) == 0x2c01 if helpers else split >> 12
    late = ctypes.c_uint(0)
    assert lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)) == 0
    before = late.value
    with dr.Environment() as one, dr.Environment() as two:
        graphs, alone, streams = [], [], []
        for env in (one, two):
            g = env.create_graph()
            streams.append(ctypes.c_void_p())
            assert lib.drhip_stream_create(ctypes.byref(streams[-1])) == 0
            lib.dR_setClEnvironment(ctypes.c_void_p(g.ptr), None, None, streams[-1], None)
            x = dr.feed_node(g, [H, W, I])
            c = dr.Conv2d_raw(x, (rng.standard_normal((I, O, 3, 3)) * 0.03).astype(np.float32), None, (1, 1), "relu")
            dr.mark_as_output(c)
            dr.prepare(g)
            dr.feed_data(x, rng.standard_normal((H, W, I)).astype(np.float32))
            alone.append(dr.apply(g)[0])
            graphs.append(g)
        for _ in range(5):
            for _ in range(20):
                for g in graphs:
                    assert lib.dR_apply(g.ptr)
            for g, want in zip(graphs, alone):
                assert np.array_equal(dr.download_outputs(g)[0], want)
    for st in streams:
        assert lib.drhip_stream_destroy(st) == 0
    assert lib.drhip_conv3x3_winograd_join_timeouts(ctypes.byref(late)) == 0 and late.value == before
