"""Host-side logic of libdeepracin.so that needs no GPU: exported C-ABI, stored-format reader/writer,
execution order, buffer planner, error behaviour, list cursor rules.  No compute call is made here.
"""
import ctypes
import filecmp
import os
import re

import numpy as np
import pytest

import deepracin_amd as dr
from deepracin_amd import configs
from conftest import GOLDEN, ROOT

MODEL = os.path.join(GOLDEN, "squeezenet_whole")


# ---------------------------------------------------------------------------------------------
# C-ABI surface
# ---------------------------------------------------------------------------------------------

def declared_symbols():
    names = set()
    for header in ("deepRACIN.h", "dR_nodes.h", "dr_hip.h"):
        text = open(os.path.join(ROOT, "include", header)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        for m in re.finditer(r"\b((?:dR|drhip)_\w+)\s*\(", text):
            names.add(m.group(1))
    return sorted(names)


def test_library_exports_every_declared_symbol(lib):
    syms = declared_symbols()
    assert len(syms) > 60
    raw = ctypes.CDLL(dr.LIB_PATH)
    missing = [s for s in syms if not hasattr(raw, s)]
    assert not missing, "declared in include/*.h but not exported: %s" % missing
    for must in ("dR_NewGraph", "dR_loadGraph", "dR_feedData", "dR_prepare", "dR_apply", "dR_getOutputBuffers",
                 "dR_downloadArray", "drhip_conv3x3_winograd_f32", "drhip_conv1x1_f32", "drhip_fc_f32"):
        assert must in syms


def test_every_symbol_the_reference_python_wrapper_looks_up_resolves(lib):
    """tests/golden/ref_wrapper_symbols.txt lists the lib.dR_* names of the reference's ctypes front-end
    (python/deepracin/__init__.py.in:36-218 bind at import; a few more are looked up when called).  All
    must resolve, or the unmodified wrapper stops with AttributeError before any graph is built."""
    names = open(os.path.join(GOLDEN, "ref_wrapper_symbols.txt")).read().split()
    assert len(names) >= 35 and "dR_MaskDependentFilter" in names and "dR_apply" in names
    raw = ctypes.CDLL(dr.LIB_PATH)
    missing = [s for s in names if not hasattr(raw, s)]
    assert not missing, "looked up by the reference wrapper but not exported: %s" % missing


def test_constructors_outside_the_layer_path_refuse(lib, capfd):
    """Image-filter, two-tensor, RoI, colour, upscaling, label and crop constructors exist for the wrapper's
    import only: they append nothing and return NULL."""
    raw = ctypes.CDLL(dr.LIB_PATH)
    g = lib.dR_NewGraph()
    sh = (ctypes.c_int * 4)(3, 3, 1, 1)
    for name, args in (("dR_RGB2gray", (g, None)), ("dR_ResolveRoI", (g, None, sh)), ("dR_CropOrPad", (g, None, sh)),
                       ("dR_ElemWise2Operation", (g, None, None, 0)), ("dR_Upscaling", (g, None, 0, 2, 2)),
                       ("dR_MaskDependentFilter", (g, None, None, sh)), ("dR_PerPixelFilter", (g, None, None, sh, sh)),
                       ("dR_LabelCreation", (g, None, 0, ctypes.c_float(0), ctypes.c_float(0), ctypes.c_float(0)))):
        f = getattr(raw, name)
        f.restype = ctypes.c_void_p
        assert f(*args) is None, name
    raw.dR_MaskDependentFilter_setVariables.restype = None
    raw.dR_MaskDependentFilter_setVariables(None, None, None)
    out = capfd.readouterr().out
    assert out.count("outside the CNN layer path") == 9


def test_no_device_is_reported_not_faked(lib):
    # on a machine without a GPU the device layer says so; on a GPU box it initialises
    info = dr.DeviceInfo()
    rc = lib.drhip_init(0, info)
    if lib.drhip_device_count() == 0:
        assert rc == -3 and b"no HIP device" in lib.drhip_last_error()
    else:
        assert rc == 0 and info.arch.startswith(b"gfx950")


# ---------------------------------------------------------------------------------------------
# stored format
# ---------------------------------------------------------------------------------------------

def test_load_stored_model_and_roundtrip_bytes(lib, tmp_path):
    with dr.Environment() as env:
        g = env.create_graph()
        nodes, feeds = dr.load_graph(g, MODEL)
        assert len(nodes) == 48 and len(feeds) == 1 and feeds[0].shape == [224, 224, 3]
        types = [dr.node_struct(n).type for n in nodes]
        assert types.count(3) == 26 and types.count(16) == 9 and types.count(15) == 3      # conv, concat, slice
        assert [dr.node_struct(n).layerID for n in nodes] == list(range(48))
        dr.save_graph(g, str(tmp_path))
    out = tmp_path / "dr_graph_export"
    assert filecmp.cmp(str(out / "graph.dr"), os.path.join(MODEL, "graph.dr"), shallow=False)
    for i in range(52):
        assert filecmp.cmp(str(out / ("%d.var" % i)), os.path.join(MODEL, "%d.var" % i), shallow=False)
    # and the written model loads again into the same topology
    with dr.Environment() as env:
        g = env.create_graph()
        nodes2, _ = dr.load_graph(g, str(out))
        assert len(nodes2) == 48


def test_saved_synthetic_graph_has_reference_grammar(lib, tmp_path):
    spec, _, outs = configs.fire_module(seed=3, size=9, cin=8, squeeze=4, expand=8)
    with dr.Environment() as env:
        g = env.create_graph()
        configs.build_graph(g, spec, outs)
        dr.save_graph(g, str(tmp_path))
    text = open(tmp_path / "dr_graph_export" / "graph.dr").read()
    lines = text.split("\n")
    assert lines[0] == "deepRACIN graph: 5 nodes, 1 feed nodes" and text.endswith("\n")
    assert lines[1:6] == ["Node 0: DataFeedNode", "params: 9 9 8", "previous_nodes:", "next_nodes: 1", "variable_files:"]
    assert lines[6:11] == ["Node 1: Conv2D", "params: 1 1 1 1 8 4 1 1 1 1", "previous_nodes: 0", "next_nodes: 2 3",
                           "variable_files: 0.var 1.var"]
    assert lines[21:26] == ["Node 4: Concat", "params: 2 2", "previous_nodes: 2 3", "next_nodes:", "variable_files:"]
    w = np.fromfile(tmp_path / "dr_graph_export" / "0.var", dtype="<f4")
    assert np.array_equal(w, spec[1]["w"].reshape(-1))


def _expect_load_failure(tmp_path, text, files=()):
    d = tmp_path / "m"
    d.mkdir(exist_ok=True)
    (d / "graph.dr").write_text(text)
    for name, arr in files:
        np.asarray(arr, "<f4").tofile(d / name)
    with dr.Environment() as env:
        g = env.create_graph()
        with pytest.raises(RuntimeError):
            dr.load_graph(g, str(d))


def test_loader_error_paths(lib, tmp_path):
    feed = "Node 0: DataFeedNode\nparams: 4 4 2\nprevious_nodes:\nnext_nodes: 1\nvariable_files:\n"
    # missing file
    with dr.Environment() as env:
        g = env.create_graph()
        with pytest.raises(RuntimeError):
            dr.load_graph(g, str(tmp_path / "nowhere"))
    # unknown node type
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Bogus\nparams:\nprevious_nodes: 0\nnext_nodes:\nvariable_files:\n")
    # node type of the reference that is outside the CNN layer path
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: RGB2Gray\nparams:\nprevious_nodes: 0\nnext_nodes:\nvariable_files:\n")
    # wrong parameter count for a conv
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Conv2D\nparams: 1 1 3 3 2\nprevious_nodes: 0\nnext_nodes:\nvariable_files: 0.var 1.var\n",
                         [("0.var", np.zeros(36)), ("1.var", np.zeros(2))])
    # variable file shorter than the tensor it should hold
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Conv2D\nparams: 1 1 3 3 2 2 1 1 1 1\nprevious_nodes: 0\nnext_nodes:\nvariable_files: 0.var 1.var\n",
                         [("0.var", np.zeros(10)), ("1.var", np.zeros(2))])
    # forward reference
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Softmax\nparams:\nprevious_nodes: 1\nnext_nodes:\nvariable_files:\n")
    # a loader only fills an empty graph
    with dr.Environment() as env:
        g = env.create_graph()
        dr.feed_node(g, [4, 4, 2])
        with pytest.raises(RuntimeError):
            dr.load_graph(g, MODEL)


def test_normalization_node_format_roundtrip(lib, tmp_path):
    """graph.dr grammar of the Normalization node: 3 parameters `type mean dev` written with %d %f %f
    (reference src/dR_nodes_misc.c:1103-1105), read back into the same node."""
    with dr.Environment() as env:
        g = env.create_graph()
        f = dr.feed_node(g, [6, 5, 3])
        n = dr.Normalization(f, "target_mean_dev", 0.25, 2.0)
        dr.Softmax(n)
        dr.save_graph(g, str(tmp_path))
    lines = open(tmp_path / "dr_graph_export" / "graph.dr").read().split("\n")
    assert lines[6:11] == ["Node 1: Normalization", "params: 2 0.250000 2.000000", "previous_nodes: 0", "next_nodes: 2", "variable_files:"]
    with dr.Environment() as env:
        g = env.create_graph()
        nodes, feeds = dr.load_graph(g, str(tmp_path / "dr_graph_export"))
        assert [dr.node_struct(x).type for x in nodes] == [12, 7, 14]          # feed, normalization, softmax
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        s = dr.node_struct(nodes[1]).oshape
        f0 = dr.node_struct(nodes[0]).oshape
        assert (s.s0, s.s1, s.s2) == (f0.s0, f0.s1, f0.s2) and sorted((s.s0, s.s1, s.s2)) == [3, 5, 6]
        dr.save_graph(g, str(tmp_path / "again"))
    assert filecmp.cmp(str(tmp_path / "again" / "dr_graph_export" / "graph.dr"), str(tmp_path / "dr_graph_export" / "graph.dr"), shallow=False)
    # wrong parameter count / unknown type are refused
    feed = "Node 0: DataFeedNode\nparams: 4 4 2\nprevious_nodes:\nnext_nodes: 1\nvariable_files:\n"
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Normalization\nparams: 2 0.0\nprevious_nodes: 0\nnext_nodes:\nvariable_files:\n")
    _expect_load_failure(tmp_path, "deepRACIN graph: 2 nodes, 1 feed nodes\n" + feed +
                         "Node 1: Normalization\nparams: 5 0.0 1.0\nprevious_nodes: 0\nnext_nodes:\nvariable_files:\n")


# ---------------------------------------------------------------------------------------------
# prepare-time errors (host side only: fail before any device call)
# ---------------------------------------------------------------------------------------------

def test_prepare_and_shape_errors(lib):
    with dr.Environment() as env:
        g = env.create_graph()
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 0            # no feed node
        mem = (ctypes.c_void_p * 10)()
        assert lib.dR_getOutputBuffers(g.ptr, mem) == 0                 # not prepared
        assert lib.dR_apply(g.ptr) == 0
    rng = np.random.default_rng(0)
    w = rng.standard_normal((2, 3, 3, 3)).astype(np.float32)
    with dr.Environment() as env:                                       # conv stride larger than the image -> zero shape
        g = env.create_graph()
        spec = [{"op": "feed", "shape": (2, 2, 2)}, {"op": "conv", "in": 0, "w": w, "b": None, "stride": (4, 4), "relu": False}]
        configs.build_graph(g, spec, [1])
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 0
    with dr.Environment() as env:                                       # FC input size mismatch
        g = env.create_graph()
        spec = [{"op": "feed", "shape": (2, 2, 2)}, {"op": "fc", "in": 0, "w": np.zeros((9, 4), np.float32), "b": None, "relu": False}]
        configs.build_graph(g, spec, [1])
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 0
    with dr.Environment() as env:                                       # conv channel mismatch
        g = env.create_graph()
        spec = [{"op": "feed", "shape": (4, 4, 3)}, {"op": "conv", "in": 0, "w": w, "b": None, "stride": (1, 1), "relu": False}]
        configs.build_graph(g, spec, [1])
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 0


def test_shape_rules(lib):
    # conv: floor(in/stride); pool: ceil(in/stride); fc: (N,1,1)   (reference conv2d.c:115, pooling.c:201, fc.c:302)
    spec, _, outs = configs.squeezenet11(seed=1)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, outs)
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        shapes = [(dr.node_struct(n).oshape.s0, dr.node_struct(n).oshape.s1, dr.node_struct(n).oshape.s2) for n in nodes]
    _, want = configs.flops(spec)
    assert shapes == [tuple(s) for s in want]
    assert shapes[1] == (112, 112, 64) and shapes[2] == (56, 56, 64) and shapes[-1] == (1, 1, 1000)
    with dr.Environment() as env:
        g = env.create_graph()
        spec = [{"op": "feed", "shape": (55, 55, 4)}, {"op": "pool", "in": 0, "window": (3, 3, 1), "stride": (2, 2, 1), "kind": 0}]
        nodes = configs.build_graph(g, spec, [1])
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        s = dr.node_struct(nodes[1]).oshape
        assert (s.s0, s.s1, s.s2) == (28, 28, 4)


# ---------------------------------------------------------------------------------------------
# execution order and buffer plan
# ---------------------------------------------------------------------------------------------

def reference_order(spec):
    """The reference's work-list walk (src/dR_core.c:121-211) restated over a layer list."""
    consumers = {i: [] for i in range(len(spec))}
    inputs = {}
    for i, n in enumerate(spec):
        ins = n.get("ins", [n["in"]] if "in" in n else [])
        inputs[i] = ins
        for j in ins:
            consumers[j].append(i)
    done, queued, work, order = set(), set(), [], []
    for i, n in enumerate(spec):
        if n["op"] == "feed":
            done.add(i)
            for c in consumers[i]:
                if c not in queued:
                    queued.add(c); work.append(c)
    while work:
        n = work.pop(0)
        if not all(j in done for j in inputs[n]):
            work.append(n)
            continue
        done.add(n); order.append(n)
        for c in consumers[n]:
            if c not in queued:
                queued.add(c); work.append(c)
    return order


class FullHandler(ctypes.Structure):
    pass


FullHandler._fields_ = [("outputFor", ctypes.c_void_p), ("size", ctypes.c_int), ("numberOfDependencies", ctypes.c_int),
                        ("bufptr", ctypes.c_void_p), ("buf", ctypes.c_void_p), ("outputBuf", ctypes.c_int),
                        ("regionOfInterest", ctypes.c_int), ("useIndexBufferForRoI", ctypes.c_int),
                        ("indexBuffer", ctypes.c_void_p), ("index", ctypes.c_int), ("roiOrigin", dr.Shape3),
                        ("drViewOf", ctypes.POINTER(FullHandler)), ("drViewOffset", ctypes.c_int),
                        ("drFirstDef", ctypes.c_int), ("drLastUse", ctypes.c_int), ("drPinned", ctypes.c_int)]


def plan_of(graph, nodes):
    """[(physical id, offset, size)] per node after dR_planBuffers."""
    out = []
    for n in nodes:
        hp = ctypes.cast(dr.node_struct(n).outputBuf, ctypes.POINTER(FullHandler))
        h = hp.contents
        if h.drViewOf:
            out.append((ctypes.addressof(h.drViewOf.contents), h.drViewOffset, h.size, h.drViewOf.contents.size))
        else:
            out.append((ctypes.addressof(h), 0, None, h.size))
    return out


@pytest.mark.parametrize("name", ["fire", "vgg_conv3", "squeezenet", "stored"])
def test_schedule_order_and_buffer_plan(lib, oracle, name):
    with dr.Environment() as env:
        g = env.create_graph()
        if name == "stored":
            nodes, _ = dr.load_graph(g, MODEL)
            spec = oracle.parse_graph_dir(MODEL)
            outs = [47]
            dr.mark_as_output(nodes[47])
        else:
            kw = {"size": 32} if name == "squeezenet" else {}
            spec, _, outs = configs.CONFIGS[name](seed=2, **kw)
            nodes = configs.build_graph(g, spec, outs)
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        pos = [dr.node_struct(n).drSchedulePos for n in nodes]
        order = [i for _, i in sorted((p, i) for i, p in enumerate(pos) if p >= 0)]
        assert order == reference_order(spec)
        assert lib.dR_planBuffers(g.ptr) == 1
        plan = plan_of(g, nodes)
        vol = [dr.node_struct(n).oshape.s0 * dr.node_struct(n).oshape.s1 * dr.node_struct(n).oshape.s2 for n in nodes]

    inputs = {i: n.get("ins", [n["in"]] if "in" in n else []) for i, n in enumerate(spec)}
    last_use = {i: pos[i] for i in range(len(spec))}
    for i, ins in inputs.items():
        for j in ins:
            last_use[j] = max(last_use[j], pos[i])
    # a 1x1 layer behind a 3x3/2 max pool that nobody else reads pools while it loads: it reads the tensor
    # in FRONT of the pooling node, which therefore has to stay intact until that layer has run
    for i, n in enumerate(spec):
        if n["op"] == "conv" and tuple(n["w"].shape[2:]) == (1, 1) and spec[n["in"]]["op"] == "pool":
            pl = spec[n["in"]]
            if tuple(pl["window"]) == (3, 3, 1) and tuple(pl["stride"]) == (2, 2, 1) and pl["kind"] == 0:
                last_use[pl["in"]] = max(last_use[pl["in"]], pos[i])
    fused_into = {}
    # a max pool stored by the convolution in front of it: the convolution then owns no tensor of
    # its own, only the pooled one in the pooling node's buffer
    for i, n in enumerate(spec):
        if n["op"] == "pool" and plan[n["in"]][0] == plan[i][0]:
            j = n["in"]
            # 2x2/2 behind a Winograd convolution, or 3x3/2 behind a first layer (3x3 filter, <= 4 input channels)
            assert spec[j]["op"] == "conv" and tuple(n["stride"]) == (2, 2, 1) and n["kind"] == 0
            k = spec[j]["w"].shape
            assert tuple(n["window"]) == (2, 2, 1) or (tuple(n["window"]) == (3, 3, 1) and k[0] <= 4 and tuple(k[2:]) == (3, 3))
            assert plan[j][1] == plan[i][1] == 0 and j not in outs
            assert sum(1 for k in inputs if j in inputs[k]) == 1
            fused_into[j] = i
            vol[j] = vol[i]
    if name == "vgg_conv3":
        assert any(spec[i]["op"] == "pool" for i in fused_into.values()), "max pools should be absorbed by their convolutions"
    region = {i: (plan[i][0], plan[i][1], plan[i][1] + vol[i]) for i in range(len(spec))}
    for i in range(len(spec)):
        assert plan[i][3] >= plan[i][1] + vol[i], "node %d does not fit its buffer" % i
    for i, n in enumerate(spec):
        if n["op"] == "concat" and all(plan[j][0] == plan[i][0] for j in n["ins"]):
            off = 0
            for j in n["ins"]:
                assert plan[j][1] == off, "producer %d not at its channel offset" % j
                off += vol[j]
                fused_into[j] = i
    if name in ("fire", "squeezenet", "stored"):
        assert fused_into, "channel concats should absorb their producers"

    def overlaps(a, b):
        return a[0] == b[0] and a[1] < b[2] and b[1] < a[2]

    # brute-force liveness: when node i writes, no other tensor that is still needed may share its bytes
    for i in range(len(spec)):
        if pos[i] < 0:
            continue
        for j in range(len(spec)):
            if j == i or fused_into.get(j) == i or fused_into.get(i) == j:
                continue
            if j in fused_into and i in fused_into and fused_into[i] == fused_into[j]:
                assert not overlaps(region[i], region[j])
                continue
            live = (pos[j] < pos[i] <= last_use[j]) or spec[j]["op"] == "feed" or j in outs
            if live and pos[j] <= pos[i]:
                assert not overlaps(region[i], region[j]), "node %d overwrites live tensor %d" % (i, j)
    # feed and output tensors own their storage
    pinned = [i for i, n in enumerate(spec) if n["op"] == "feed"] + list(outs)
    for i in pinned:
        assert sum(1 for j in range(len(spec)) if plan[j][0] == plan[i][0] and fused_into.get(j) != i) == 1
    # and recycling does happen on the deep nets
    if name in ("squeezenet", "stored"):
        assert len({p[0] for p in plan}) < len(spec) // 2


def test_tensors_that_fusions_remove_have_no_memory(lib):
    """SqueezeNet's fire modules leave sums in workspaces: of its tensors there is memory for the image, the last module's outputs
    (pixel by pixel) and the outputs of the graph, and for all of them where every layer is an output."""
    class Handler(ctypes.Structure):
        _fields_ = FullHandler._fields_ + [("drUnstored", ctypes.c_int)]

    def planned(outputs):
        spec, _, outs = configs.CONFIGS["squeezenet"](seed=2)
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, outs if outputs is None else [i for i in range(1, len(spec))])
            assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1 and lib.dR_planBuffers(g.ptr) == 1
            stored, removed = {}, 0
            for n in nodes:
                h = ctypes.cast(dr.node_struct(n).outputBuf, ctypes.POINTER(Handler))
                if h.contents.drViewOf:
                    h = ctypes.cast(h.contents.drViewOf, ctypes.POINTER(Handler))
                if h.contents.drUnstored:
                    removed += 1
                else:
                    stored[ctypes.addressof(h.contents)] = h.contents.size
            return len(nodes), removed, sum(stored.values())
    nodes, removed, floats = planned(None)
    assert removed > nodes // 2 and floats <= 224 * 224 * 3 + 14 * 14 * 512 + 2 * 1000 + 14 * 14 * 64
    assert planned("all")[1] == 0


def _odd_offset_norm_spec():
    """feed 5x5x3 -> {1x1 conv to 3 channels (75 floats), Normalization} -> channel concat."""
    rng = np.random.default_rng(5)
    w = rng.standard_normal((3, 3, 1, 1)).astype(np.float32)
    spec = [{"op": "feed", "shape": (5, 5, 3)},
            {"op": "conv", "in": 0, "w": w, "b": None, "stride": (1, 1), "relu": False},
            {"op": "norm", "in": 0, "kind": 2, "mean": 0.0, "dev": 1.0},
            {"op": "concat", "ins": [1, 2], "dim": 2}]
    x = rng.standard_normal((3, 5, 5)).astype(np.float32)
    return spec, x


def test_normalization_is_never_planned_at_an_unaligned_concat_offset(lib):
    """The normalization kernels move 16 bytes per lane.  Behind a producer of 75 floats the fused concat
    would put the Normalization node at byte offset 300: the planner must not fuse such a concat (and may
    fuse it when the normalization comes first, at offset 0)."""
    spec, _ = _odd_offset_norm_spec()
    for ins, fused in (([1, 2], False), ([2, 1], True)):
        spec[3] = {"op": "concat", "ins": ins, "dim": 2}
        with dr.Environment() as env:
            g = env.create_graph()
            nodes = configs.build_graph(g, spec, [3])
            assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1 and lib.dR_planBuffers(g.ptr) == 1
            plan = plan_of(g, nodes)
        assert (plan[2][0] == plan[3][0]) == fused
        if plan[2][0] == plan[3][0]:
            assert plan[2][1] % 4 == 0


def test_second_prepare_is_refused_not_silently_empty(lib, capfd):
    """A graph is prepared once.  A second walk would find every node already queued and schedule nothing:
    the call must say so and return FALSE, and the first schedule must still stand."""
    spec, _, outs = configs.CONFIGS["fire"](seed=3)
    with dr.Environment() as env:
        g = env.create_graph()
        nodes = configs.build_graph(g, spec, outs)
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        first = [dr.node_struct(n).drSchedulePos for n in nodes]
        capfd.readouterr()
        assert lib.dR_prepare(g.ptr) == 0
        out = capfd.readouterr().out
        assert "scheduled before" in out and "prepared already" not in out      # (scheduled by hand, never prepared)
        assert [dr.node_struct(n).drSchedulePos for n in nodes] == first


# ---------------------------------------------------------------------------------------------
# list cursor rules and helpers
# ---------------------------------------------------------------------------------------------

def test_list_cursor_rules():
    raw = ctypes.CDLL(dr.LIB_PATH)
    vp = ctypes.c_void_p
    raw.dR_list_createEmptyList.restype = vp
    raw.dR_list_next.restype = vp
    raw.dR_list_pop.restype = vp
    for f in (raw.dR_list_append, raw.dR_list_removeFirstOcc):
        f.argtypes = [vp, vp]
    for f in (raw.dR_list_next, raw.dR_list_pop, raw.dR_list_resetIt, raw.dR_list_cleanup):
        f.argtypes = [vp]
    l = raw.dR_list_createEmptyList()
    for v in (11, 22, 33, 44):
        raw.dR_list_append(l, v)
    assert [raw.dR_list_next(l) for _ in range(5)] == [11, 22, 33, 44, None]      # wraps to reset after the end
    assert raw.dR_list_next(l) == 11 and raw.dR_list_next(l) == 22
    assert raw.dR_list_removeFirstOcc(l, 22) == 1                                  # remove under the cursor
    assert raw.dR_list_next(l) == 33                                               # successor comes next
    raw.dR_list_resetIt(l)
    assert raw.dR_list_next(l) == 11
    assert raw.dR_list_removeFirstOcc(l, 11) == 1                                  # remove the head under the cursor
    assert raw.dR_list_next(l) == 33
    assert raw.dR_list_pop(l) == 33 and raw.dR_list_pop(l) == 44 and raw.dR_list_pop(l) is None
    assert raw.dR_list_removeFirstOcc(l, 5) == 0
    raw.dR_list_cleanup(l)


def test_matmul_helpers():
    raw = ctypes.CDLL(dr.LIB_PATH)
    fp = ctypes.POINTER(ctypes.c_float)
    rng = np.random.default_rng(1)
    a, b = rng.standard_normal((4, 3)).astype(np.float32), rng.standard_normal((3, 5)).astype(np.float32)
    out = np.zeros((4, 5), np.float32)
    assert raw.dR_matmul(a.ctypes.data_as(fp), 4, 3, b.ctypes.data_as(fp), 3, 5, out.ctypes.data_as(fp)) == 1
    assert np.allclose(out, a @ b, atol=1e-6)
    bt = rng.standard_normal((6, 3)).astype(np.float32)
    out2 = np.zeros((4, 6), np.float32)
    assert raw.dR_matmulT(a.ctypes.data_as(fp), 4, 3, bt.ctypes.data_as(fp), 6, 3, out2.ctypes.data_as(fp)) == 1
    assert np.allclose(out2, a @ bt.T, atol=1e-6)
    assert raw.dR_matmul(a.ctypes.data_as(fp), 4, 3, bt.ctypes.data_as(fp), 6, 3, out2.ctypes.data_as(fp)) == 0


def _kernel_line(node):
    """The 'Kernel: ...' line of a conv node's printLayer text (which algorithm schedule() settled on)."""
    fn = ctypes.CFUNCTYPE(ctypes.c_void_p, ctypes.c_void_p)(dr.node_struct(node).printLayer)
    text = ctypes.string_at(fn(node.ptr)).decode()
    return [l for l in text.splitlines() if "Kernel:" in l][0]


def test_layers_beyond_the_packed_argument_fields_take_the_general_kernel(lib):
    """The matrix-core convolution kernels carry W, H, I and O in 16-bit fields: a 3x3 layer with a dimension above
    65535 is scheduled onto the general direct kernel, and a first layer of that size is not fused with its pool."""
    rng = np.random.default_rng(0)
    for width, expect in ((64, "Winograd"), (70000, "direct")):
        with dr.Environment() as env:
            g = env.create_graph()
            x = dr.feed_node(g, [2, width, 1])                                   # HWC: 2 rows, `width` columns
            c = dr.Conv2d_raw(x, rng.standard_normal((1, 2, 3, 3)), None, (1, 1), "relu")
            p = dr.Pooling(c, "max", [1, 3, 3, 1], [1, 2, 2, 1])
            dr.mark_as_output(p)
            assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
            assert expect in _kernel_line(c), _kernel_line(c)
            assert lib.dR_planBuffers(g.ptr) == 1
            # (the conv is a "first layer": with the stride-1 3x3 filter it is a Winograd node, never the fused
            # first-layer + pool kernel; the wide one, now direct, must not be fused either)
            plan = plan_of(g, [c, p])
            if width > 65535:
                assert plan[0][0] != plan[1][0]                  # the convolution keeps a tensor of its own


@pytest.mark.parametrize("W,H,I,O,k,stride,kernel", [
    (112, 112, 128, 128, 3, 1, "Winograd F(2x2,3x3) split-operand bf16 MFMA"), (14, 14, 16, 64, 3, 1, "Winograd F(2x2,3x3) MFMA"),
    (56, 56, 64, 96, 5, 1, "direct, split-operand bf16 MFMA"), (56, 56, 64, 96, 3, 2, "direct MFMA"), (33, 31, 3, 9, 3, 2, "direct"), (9, 9, 8, 8, 1, 1, "1x1 MFMA GEMM")])
def test_a_layer_says_which_kernel_it_runs(lib, W, H, I, O, k, stride, kernel):
    with dr.Environment() as env:
        g = env.create_graph()
        x = dr.feed_node(g, [H, W, I])
        c = dr.Conv2d_raw(x, np.ones((I, O, k, k), np.float32), None, (stride, stride), "relu")
        dr.mark_as_output(c)
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        assert re.fullmatch(" Kernel: %s \\(variant \\d+\\)" % re.escape(kernel), _kernel_line(c)), _kernel_line(c)


@pytest.mark.parametrize("W,H,I,O,k,stride,pool,taken", [
    (65, 47, 3, 64, 3, 2, 3, True), (64, 48, 2, 33, 3, 2, 3, True), (65, 47, 3, 64, 7, 2, 2, False), (64, 48, 4, 32, 5, 1, 2, False),
    (30, 34, 8, 64, 5, 1, 2, False), (60, 52, 16, 32, 3, 2, 2, False), (65, 47, 3, 64, 7, 2, 3, False), (65, 47, 1, 64, 3, 2, 3, False)])
def test_a_squeeze_layer_rides_with_image_layers_only(lib, W, H, I, O, k, stride, pool, taken):
    """Layer -> pooling -> fire module: the launch of the first two takes the squeeze layer along where it is a 3x3 layer over an image
    with a 3x3/2 pooling, and no other layer that has its pooling in its launch does."""
    w = lambda i, o, side: np.ones((i, o, side, side), np.float32)
    with dr.Environment() as env:
        g = env.create_graph()
        c = dr.Conv2d_raw(dr.feed_node(g, [H, W, I]), w(I, O, k), None, (stride, stride), "relu")
        squeeze = dr.Conv2d_raw(dr.Pooling(c, "max", [1, pool, pool, 1], [1, 2, 2, 1]), w(O, 16, 1), None, (1, 1), "relu")
        one, three = dr.Conv2d_raw(squeeze, w(16, 32, 1), None, (1, 1), "relu"), dr.Conv2d_raw(squeeze, w(16, 32, 3), None, (1, 1), "relu")
        dr.mark_as_output(dr.Concat([one, three], 2))
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1 and lib.dR_planBuffers(g.ptr) == 1
        assert ("in the launch of the layers in front" in _kernel_line(squeeze)) == taken, _kernel_line(squeeze)


@pytest.mark.parametrize("W,S,E,modules,joined", [
    (14, 64, 256, 2, True), (28, 32, 128, 2, True), (56, 16, 512, 2, True), (112, 16, 64, 2, True), (14, 64, 32, 2, True), (112, 32, 128, 6, True), (320, 16, 64, 2, True),
    (56, 64, 1024, 2, False), (80, 32, 1024, 2, False), (28, 64, 1024, 2, False), (56, 64, 512, 2, False), (224, 64, 32, 2, False), (112, 64, 128, 2, False),
    (160, 32, 256, 2, False), (56, 64, 1024, 6, False), (80, 32, 1024, 6, False), (320, 64, 32, 6, False)])
def test_fire_modules_ride_along_where_that_is_faster(lib, W, S, E, modules, joined):
    """Runs of alike modules on square maps, on the side that measures at least 5 % faster."""
    w = lambda i, o, k: np.zeros((i, o, k, k), np.float32)
    with dr.Environment() as env:
        g = env.create_graph()
        x, channels, squeezes = dr.feed_node(g, [W, W, 32]), 32, []
        for _ in range(modules):
            squeezes.append(dr.Conv2d_raw(x, w(channels, S, 1), None, (1, 1), "relu"))
            x = dr.Concat([dr.Conv2d_raw(squeezes[-1], w(S, E, 1), None, (1, 1), "relu"), dr.Conv2d_raw(squeezes[-1], w(S, E, 3), None, (1, 1), "relu")], 2)
            channels = 2 * E
        dr.mark_as_output(dr.Conv2d_raw(x, w(channels, 8, 1), None, (1, 1), "relu"))
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1 and lib.dR_planBuffers(g.ptr) == 1
        assert ["in the launch of the layers in front" in _kernel_line(s) for s in squeezes[1:]] == [joined] * (modules - 1)


@pytest.mark.parametrize("W,H,I,O,stride,variant", [(40, 40, 24, 16, 1, 0), (86, 94, 64, 32, 2, 0), (32, 32, 24, 16, 1, 0x24), (64, 64, 64, 16, 2, 0x28)])
def test_averaged_layers_have_at_most_64_tiles(lib, monkeypatch, W, H, I, O, stride, variant):
    """A direct 3x3 layer whose tiles of 16 pixels are more than 64 leaves a global average to tiles of 32 (variant 0: by that form's own rule)."""
    monkeypatch.setenv("DR_CONV3X3", "direct")
    w, size = lambda i, o, k: np.ones((i, o, k, k), np.float32), (W // stride, H // stride)
    with dr.Environment() as env:
        g = env.create_graph()
        c = dr.Conv2d_raw(dr.feed_node(g, [H, W, I]), w(I, O, 3), None, (stride, stride), "relu")
        dr.mark_as_output(dr.Softmax(dr.Pooling(c, "average", [1, *size, 1], [1, *size, 1])))
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
        assert int(re.search(r"variant (\d+)", _kernel_line(c))[1]) == lib.drhip_conv3x3_direct_pick_variant(*size, I, O)
        assert lib.dR_planBuffers(g.ptr) == 1
        assert int(re.search(r"variant (\d+)", _kernel_line(c))[1]) == variant


@pytest.mark.parametrize("W,H,I,O,reader,inLaunch", [
    (200, 200, 3, 64, True, True), (300, 300, 3, 64, True, True), (96, 96, 3, 24, True, False), (128, 128, 3, 32, True, False), (96, 96, 3, 24, False, True)])
def test_who_takes_a_pooling_of_three_behind_other_filters(lib, W, H, I, O, reader, inLaunch):
    """7x7/2 layer -> 3x3/2 max pooling (-> 1x1 layer): the first layer stores the pooled tensor where that beats the pooling's alternative, which is the
    1x1 layer taking the maxima on load where there is one (96x96 3->24: in the launch without a reader, on load with it)."""
    w = lambda i, o, k: np.ones((i, o, k, k), np.float32)
    pick = lambda against: lib.drhip_conv_bank_maxpool3s2_pick_variant(W, H, I, O, 7, 7, 2, 2, against) != 0
    assert pick(1 if reader else 0) == inLaunch
    with dr.Environment() as env:
        g = env.create_graph()
        c = dr.Conv2d_raw(dr.feed_node(g, [H, W, I]), w(I, O, 7), None, (2, 2), "relu")
        p = dr.Pooling(c, "max", [1, 3, 3, 1], [1, 2, 2, 1])
        dr.mark_as_output(dr.Conv2d_raw(p, w(O, 16, 1), None, (1, 1), "relu") if reader else p)
        assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1 and lib.dR_planBuffers(g.ptr) == 1
        pixels, pooled = (W // 2) * (H // 2), -(-(W // 2) // 2) * -(-(H // 2) // 2)
        assert plan_of(g, [c])[0][3] == O * (pooled if inLaunch else pixels)        # (floats)


def test_layers_beyond_32_bit_byte_offsets_take_the_general_kernels(lib):
    """Every dimension fits the 16-bit argument fields, but the input holds 2^29 elements or more: the matrix-core
    3x3 kernels and the pooling-on-load 1x1 kernel (32-bit byte offsets) are not scheduled for such a layer."""
    rng = np.random.default_rng(0)
    for width, bank in ((64, True), (65000, False)):
        with dr.Environment() as env:                                         # strided 3x3: direct kernel, with or without its filter bank
            g = env.create_graph()
            x = dr.feed_node(g, [1033, width, 8])
            c = dr.Conv2d_raw(x, rng.standard_normal((8, 2, 3, 3)), None, (2, 2), "relu")
            dr.mark_as_output(c)
            assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
            line = _kernel_line(c)
            assert "direct" in line and (("variant 0" not in line) == bank), line
    class PoolData(ctypes.Structure):                                         # dR_Pooling_Data (include/dR_nodes.h)
        _fields_ = [("ishape", ctypes.c_int * 3), ("shape", ctypes.c_int * 4), ("stride", ctypes.c_int * 4), ("poolingType", ctypes.c_int),
                    ("shaderSrc", ctypes.c_void_p), ("useLMEM", ctypes.c_int), ("drFused", ctypes.c_int)]
    for width, fused in ((64, True), (65000, False)):
        with dr.Environment() as env:                                         # 3x3/2 max pool -> 1x1 conv
            g = env.create_graph()
            x = dr.feed_node(g, [1033, width, 8])
            p = dr.Pooling(x, "max", [1, 3, 3, 1], [1, 2, 2, 1])
            c = dr.Conv2d_raw(p, rng.standard_normal((8, 2, 1, 1)), None, (1, 1), "relu")
            dr.mark_as_output(c)
            assert lib.dR_propagateShapesAndSchedule(g.ptr) == 1
            assert lib.dR_planBuffers(g.ptr) == 1
            pd = ctypes.cast(dr.node_struct(p).layer, ctypes.POINTER(PoolData)).contents
            assert bool(pd.drFused) == fused, (width, pd.drFused)


def test_c_host_program_compiles_against_the_public_headers(lib, tmp_path):
    """tests/c_caller.c: plain C11 against include/deepRACIN.h, with one _Static_assert per field of the structs a
    host program of the reference reaches into (offsets from the reference's own header, tests/golden/
    ref_struct_offsets.h).  Compiling it is the layout check; it links against the library without a GPU."""
    from deepracin_amd import build
    exe = build.build_c_caller(out=str(tmp_path / "c_caller"), verbose=False)
    import subprocess
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 2 and "usage" in r.stderr


def test_pick_variants_are_launchable(lib):
    for (W, H, I, O) in [(224, 224, 3, 64), (224, 224, 64, 64), (56, 56, 256, 256), (14, 14, 512, 512), (55, 55, 16, 64), (1, 1, 1, 1)]:
        v = lib.drhip_conv3x3_winograd_pick_variant(W, H, I, O)
        assert v >= 1
        c = lib.drhip_conv1x1_pick_variant(W * H, I, O)          # waves per tile | 0x100 for 16x16 tiles
        assert (c in (1, 2, 4, 8)) or (c & 0x100 and (c & 0xff) in (1, 2, 4, 8, 16) and c >> 9 == 0)


@pytest.mark.parametrize("K,N", [(1, 1), (64, 10), (65, 1000), (1024, 1000), (8192, 100), (8256, 20), (16384, 60), (30000, 30), (100032, 10), (25088, 4096), (4096, 1000)])
def test_fc_slices_hold_no_more_than_256_rows(lib, K, N):
    """No slice has more than 256 rows unless 256 workgroups, one per CU, have more to share between them (columns go out in panels
    of 64, from 1024 on in 16 and more); up to 8192 rows a matrix of at most 2^20 weights is cut finer, into 32 slices at most."""
    slices, panels = lib.drhip_fc_slices(K, N), -(-N // 64) if N < 1024 else 16
    rows, shared = -(-K // slices), 64 * -(-K // (64 * -(-256 // panels)))
    assert rows <= max(256, shared)
    if K * N <= 1 << 20 and K <= 8192:
        assert slices <= 32 and rows <= max(64 * -(-K // 2048), shared)


def test_bench_refuses_more_than_one_gpu():
    """bench.py measures one GPU: any other --gpus value ends with a message, not with a number."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert r.returncode != 0
    assert "exactly one GPU" in (r.stdout + r.stderr)
    assert not r.stdout.strip().startswith("{")


@pytest.fixture(scope="module")
def split_kernel_code(tmp_path_factory):
    """{kernel: lines} of the assembly that the build's compiler and flags make of k_winograd_split.hip."""
    import subprocess
    from deepracin_amd import build
    out = str(tmp_path_factory.mktemp("asm") / "split.s")
    src = os.path.join(build.CSRC, "device", "k_winograd_split.hip")
    subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE + ["--cuda-device-only", "-S", src, "-o", out], check=True, capture_output=True)
    kernels, name = {}, None
    for line in open(out):
        if line.startswith("_ZN5drhip25winograd_f23_split_kernel") and line.split(";")[0].strip().endswith(":"):
            name = line.split(":")[0]
            kernels[name] = []
        elif name and line.strip().startswith(".section"):
            name = None
        elif name:
            kernels[name].append(line.strip())
    assert len(kernels) == 6
    return kernels


def test_split_kernel_leaves_m0_as_the_compiler_has_it(split_kernel_code):
    """The fetches to LDS take their destination from M0, which no inline assembly can declare as overwritten: each puts it back."""
    for name, lines in split_kernel_code.items():
        n = 0
        for k, line in enumerate(lines):
            if line.startswith("buffer_load") and line.endswith(" lds"):
                n += 1
                saved = lines[k - 3].split()[1].rstrip(",")
                assert lines[k - 3].split()[2] == "m0" and lines[k - 2].startswith("s_mov_b32 m0, ") and lines[k + 1] == "s_mov_b32 m0, " + saved, (name, lines[k - 4:k + 2])
        assert n >= 15, (name, n)


def test_split_kernel_waits_for_its_samples(split_kernel_code):
    """The split-operand Winograd kernel waits for its fetches to LDS by hand: a wait for all but the last n memory instructions
    covers a fetch only if at least n were issued behind it.  Counted in the assembly: behind the first step's fetch in
    front of the loop, and behind a step's fetch once round the loop to the wait of the next step."""
    for name, lines in split_kernel_code.items():
        fetches = 6 if "ILi2ELi24E" in name else 5      # of a wave per step
        blocks, inline = [[]], False                    # of code; F fetch, M other memory instruction, (n) a wait by hand
        for line in lines:
            inline = (inline or line == ";;#ASMSTART") and line != ";;#ASMEND"
            if line.startswith(".LBB"):
                blocks.append([line.split(":")[0]])
            elif re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", line):
                blocks[-1].append("F" if line.endswith(" lds") else "M")
            elif inline and line.startswith("s_waitcnt vmcnt"):
                blocks[-1].append(int(re.search(r"\((\d+)\)", line).group(1)))
        memory = lambda events: sum(e in ("F", "M") for e in events)
        fetching = [b for b in blocks if "F" in b]      # straight on through these: the blocks between them only choose addresses
        body, front = fetching[-1][1:], [e for b in fetching[:-1] for e in b if e in ("F", "M")]
        assert body.count("F") == fetches and front.count("F") == 2 * fetches, name
        waits = [k for k, e in enumerate(body) if isinstance(e, int)]
        last = max(k for k, e in enumerate(body) if e == "F")
        assert len(waits) == 1 and last < waits[0], name
        assert memory(body[last + 1:]) + memory(body[:waits[0]]) >= body[waits[0]], name
        first = [k for k, e in enumerate(front) if e == "F"][fetches - 1]
        wait = next(e for b in blocks for e in b if isinstance(e, int))
        assert memory(front[first + 1:]) >= wait > 0, (name, front, wait)


@pytest.fixture(scope="module")
def pair_kernel_code(tmp_path_factory):
    """{kernel: lines} of the two-part kernel's assembly."""
    import subprocess
    from deepracin_amd import build
    out = str(tmp_path_factory.mktemp("asm") / "pair.s")
    src = os.path.join(build.CSRC, "device", "k_winograd_split.hip")
    subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE + ["--cuda-device-only", "-S", src, "-o", out], check=True, capture_output=True)
    kernels, name = {}, None
    for line in open(out):
        if line.startswith("_ZN5drhip24winograd_f23_pair_kernel") and line.split(";")[0].strip().endswith(":"):
            name = line.split(":")[0]
            kernels[name] = []
        elif name and line.strip().startswith(".section"):
            name = None
        elif line.strip().startswith(".amdhsa_kernel"):
            described = line.split()[1]
        elif ".amdhsa_private_segment_fixed_size" in line and described in kernels:
            kernels[described].append(line.strip())
        elif name:
            kernels[name].append(line.strip())
    assert len(kernels) == 5                # (narrow maps always take turns)
    return kernels


def test_pair_kernel_keeps_nothing_in_scratch(pair_kernel_code):
    """A kernel that has scratch starts about 1 us later."""
    for name, lines in pair_kernel_code.items():
        assert not [l for l in lines if l.startswith("scratch_")], name
        assert ".amdhsa_private_segment_fixed_size 0" in lines, name


def test_pair_kernel_waits_for_its_samples_and_leaves_m0(pair_kernel_code):
    """As for the three-part kernel: fetches to LDS put M0 back, and a wait for all but the last n memory instructions has at least n behind the fetch
    that it is for: the first step's in front of the loop, and a step's once round the loop."""
    for name, lines in pair_kernel_code.items():
        fetches = 6 if "ILi2ELi24E" in name else 5
        blocks, inline = [[]], False
        for k, line in enumerate(lines):
            inline = (inline or line == ";;#ASMSTART") and line != ";;#ASMEND"
            if line.startswith(".LBB"):
                blocks.append([])
            elif re.match(r"(buffer|global|flat|scratch)_(load|store|atomic)", line):
                if line.endswith(" lds"):
                    saved = lines[k - 3].split()[1].rstrip(",")
                    assert lines[k - 3].split()[2] == "m0" and lines[k - 2].startswith("s_mov_b32 m0, ") and lines[k + 1] == "s_mov_b32 m0, " + saved, name
                blocks[-1].append("F" if line.startswith("buffer_load_dwordx4") and line.endswith(" lds") else "M")
            elif inline and line.startswith("s_waitcnt vmcnt"):
                blocks[-1].append(int(re.search(r"\((\d+)\)", line).group(1)))
        memory = lambda events: sum(e in ("F", "M") for e in events)
        fetching = [b for b in blocks if "F" in b]
        body, front = fetching[-1], [e for b in fetching[:-1] for e in b if e in ("F", "M")]
        assert body.count("F") == fetches and front.count("F") == 2 * fetches, name
        waits = [k for k, e in enumerate(body) if isinstance(e, int)]
        last = max(k for k, e in enumerate(body) if e == "F")
        assert len(waits) == 1 and memory(body[last + 1:]) + memory(body[:waits[0]]) >= body[waits[0]] > 0, name
        places = [k for k, e in enumerate(front) if e == "F"]
        wait = next(e for b in blocks for e in b if isinstance(e, int))
        assert memory(front[places[fetches - 1] + 1:]) >= wait > 0, (name, front, wait)
        # and the second step's, which the loop's first wait is for
        assert memory(front[places[-1] + 1:]) + memory(body[:waits[0]]) >= body[waits[0]], name


@pytest.mark.parametrize("what,fits", [("random", True), ("zero channel", True), ("tiny filter", False), ("zero filter", False), ("nan", False), ("inf", False),
                                       ("small", True), ("too small", False), ("too large", False)])
def test_filters_that_two_parts_can_hold(lib, what, fits):
    """Finite, none of an output channel's filters far below its largest; an output channel without any is exact."""
    w = np.random.default_rng(1).standard_normal((70, 33, 9)).astype(np.float32)
    if what == "zero channel":
        w[:, 5] = 0
    elif what in ("tiny filter", "zero filter", "nan", "inf"):
        w[69, 32] = {"tiny filter": 2.0 ** -14, "zero filter": 0.0, "nan": w[69, 32], "inf": w[69, 32]}[what]
        if what in ("nan", "inf"):
            w[69, 32, 8] = np.nan if what == "nan" else np.inf
    else:
        w *= np.float32({"small": 2.0 ** -90, "too small": 2.0 ** -110, "too large": 2.0 ** 110}.get(what, 1.0))
    p = np.ascontiguousarray(w).ctypes.data_as(ctypes.c_void_p)
    assert lib.drhip_winograd_pair_fits(p, 70, 33, 9) == fits
    one = np.ascontiguousarray(w[:, :, 8])
    if what == "random":
        one[:] = np.abs(one) + 0.01
    assert what not in ("random", "nan", "inf") or lib.drhip_winograd_pair_fits(one.ctypes.data_as(ctypes.c_void_p), 70, 33, 1) == fits


def test_outputs_of_an_unprepared_graph_are_none_at_all(lib):
    """download_outputs in front of prepare returns an empty list, as the reference's wrapper does: dR_getOutputBuffers counts none."""
    with dr.Environment() as env:
        g = env.create_graph()
        x = dr.feed_node(g, [8, 8, 2])
        dr.mark_as_output(dr.Pooling(x, "max", [1, 2, 2, 1], [1, 2, 2, 1]))
        assert dr.download_outputs(g) == [] and dr.download_outputs(g, squeeze=False) == []


def test_split_winograd_variants_are_those_that_the_rule_can_pick(lib):
    """One set of waves joins halves, two join up to four pieces; other numbers of pieces are refused."""
    joins = lambda base, n: lib.drhip_conv3x3_winograd_split_workspace_floats(160, 120, 256, 256, base | n << 12 | n << 16) > 0
    assert [n for n in range(16) if joins(0x100, n)] == [2] and [n for n in range(16) if joins(0x101, n)] == [2, 3, 4]


def test_pair_winograd_joins_up_to_four_pieces(lib):
    joins = lambda base, n: lib.drhip_conv3x3_winograd_split_workspace_floats(160, 120, 256, 256, base | n << 12 | n << 16) > 0
    assert [n for n in range(16) if joins(0x300, n)] == [n for n in range(16) if joins(0x301, n)] == [2, 3, 4]


def test_split_winograd_workspace_holds_pieces_only(lib):
    """160x120 256->256 is 600 panels, 75 per XCD: slots of 32 KiB for the pieces, none for panels that stay whole."""
    floats = lambda v: lib.drhip_conv3x3_winograd_split_workspace_floats(160, 120, 256, 256, v)
    assert lib.drhip_conv3x3_winograd_split_pick_variant(160, 120, 256, 256) == 0x100 | 64 << 20 | 1 << 12 | 2 << 16
    for nA, sA, sB, slots in ((64, 1, 2, 22), (75, 1, 2, 1), (75, 2, 1, 150), (10, 2, 1, 20), (10, 2, 2, 150), (0, 1, 2, 150), (0, 1, 1, 0)):
        assert floats(0x100 | nA << 20 | sA << 12 | sB << 16) == slots * 8 * 8192, (nA, sA, sB)


@pytest.mark.parametrize("W,H,I,O,variant", [
    (56, 56, 256, 256, 0x2c01), (56, 56, 128, 256, 0x401),          # 200 panels: helpers, or too few stages for them
    (48, 48, 128, 256, 0x2c01), (46, 46, 64, 256, 0x401),           # 144, 136 panels: no halves of them
    (34, 32, 256, 256, 0xc11), (34, 32, 128, 256, 0xc11), (34, 32, 64, 256, 0x101),     # 72 panels: halves, or the 16-tile form
    (36, 36, 256, 96, 0xc21), (14, 14, 512, 512, 0x831), (28, 28, 512, 512, 0xc11), (56, 56, 64, 64, 0x501)])
def test_winograd_variant_by_panels_and_stages(lib, W, H, I, O, variant):
    assert lib.drhip_conv3x3_winograd_pick_variant(W, H, I, O) == variant


@pytest.mark.parametrize("W,H,I,O,variant,donated,finer", [
    (131, 35, 384, 16, 0xc21, 0, 8), (44, 53, 479, 64, 0xc21, 0, 8), (8, 32, 285, 514, 0xc21, 0, 8),    # quarters where eighths would need a second round
    (349, 5, 571, 5, 0xc31, 0, 16), (7, 268, 250, 3, 0xc31, 0, 16),                                     # eighths, sixteenths
    (45, 79, 537, 138, 0x22, 0, 4), (188, 30, 627, 93, 0x22, 0, 4),                                     # 129 to 159 panels, long sums: quarters as they were
    (188, 30, 500, 93, 0x2c01, 20, 2), (45, 386, 600, 1, 0x2c01, 24, 2), (46, 46, 64, 256, 0x401, 0, 2)])   # helpers or two wave sets where there were halves
def test_sums_of_a_cut_are_as_short_as_the_finer_one_s(lib, W, H, I, O, variant, donated, finer):
    """Stages of eight channels that one accumulator adds up: where a cut is not made because its pieces would not fit one round, or helpers
    take its place, no more than with that cut."""
    v, stages, div = lib.drhip_conv3x3_winograd_pick_variant(W, H, I, O), -(-I // 8), lambda a, b: -(-a // b)
    assert v == variant
    assert div(div(stages - donated, 1 << (v >> 4 & 15)), 2 if v & 0x400 else 1) <= div(stages, finer)


@pytest.mark.parametrize("W,H,I,O,pieces", [
    (48, 48, 256, 256, 3), (48, 48, 512, 256, 3), (40, 30, 512, 512, 3),        # which helpers, or joined halves, would do as fast
    (42, 143, 504, 80, 2), (62, 57, 497, 134, 2), (56, 41, 783, 114, 4),        # with an odd number of chunks, too
    (172, 9, 1020, 154, 4),                                                     # faster than joined halves, not than quarters in two launches
    (56, 56, 256, 256, 0), (28, 28, 512, 512, 0), (34, 32, 256, 256, 0)])       # no faster than halves and whole panels
def test_layers_stay_in_pieces_for_their_exactness(lib, W, H, I, O, pieces):
    """Split-operand pieces are more exact than the joined halves and helpers of the fp32 kernel, and are measured against its other forms."""
    assert lib.drhip_conv3x3_winograd_split_pick_variant(W, H, I, O) == (0x101 | pieces << 12 | pieces << 16 if pieces else 0)


@pytest.mark.parametrize("W,H,I,O,variant", [
    (56, 56, 256, 256, 0x22301), (28, 28, 512, 512, 0x44301), (62, 41, 376, 106, 0x44301), (47, 61, 192, 192, 0x33301),     # pieces where they are the faster ones
    (21, 148, 232, 79, 0), (12, 359, 236, 48, 0), (12, 75, 304, 304, 0), (22, 107, 380, 281, 0x22301), (25, 32, 434, 296, 0x44301), (23, 46, 453, 472, 0x33301),      # narrow maps
    (56, 56, 128, 256, 0), (28, 28, 256, 512, 0), (84, 68, 224, 64, 0), (14, 14, 512, 512, 0), (45, 60, 480, 64, 0),
    (112, 112, 64, 128, 0x300), (112, 112, 127, 128, 0x301), (112, 112, 112, 128, 0x300), (112, 112, 63, 128, 0),           # one round that fills more than half of the CUs
    (73, 28, 128, 476, 0), (34, 159, 69, 141, 0), (40, 40, 146, 294, 0), (39, 152, 198, 68, 0),                             # one round or helpers of the fp32 kernel
    (73, 28, 400, 476, 0x33300), (80, 60, 304, 256, 0x33300), (80, 60, 288, 256, 0x301), (88, 64, 304, 256, 0x301),         # thirds, all at once
    (75, 53, 256, 512, 0x1841300), (71, 119, 256, 256, 0x1941300), (62, 71, 512, 512, 0x1121300), (80, 60, 512, 512, 0x1321300), (113, 44, 384, 512, 0x1421300),    # half in halves, for short sums
    (80, 60, 500, 500, 0x2041301), (114, 91, 384, 256, 0x2031301), (80, 52, 192, 512, 0x1c41300), (144, 120, 256, 256, 0x4041300), (160, 120, 256, 256, 0x4021300), (128, 96, 128, 256, 0x2021300), (122, 93, 256, 256, 0x1c21300),   # whole panels beside halves
    (124, 101, 384, 200, 0x300), (108, 90, 112, 256, 0x300), (112, 128, 112, 128, 0x300),
    (64, 64, 64, 256, 0), (64, 66, 64, 256, 0x300), (28, 30, 64, 1024, 0)])                                                # 128 panels, 132, and none of them on maps that narrow
def test_winograd_pair_variant_by_panels_and_chunks(lib, W, H, I, O, variant):
    assert lib.drhip_conv3x3_winograd_pair_pick_variant(W, H, I, O) == variant


@pytest.mark.parametrize("pixels,channels", [(1, 1), (1, 5), (63, 7), (64, 2), (65, 3), (1000, 64)])
def test_interleaved_to_planes(lib, pixels, channels):
    a = np.random.default_rng(0).standard_normal((pixels, channels)).astype(np.float32)
    out = np.full((channels, pixels), np.nan, np.float32)
    lib.drhip_interleaved_to_planes(out.ctypes.data, a.ctypes.data, pixels, channels)
    assert np.array_equal(out, a.T)


@pytest.mark.parametrize("source", ["k_winograd.hip", "k_winograd_split.hip"])
def test_wide_stores_keep_their_data(tmp_path, source):
    """A buffer store of 16 bytes with a scalar offset has been seen on gfx950 to take what the next vector instruction writes to its data.  The
    compiler knows of no such hazard: in the assembly of the kernels that join partial tiles no such store has one, nor may one of the two
    instructions behind it write there."""
    import subprocess
    from deepracin_amd import build
    out = str(tmp_path / "k.s")
    subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE + ["--cuda-device-only", "-S", os.path.join(build.CSRC, "device", source), "-o", out],
                   check=True, capture_output=True)
    code = [l.split(";")[0].strip() for l in open(out)]
    code = [l for l in code if l and l[0] != "." and not l.endswith(":")]
    stores = 0
    for k, line in enumerate(code):
        m = re.match(r"buffer_store_dwordx[34] v\[(\d+):(\d+)\], (?:v\d+|off), s\[\d+:\d+\], (\S+)", line)
        if not m:
            continue
        stores += 1
        assert not m[3].startswith("s"), line
        for after in code[k + 1:k + 3] if m[3].startswith("s") else []:
            w = re.match(r"v_(?!cmp)\S+ v(?:(\d+)|\[(\d+):(\d+)\])", after)
            if w:
                lo, hi = (int(w[1]), int(w[1])) if w[1] else (int(w[2]), int(w[3]))
                assert hi < int(m[1]) or lo > int(m[2]), (line, after)
    assert stores


def test_pixel_loads_end_with_the_tensor(tmp_path):
    """The 1x1 kernel in front of a global average takes zeros behind the last pixel from the range check of its input's resource,
    which need not see scalar offsets: in the assembly only the filters' resource is read at one, and the input's is another."""
    import subprocess
    from deepracin_amd import build
    out = str(tmp_path / "k.s")
    subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE + ["--cuda-device-only", "-S", os.path.join(build.CSRC, "device", "k_conv1x1.hip"), "-o", out],
                   check=True, capture_output=True)
    kernels, loads = 0, None
    for line in open(out):
        if line.startswith("_ZN5drhip29conv1x1_pixels_poolsum_kernel") and line.split(";")[0].strip().endswith(":"):
            kernels, loads = kernels + 1, []
        elif loads is not None and line.strip().startswith("buffer_load_dwordx4"):
            loads.append(re.match(r"\s+buffer_load_dwordx4 v\[\d+:\d+\], v\d+, (s\[\d+:\d+\]), (\S+) offen", line).groups())
        elif loads and "s_endpgm" in line:
            scalar = {resource for resource, offset in loads if offset != "0"}
            assert len(scalar) == 1 and loads[0][0] not in scalar and sum(r == loads[0][0] for r, _ in loads) == 5, loads
            loads = None
    assert kernels == 2


@pytest.mark.parametrize("source,kernels", [("k_conv_direct.hip", 2), ("k_winograd.hip", 6)])
def test_filter_loads_end_with_the_bank(tmp_path, source, kernels):
    """Filter banks of the fp32 3x3 kernels are padded to 32 output channels, and a panel may be wider: the blocks of 32 channels that the bank
    lacks read zeros by the range check, which need not see the scalar offset.  So such a block has a vector offset of its
    own: with a scalar one no load goes 1024 bytes (a block) on from another's place by its immediate offset."""
    import subprocess
    from deepracin_amd import build
    out = str(tmp_path / "k.s")
    subprocess.run([build.HIPCC] + build.COMMON + build.DEVICE + ["--cuda-device-only", "-S", os.path.join(build.CSRC, "device", source), "-o", out],
                   check=True, capture_output=True)
    name, places = None, {}
    for line in open(out):
        if re.match(r"_ZN5drhip\S+:", line):
            name = line.split(":")[0]
        m = re.match(r"\s+buffer_load_dwordx4 v\[\d+:\d+\], (v\d+), s\[\d+:\d+\], s\d+ offen(?: offset:(\d+))?", line)
        if m:
            places.setdefault(name, set()).add(m[1])
            assert int(m[2] or 0) < 1024, (name, line)
    wide = [n for n in places if re.search(r"direct_mfma_kernelILi2|f23_mfma_kernelILi[24]|f23_mfma16_kernelILi4", n)]
    assert len(wide) == kernels and all(len(places[n]) >= 2 for n in wide), (wide, places)


def test_direct_variant_of_small_maps():
    """Which direct 3x3 layers get tiles of 16 pixels: those that make no more workgroups than CUs (256) with 16 or 32 channels each."""
    pick = dr.load_library().drhip_conv3x3_direct_pick_variant
    assert [pick(14, 14, 128, 192), pick(28, 28, 96, 128), pick(64, 64, 64, 16), pick(64, 62, 64, 17), pick(14, 14, 32, 16)] == [0x28, 0x38, 0x28, 0x38, 0x24]
    assert pick(62, 64, 64, 33) == 8 and pick(28, 28, 128, 288) == 8 and pick(56, 56, 256, 256) & 0x20 == 0
