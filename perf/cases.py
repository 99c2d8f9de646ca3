"""Timed workloads of the CNN layer path: what programs use this library for, over the range they use it in.

A case is one graph and one way of calling it:

  call "image"   a serving loop through the Python front-end: a new HWC image from host memory, one forward pass, every
                 output back in host memory (feed_data + apply).  What one image costs its caller.
  call "pass"    dR_apply alone with the input resident, on the caller's stream: passes enqueued one behind the other,
                 outputs left on the device.  What the network itself costs.

Graphs: the five benchmark configurations (a single 3x3 layer, a fire module, VGG16's conv3 block, SqueezeNet v1.1,
VGG16), the stored SqueezeNet model with its in-graph mean subtraction, VGG16's convolutions over a photograph, a
classifier of thumbnails, and a trunk of strided and large filters.  Weights are He-normal, biases N(0, 0.01), images
uniform; all of it follows from the seed alone.
"""
import math

import torch

import deepracin_amd as dr

STORED_MODEL = "tests/golden/squeezenet_whole"


def listed():
    return [
        # A classifier of thumbnails: eight launches of next to no work, so what counts is the cost of a call.
        {"name": "small_image", "net": "small", "call": "image", "w": 28, "h": 28, "c": 1, "f1": 16, "f2": 32, "hidden": 128, "classes": 10},
        # Configuration 1: one 3x3 layer with bias and ReLU.
        {"name": "conv3x3_pass", "net": "conv3x3", "call": "pass", "w": 56, "h": 56, "c": 64, "o": 64},
        # Configuration 2: one fire module.
        {"name": "fire_pass", "net": "fire", "call": "pass", "w": 55, "h": 55, "c": 128, "squeeze": 16, "expand": 64},
        # Configuration 3: three 3x3 layers and a pooling.
        {"name": "conv3_block_pass", "net": "conv3_block", "call": "pass", "w": 56, "h": 56, "c": 128, "o": 256},
        # Everything that is not 3x3/1 or 1x1: a 7x7/2 stem, a 5x5 layer, strided 3x3 layers, a global average.
        {"name": "strided_pass", "net": "strided", "call": "pass", "w": 224, "h": 224, "c": 3, "base": 64, "classes": 1000},
        # Configuration 4, served image by image and as bare passes.
        {"name": "squeezenet_image", "net": "squeezenet", "call": "image", "w": 224, "h": 224, "normalise": False, "classes": 1000},
        {"name": "squeezenet_pass", "net": "squeezenet", "call": "pass", "w": 224, "h": 224, "normalise": False, "classes": 1000},
        # A photograph of odd sides, normalised inside the graph.
        {"name": "squeezenet_photo_image", "net": "squeezenet", "call": "image", "w": 451, "h": 299, "normalise": True, "classes": 365},
        # The stored model: mean subtraction by Slice, ElemWise1Op and Concat nodes, stride 1 and pooling instead of stride 2.
        {"name": "stored_squeezenet_image", "net": "stored", "call": "image", "w": 224, "h": 224},
        # Configuration 5, served image by image and as bare passes.
        {"name": "vgg16_image", "net": "vgg16", "call": "image", "w": 224, "h": 224, "width": 4096, "classes": 1000},
        {"name": "vgg16_pass", "net": "vgg16", "call": "pass", "w": 224, "h": 224, "width": 4096, "classes": 1000},
        # Features of a photograph: VGG16's thirteen 3x3 layers and five poolings, 640 x 480.
        {"name": "vgg_trunk_pass", "net": "vgg_trunk", "call": "pass", "w": 640, "h": 480},
    ]


def draw(rng):
    """One more case of the same ranges, no more expensive than the largest listed one."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    net = rng.choice(["small", "conv3x3", "fire", "conv3_block", "strided", "squeezenet", "squeezenet", "vgg16", "vgg_trunk"])
    call = rng.choice(["image", "pass"]) if net in ("small", "squeezenet", "vgg16") else "pass"
    most = {"conv3x3": 1e10, "conv3_block": 4e10}.get(net, work(listed()[-1])["flops"])
    while True:
        case = {"net": net, "call": call}
        if net == "small":
            case.update(w=log_int(20, 64), h=log_int(20, 64), c=rng.randint(1, 4), f1=log_int(6, 32), f2=log_int(8, 64), hidden=log_int(32, 512), classes=log_int(2, 100))
        elif net == "conv3x3":
            case.update(w=log_int(7, 224), h=log_int(7, 224), c=log_int(3, 512), o=log_int(8, 512))
        elif net == "fire":
            case.update(w=log_int(13, 112), h=log_int(13, 112), c=log_int(32, 512), squeeze=log_int(8, 64), expand=log_int(32, 256))
        elif net == "conv3_block":
            case.update(w=log_int(14, 112), h=log_int(14, 112), c=log_int(32, 256), o=log_int(64, 512))
        elif net == "strided":
            case.update(w=rng.randint(96, 384), h=rng.randint(96, 384), c=rng.randint(1, 4), base=log_int(24, 96), classes=log_int(10, 1000))
        elif net == "squeezenet":
            case.update(w=log_int(64, 512), h=log_int(64, 512), normalise=rng.random() < 0.5, classes=log_int(10, 1000))
        elif net == "vgg16":
            case.update(w=log_int(64, 288), h=log_int(64, 288), width=log_int(512, 4096), classes=log_int(10, 1000))
        else:
            case.update(w=log_int(96, 640), h=log_int(96, 640))
        w = work(case)
        if w["flops"] <= most and w["bytes"] <= 6e8:
            return case


class _Plan:
    """A graph as a list of nodes, with shapes (W, H, C) by the library's rules and the work of a pass."""

    def __init__(self, w, h, c):
        self.nodes, self.shapes, self.outputs = [("feed",)], [(w, h, c)], []
        self.weights = self.flops = 0

    def _add(self, node, shape):
        self.nodes.append(node)
        self.shapes.append(shape)
        return len(self.nodes) - 1

    def conv(self, src, k, o, stride=1):
        w, h, c = self.shapes[src]
        self.weights += k * k * c * o + o
        self.flops += 2 * k * k * c * o * (w // stride) * (h // stride)
        return self._add(("conv", src, k, c, o, stride), (w // stride, h // stride, o))

    def fc(self, src, n, relu):
        w, h, c = self.shapes[src]
        self.weights += w * h * c * n + n
        self.flops += 2 * w * h * c * n
        return self._add(("fc", src, w * h * c, n, relu), (n, 1, 1))

    def pool(self, src, kind, kw, kh, sw, sh):
        w, h, c = self.shapes[src]
        return self._add(("pool", src, kind, kw, kh, sw, sh), (-(-w // sw), -(-h // sh), c))

    def max_pool(self, src, k, s):
        return self.pool(src, "max", k, k, s, s)

    def global_average(self, src):
        w, h, _ = self.shapes[src]
        return self.pool(src, "average", w, h, w, h)

    def softmax(self, src):
        return self._add(("softmax", src), self.shapes[src])

    def norm(self, src):
        return self._add(("norm", src), self.shapes[src])

    def fire(self, src, squeeze, expand):
        s = self.conv(src, 1, squeeze)
        one, three = self.conv(s, 1, expand), self.conv(s, 3, expand)
        w, h, _ = self.shapes[one]
        return self._add(("concat", one, three), (w, h, 2 * expand))


def _plan(case):
    net = case["net"]
    p = _Plan(case["w"], case["h"], case.get("c", 3))
    x = 0
    if net == "small":
        x = p.max_pool(p.conv(x, 5, case["f1"]), 2, 2)
        x = p.max_pool(p.conv(x, 5, case["f2"]), 2, 2)
        logits = p.fc(p.fc(x, case["hidden"], True), case["classes"], False)
        p.outputs = [p.softmax(logits), logits]
    elif net == "conv3x3":
        p.outputs = [p.conv(x, 3, case["o"])]
    elif net == "fire":
        p.outputs = [p.fire(x, case["squeeze"], case["expand"])]
    elif net == "conv3_block":
        for _ in range(3):
            x = p.conv(x, 3, case["o"])
        p.outputs = [p.max_pool(x, 2, 2)]
    elif net == "strided":
        base = case["base"]
        x = p.max_pool(p.conv(x, 7, base, 2), 3, 2)
        x = p.conv(x, 5, base + base // 2)
        x = p.conv(p.conv(x, 3, 2 * base, 2), 3, 3 * base, 2)
        x = p.global_average(x)
        logits = p.fc(x, case["classes"], False)
        p.outputs = [p.softmax(logits), logits]
    elif net == "squeezenet":
        if case["normalise"]:
            x = p.norm(x)
        x = p.max_pool(p.conv(x, 3, 64, 2), 3, 2)
        for squeeze, expand in ((16, 64), (16, 64), (0, 0), (32, 128), (32, 128), (0, 0), (48, 192), (48, 192), (64, 256), (64, 256)):
            x = p.fire(x, squeeze, expand) if squeeze else p.max_pool(x, 3, 2)
        x = p.global_average(p.conv(x, 1, case["classes"]))
        p.outputs = [p.softmax(x), x]
    elif net in ("vgg16", "vgg_trunk"):
        for o, layers in ((64, 2), (128, 2), (256, 3), (512, 3), (512, 3)):
            for _ in range(layers):
                x = p.conv(x, 3, o)
            x = p.max_pool(x, 2, 2)
        p.outputs = [x]
        if net == "vgg16":
            logits = p.fc(p.fc(p.fc(x, case["width"], True), case["width"], True), case["classes"], False)
            p.outputs = [p.softmax(logits), logits]
    else:
        raise ValueError("unknown net %r" % net)
    return p


class _Program:
    """A graph and its environment, given back when nobody holds them any more."""

    def __init__(self):
        self.env = dr.Environment()
        self.env.model_path = "/tmp"
        self.graph = self.env.create_graph()

    def __del__(self):
        self.env.close()


class _State:
    """What a program holds between calls: the prepared graph, its feed node, the picture that comes in, and for
    "pass" the output buffers."""

    def __init__(self, prog, feed, image, outputs):
        self.prog, self.graph, self.feed, self.image, self.outputs = prog, prog.graph, feed, image, outputs


class _DeviceArray:
    """A buffer of the graph, as an array that torch can look at; the graph lives as long as the array does."""

    def __init__(self, prog, address, shape):
        self.prog = prog
        self.__cuda_array_interface__ = {"data": (address, False), "shape": shape, "typestr": "<f4", "version": 2}


_stream = None


def _build(graph, plan, gen):
    """The plan's nodes in the graph, weights drawn from `gen` on the GPU, where that takes no time: (feed node, output nodes)."""
    def normal(shape, std):
        return (torch.randn(shape, device="cuda", generator=gen) * std).cpu().numpy()

    nodes = []
    for node, (w, h, c) in zip(plan.nodes, plan.shapes):
        op = node[0]
        if op == "feed":
            nodes.append(dr.feed_node(graph, [h, w, c]))
        elif op == "conv":
            _, src, k, i, o, stride = node
            nodes.append(dr.Conv2d_raw(nodes[src], normal((i, o, k, k), math.sqrt(2 / (k * k * i))), normal((o,), 0.01), (stride, stride), "relu"))
        elif op == "fc":
            _, src, k, n, relu = node
            nodes.append(dr.Fully_Connected(nodes[src], (k, n), "relu" if relu else "linear", normal((k, n), math.sqrt(2 / k)), normal((n,), 0.01)))
        elif op == "pool":
            _, src, kind, kw, kh, sw, sh = node
            nodes.append(dr.Pooling(nodes[src], kind, (1, kw, kh, 1), (1, sw, sh, 1)))
        elif op == "softmax":
            nodes.append(dr.Softmax(nodes[node[1]]))
        elif op == "norm":
            nodes.append(dr.Normalization(nodes[node[1]], "target_mean_dev", 0.0, 1.0))
        else:
            nodes.append(dr.Concat([nodes[i] for i in node[1:]], 2))
    return nodes[0], [nodes[i] for i in plan.outputs]


def prepare(case, seed):
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()       # one stream for all graphs, as a program with one device queue has it
    gen = torch.Generator(device="cuda").manual_seed(seed)
    prog = _Program()
    graph = prog.graph
    graph.lib.dR_setClEnvironment(dr.c_void_p(graph.ptr), None, None, dr.c_void_p(_stream.cuda_stream), None)
    if case["net"] == "stored":
        nodes, feeds = dr.load_graph(graph, STORED_MODEL)
        feed, nodes, channels = feeds[0], nodes[-1:], 3
    else:
        plan = _plan(case)
        feed, nodes = _build(graph, plan, gen)
        channels = plan.shapes[0][2]
    for node in nodes:
        dr.mark_as_output(node)
    dr.prepare(graph)
    image = torch.rand((case["h"], case["w"], channels), device="cuda", generator=gen)
    if case["net"] in ("stored", "squeezenet"):
        image = (image * 256).floor()       # the values of an 8-bit picture
        if case["net"] == "squeezenet" and not case["normalise"]:
            image = (image - image.mean()) / image.std()
    image = image.cpu().numpy()
    if case["call"] == "image":
        return _State(prog, feed, image, None)
    dr.feed_data(feed, image)
    buffers, outputs = (dr.c_void_p * len(nodes))(), []
    graph.lib.dR_getOutputBuffers(graph.ptr, buffers)
    for node, buffer in zip(nodes, buffers):
        w, h, c = node.out_shape
        address = dr.c_void_p.from_address(buffer).value
        outputs.append(torch.as_tensor(_DeviceArray(prog, address, (c, h, w)), device="cuda"))
    return _State(prog, feed, image, outputs)


def run(state):
    if state.outputs is None:
        dr.feed_data(state.feed, state.image)
        return dr.apply(state.graph)
    if not state.graph.lib.dR_apply(state.graph.ptr):
        raise RuntimeError("dR_apply failed")
    return state.outputs


def work(case):
    """Image, weights and outputs once each; multiplications and additions of the convolutions and matrices as
    their definitions have them (a Winograd kernel does with fewer)."""
    if case["net"] == "stored":             # 56x56x64 behind the stem, otherwise SqueezeNet v1.1's layers
        plan = _plan(dict(case, net="squeezenet", normalise=False, classes=1000))
        plan.flops += 3 * (2 * 9 * 3 * 64 * 112 * 112)     # its first layer is evaluated at all 224 x 224 places
        outputs = 1000
    else:
        plan = _plan(case)
        outputs = sum(w * h * c for w, h, c in (plan.shapes[i] for i in plan.outputs))
    w, h, c = plan.shapes[0]
    return {"bytes": 4 * (w * h * c + plan.weights + outputs), "flops": plan.flops}


def tolerance(case):
    """fp32 throughout: 1e-5 for a layer or a few; the networks carry the rounding of 15 to 26 layers into the
    exponentials of their softmax."""
    return {"rel": 2e-5 if case["net"] in ("squeezenet", "vgg16", "stored") else 1e-5}
