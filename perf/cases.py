"""What users of this framework have it do, as cases that can be timed and compared.

A case names a network, the storage of its tensors, the size of a frame and one of three ways of driving it:

  frame     host frame in, host result out, one after the other: setInput -> forward -> getOutput (or getArgMax)
  stream    a run of host frames through a FramePool of one or more instances, results delivered under tickets
  resident  the frame lies in GPU memory already and the result is taken over there by a layer of the application
            (CustomLayerBuilder): forward and finish, eager or from the captured graph

Networks: the style-transfer net (3x3 or 9x9 residual kernels), the style nets and the ResNet-50 of the samples,
ResNet-50, a MobileNetV2-style stack, one 3x3 convolution, and a small segmentation network made of the other layer
types (depthwise and pointwise convolutions, pooling, scaling, concatenation, batch-norm, transposed convolution,
arg-max).  Weights are synthetic and belong to the network, not to the frame: every seed gives other frames.
"""
import functools
import math

import numpy as np
import torch

import fyusenet_amd as fa
from fyusenet_amd import networks, prng, samples

STORAGE = {"f32": fa.STORAGE_F32, "f16": fa.STORAGE_F16}


def listed():
    return [
        # a thumbnail through the small style net of the samples: the smallest call, launches and host latency count
        {"name": "sample3_64x48_frame", "net": "sample3", "storage": "f32", "width": 64, "height": 48, "drive": "frame", "order": "chw"},
        # the style-transfer net on its usual frame, called like a function on host images
        {"name": "style_512x624_frame", "net": "style", "storage": "f32", "width": 512, "height": 624, "drive": "frame", "order": "chw"},
        # the same where the frame is produced and used on the GPU
        {"name": "style_512x624_resident", "net": "style", "storage": "f32", "width": 512, "height": 624, "drive": "resident", "graph": False},
        # a full-HD photograph, interleaved pixels as image files have them
        {"name": "style_1920x1080_frame", "net": "style", "storage": "f32", "width": 1920, "height": 1080, "drive": "frame", "order": "hwc"},
        # the largest network: 9x9 residual layers on a large photograph, 16-bit tensors
        {"name": "style9_1524x1856_resident", "net": "style9", "storage": "f16", "width": 1524, "height": 1856, "drive": "resident", "graph": False},
        # video through the sample's style net with 9x9 outer layers: one network, frames handed over and fetched as they come
        {"name": "sample9_512x624_stream", "net": "sample9", "storage": "f32", "width": 512, "height": 624, "drive": "stream", "order": "hwc", "instances": 1, "frames": 12},
        # one image to classify, answer wanted at once
        {"name": "resnet50_224_frame", "net": "resnet50", "storage": "f32", "width": 224, "height": 224, "drive": "frame", "order": "chw"},
        # the sample's graph with its explicit batch-norm layers, replayed as one captured graph
        {"name": "resnet50sample_resident", "net": "resnet50sample", "storage": "f32", "width": 224, "height": 224, "drive": "resident", "graph": True},
        # classification as a service: several instances side by side on 16-bit tensors
        {"name": "resnet50_224_stream", "net": "resnet50", "storage": "f16", "width": 224, "height": 224, "drive": "stream", "order": "chw", "instances": 4, "frames": 32},
        # the light classifier on one image of a size that nothing divides
        {"name": "mobilenet_211_frame", "net": "mobilenet", "storage": "f16", "width": 211, "height": 211, "drive": "frame", "order": "chw"},
        # a label map for a camera frame
        {"name": "segment_644x484_frame", "net": "segment", "storage": "f16", "width": 644, "height": 484, "drive": "frame", "order": "hwc"},
        # one convolution layer by itself
        {"name": "conv64_256x256_resident", "net": "conv", "storage": "f32", "width": 256, "height": 256, "channels": 64, "drive": "resident", "graph": False},
    ]


# net -> (shortest side drawn, longest side drawn, sides are multiples of)
SIDES = {"sample3": (48, 1024, 4), "sample9": (48, 1024, 4), "style": (48, 1400, 4), "style9": (48, 1400, 4),
         "segment": (64, 1400, 4), "resnet50": (96, 320, 1), "mobilenet": (96, 320, 1), "conv": (20, 400, 1)}


def draw(rng):
    net = rng.choice(sorted(SIDES))
    lo, hi, step = SIDES[net]

    def side():
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step

    width, height = side(), side()
    if net in ("resnet50", "mobilenet"):
        height = width
    c = {"net": net, "storage": "f16" if net == "style9" else rng.choice(["f32", "f16"]), "width": width, "height": height}
    if net == "conv":
        c["channels"] = rng.choice([16, 24, 40, 64, 96, 128, 160])
    c["drive"] = "resident" if net == "conv" else rng.choice(["frame", "resident"] if net in ("style9", "segment") else ["frame", "stream", "resident"])
    if c["drive"] == "resident":
        c["graph"] = rng.random() < 0.5
    else:
        c["order"] = rng.choice(["chw", "hwc"])
    if c["drive"] == "stream":
        c["instances"] = rng.choice([1, 2, 4])
        c["frames"] = max(1, min(rng.randint(3, 16), 12 * 512 * 624 // (width * height)))     # (fewer of the large ones)
    return c


# ---------------------------------------------------------------------------------------------------------------------
# networks
# ---------------------------------------------------------------------------------------------------------------------
class Segment(networks._StreamNet):
    """Encoder and decoder in the light style: label map (argmax_layer) and scores (output_layer) at the frame's size."""
    CLASSES = 21
    input_key = (0, 0)
    config_id = 9

    def __init__(self, storage, width, height):
        super().__init__(storage)
        self.W, self.H = width, height

    def define(self):
        A, W, H = fa.ActType.RELU, self.W, self.H
        self._add(fa.UpDownLayerBuilder(fa.UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(3, H, W, 3).outputPadding(2))
        self.conv(1, "stem", 5, 3, 16, H, W, 0, stride=2, pad_out=1)
        W, H = W // 2, H // 2
        self.conv(2, "dw1", 3, 16, 16, H, W, 1, act=A, groups=16)
        self.conv(3, "pw1", 1, 16, 48, H, W, 2, act=A)
        pool = fa.PoolLayerBuilder(fa.PoolLayerBuilder.POOL_MAX, "pool").number(4).shape(48, H, W, 48).poolSize(2).downsample(2).prefixAct(A).outputPadding(1)
        self._add(pool.deep())
        self._edges.append((3, 4, 0))
        self.conv(5, "mid1", 3, 48, 48, H // 2, W // 2, 4, pad_out=1)
        self.conv(6, "mid2", 3, 48, 48, H // 2, W // 2, 5, act=A, residual=4, res_pad=1, bn_scale=(0.25, 0.75))
        up = fa.ScaleLayerBuilder("up").number(7).shape(48, H // 2, W // 2, 48).scale(2.0).scaleType(fa.ScalingType.LINEAR).prefixAct(A)
        self._add(up.deep())
        self._edges.append((6, 7, 0))
        cat = fa.ConcatLayerBuilder("cat").number(8).deep().input(48, 0).input(48, 0)
        cat.size(W, H)
        cat.outputChannels_ = 96
        self._add(cat)
        self._edges += [(7, 8, 0), (3, 8, 1)]
        bn = fa.GPULayerBuilder("bn").type(fa.LayerType.BATCHNORM).number(9).shape(96, H, W, 96).prefixAct(A).deep()
        seed = self._next_seed()
        self._add(bn, lambda: np.concatenate([prng.uniform(seed, (96,), 0.5, 1.5), prng.normal(seed + 1, (96,), 0.0, 0.1)]))
        self._edges.append((8, 9, 0))
        self.conv(10, "mix", 1, 96, 32, H, W, 9, act=A, pad_out=1)
        t = fa.ConvLayerBuilder(3, "up2").type(fa.LayerType.TRANSCONVOLUTION2D).number(11).shape(32, H, W, 32).deep()
        t.upsample(2).inputPadding(1).prefixAct(A).postfixNorm(fa.NormType.BATCHNORM).crop(1)
        seed2 = self._next_seed()
        self._add(t, lambda: networks.conv_block(seed2, 32, 3, 32, bn=True))
        self._edges.append((10, 11, 0))
        self.conv(12, "scores", 1, 32, self.CLASSES, 2 * H, 2 * W, 11, act=A, bn=False)
        self._add(fa.ArgMaxLayerBuilder("labels").number(13).shape(2, 2 * H, 2 * W, self.CLASSES).deep())
        self._edges.append((12, 13, 0))
        self.output_layer, self.argmax_layer = 12, 13

    def setInput(self, x):
        self.layers[0].setInput(x, 0)


class Taken:
    """The application's layer behind the result of a network: learns where the tensor lies, for the GPU work around it."""

    def setup(self, inputs, output):
        v = inputs[0]
        self.shape = (v.height + 2 * v.padding, v.width + 2 * v.padding, v.channel_pitch)
        self.inside = (slice(v.padding, v.padding + v.height), slice(v.padding, v.padding + v.width), slice(0, v.channels))
        self.type, self.address = "<f2" if v.storage == fa.STORAGE_F16 else "<f4", v.data

    def forward(self, inputs, output, stream, sequence):
        pass


class Memory:
    """A network's tensor as memory for torch; the network lives as long as what is made of it."""

    def __init__(self, net, taken):
        self.net = net
        self.__cuda_array_interface__ = {"shape": taken.shape, "typestr": taken.type, "data": (taken.address, False), "version": 2}


def make(case, taken=None):
    """The case's network, not yet set up; with `taken`, that layer of the application behind its result."""
    kind, st, w, h = case["net"], STORAGE[case["storage"]], case["width"], case["height"]
    base, args, kw = {
        "style": (networks.StyleNet, (st, w, h, 3), {}), "style9": (networks.StyleNet, (st, w, h, 9), {}),
        "resnet50": (networks.ResNet50, (st, w), {}), "mobilenet": (networks.MobileNetV2, (st, w), {}),
        "conv": (networks.SingleConvNet, (st,), {"channels": case.get("channels"), "width": w, "height": h}),
        "segment": (Segment, (st, w, h), {}),
        "sample3": (samples.StyleNetSample, (3, w, h, st), {}), "sample9": (samples.StyleNetSample, (9, w, h, st), {}),
        "resnet50sample": (samples.ResNet50Sample, (st, synthetic_file()) if kind == "resnet50sample" else (), {}),
    }[kind]

    class Network(base):
        def buildLayers(self, factory):
            super().buildLayers(factory)
            if taken is not None:
                c, rows, cols = result_shape(case)
                last = fa.CustomLayerBuilder("taken", lambda builder: taken).number(1000)
                last.shape(c, rows, cols, c).deep().push(factory)

        def connectLayers(self, layers, bm):
            super().connectLayers(layers, bm)
            if taken is not None:
                # (a download layer hands its input on to the host: the tensor is the one in front of it)
                download = int(layers[self.output_layer].builder.type_) == int(fa.LayerType.DOWNLOAD)
                bm.connectLayers(layers[self.output_layer - 1 if download else self.output_layer], layers[1000], 0)

    net = Network(*args, **kw)
    if isinstance(net, networks._StreamNet):
        share_weights(net, kind)
    return net


_weights = {}


def share_weights(net, kind):
    """Networks of one kind take their weights from one stream, generated once."""
    key = (kind, getattr(net, "ch", 0))
    if key not in _weights:
        generate = net.initializeWeights

        def keep(layers):
            generate(layers)
            _weights[key] = (net.weightStream, dict(net.offsets))
        net.initializeWeights = keep
    else:
        net.weightStream, net.offsets = _weights[key]


@functools.lru_cache(maxsize=1)
def synthetic_file():
    class Weights(samples.ResNet50Sample):
        def setup(self):
            return self.synthetic_weights()
    return Weights().setup()


def result_shape(case):
    """(channels, rows, columns) of the result."""
    w, h = case["width"], case["height"]
    if case["net"] == "conv":
        return case["channels"], h, w
    if case["net"] == "segment":
        return Segment.CLASSES, h // 4 * 4, w // 4 * 4
    if case["net"] in ("resnet50", "resnet50sample"):
        return 1000, 1, 1
    if case["net"] == "mobilenet":
        return 320, w // 32, w // 32
    return 3, h, w


# ---------------------------------------------------------------------------------------------------------------------
# preparing and running
# ---------------------------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=1)
def _driven(items):
    """The network (or pool of instances) that a program keeps and hands its frames to."""
    case = dict(items)
    if case["drive"] == "stream":
        order = fa.ORDER_GPU_SHALLOW if case["order"] == "hwc" else fa.ORDER_CHANNELWISE
        small = result_shape(case)[0] <= 4
        return fa.FramePool(lambda: make(case), instances=case["instances"], inOrder=order, outOrder=order if small else fa.ORDER_CHANNELWISE)
    net = make(case)
    net.setup()
    return net


def _frame(case, rng):
    """One frame on the host: image values, normalised ones for the classifiers, signed features for the single layer."""
    w, h = case["width"], case["height"]
    if case["net"] == "conv":
        return rng.random((case["channels"], h, w), dtype=np.float32) * 2 - 1
    shape = (h, w, 3) if case.get("order") == "hwc" else (3, h, w)
    if case["net"] in ("resnet50", "resnet50sample", "mobilenet"):
        return rng.standard_normal(shape, dtype=np.float32)
    return rng.random(shape, dtype=np.float32)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["drive"] == "resident":
        taken = Taken()
        net = make(case, taken)
        net.setup()
        net.useGraph(case["graph"])
        net.setInput(_frame(case, rng))
        return {"case": case, "net": net, "result": torch.as_tensor(Memory(net, taken), device="cuda")[taken.inside]}
    driven = _driven(tuple(sorted((k, v) for k, v in case.items() if k not in ("name", "frames"))))
    state = {"case": case, "net": driven}
    if case["drive"] == "stream":
        state["frames"] = [_frame(case, rng) for _ in range(case["frames"])]
        c, rows, cols = result_shape(case)
        shape = (rows, cols, 4) if case["order"] == "hwc" and c == 3 else (c, rows, cols)
        state["results"] = [np.zeros(shape, np.float32) for _ in state["frames"]]
    else:
        state["frame"] = _frame(case, rng)
    return state


def run(state):
    case, net = state["case"], state["net"]
    if case["drive"] == "resident":
        net.forward()
        net.finish()        # the application's own stream goes on from here
        return state["result"]
    if case["drive"] == "stream":
        ticket = 0
        for frame, result in zip(state["frames"], state["results"]):
            ticket = net.submit(frame, result)
        net.wait(ticket)
        return state["results"]
    order = fa.ORDER_GPU_SHALLOW if case["order"] == "hwc" else fa.ORDER_CHANNELWISE
    layer, port = (1, 0) if case["net"] == "conv" else (0, 0)
    net.layers[layer].setInput(state["frame"], port, order)
    net.forward()
    if case["net"] == "segment":
        labels, best = net.getArgMax(net.argmax_layer)
        return {"labels": labels, "best": best}
    return net.getOutput(net.output_layer, order if result_shape(case)[0] <= 4 else fa.ORDER_CHANNELWISE)


# ---------------------------------------------------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------------------------------------------------
def _layers(case):
    """(kernel, input channels per output, output channels, output positions) of the convolutions and products."""
    w, h, kind = case["width"], case["height"], case["net"]
    full, half, quarter = w * h, (w // 2) * (h // 2), (w // 4) * (h // 4)
    if kind in ("style", "style9"):
        k = 9 if kind == "style9" else 3
        return [(9, 3, 32, full), (3, 32, 64, half), (3, 64, 128, quarter)] + 10 * [(k, 128, 128, quarter)] + \
            [(3, 128, 64, quarter), (3, 64, 32, half), (9, 32, 3, full)]     # (a transposed layer multiplies once per input position)
    if kind in ("sample3", "sample9"):
        k, n = (3, 4) if kind == "sample3" else (9, 10)
        return [(k, 3, 12, full), (3, 12, 20, half), (3, 20, 40, quarter)] + n * [(3, 40, 40, quarter)] + \
            [(3, 40, 20, quarter), (3, 20, 12, half), (k, 12, 3, full)]
    if kind == "conv":
        return [(3, case["channels"], case["channels"], full)]
    if kind == "segment":
        return [(5, 3, 16, half), (3, 1, 16, half), (1, 16, 48, half), (3, 48, 48, quarter), (3, 48, 48, quarter), (1, 96, 32, half),
                (3, 32, 32, half), (1, 32, 21, full)]
    if kind == "mobilenet":
        s, cin, out = w // 2, 32, [(3, 3, 32, (w // 2) ** 2)]
        for t, cout, stride in networks.MobileNetV2.BLOCKS:
            if t != 1:
                out.append((1, cin, cin * t, s * s))
            s //= stride
            out += [(3, 1, cin * t, s * s), (1, cin * t, cout, s * s)]
            cin = cout
        return out
    s, cin, out = w // 4, 64, [(7, 3, 64, half)]
    for stage, (blocks, mid) in enumerate(samples.ResNet50Sample.STAGES):
        for blk in range(blocks):
            o = s // 2 if stage and not blk else s
            if not blk:
                out.append((1, cin, 4 * mid, o * o))
            out += [(1, cin, mid, s * s), (3, mid, mid, o * o), (1, mid, 4 * mid, o * o)]
            s, cin = o, 4 * mid
    return out + [(1, 2048, 1000, 1)]


def work(case):
    layers, item = _layers(case), 2 if case["storage"] == "f16" else 4
    frames = case.get("frames", 1)
    flops = frames * sum(2.0 * k * k * ci * co * n for k, ci, co, n in layers)
    weights = item * sum(k * k * ci * co for k, ci, co, _ in layers)
    c, rows, cols = result_shape(case)
    values_in = (case["channels"] if case["net"] == "conv" else 3) * case["width"] * case["height"]
    values_out = (2 if case["net"] == "segment" and case["drive"] == "frame" else c) * rows * cols
    one = item if case["drive"] == "resident" else 4      # (host buffers hold 32-bit values in either storage)
    return {"bytes": weights + frames * one * (values_in + values_out), "flops": flops}


def tolerance(case):
    """32-bit tensors: sums of hundreds to thousands of products over up to fifty layers, each of which carries the
    operands to 2^-16 and better.  16-bit tensors: rounded to 11 bits behind every layer; a last bit that falls the
    other way early in a deep network is a few thousandths to a hundredth at its end (near-ties change their label)."""
    if case["storage"] == "f32":
        return {"rel": 1e-4, "differ": 1e-3}
    if case["net"] == "conv":
        return {"rel": 1e-3}
    return {"rel": 2e-2 if case["net"] in ("resnet50", "mobilenet") else 1e-2, "differ": 1e-2}
