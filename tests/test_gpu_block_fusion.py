"""A bottleneck -- a 1x1, a 3x3 and a 1x1 layer, with an identity residual, a batch-norm layer in front or the shortcut
projection -- as one launch.  Parity against the oracle, agreement with the layers' own launches, and the conditions under
which the engine keeps them apart.  Tolerances: fp32 storage 3e-6 (three convolutions of 22-bit operands and fp32 sums, 3e-7
each; the bar of 1e-4 holds all the more), fp16 storage 2e-3 (every layer rounds to 11 bits)."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng
from fyusenet_amd.builders import ActType, UpDownLayerBuilder
from oracle import oracle as O
from util import combos, device_bytes, rel_l2

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 3e-6, fa.STORAGE_F16: 2e-3}
# (the layers apart: a 3x3 layer on fp32 tensors may run the form whose correction terms are fp8 products, 1e-5 by itself)
AGREE = {fa.STORAGE_F32: 2e-5, fa.STORAGE_F16: 2e-3}


class Block(networks._StreamNet):
    """upload -> 1x1 front [-> batch-norm] -> 1x1 reduce -> 3x3 -> 1x1 expand (+ front | + projection of it) -> download."""
    config_id = 4
    input_key = (0, 0)

    def __init__(self, storage, cin, mid, cout, h, w, kind="identity", act=ActType.RELU, mid_act=ActType.RELU, res_act=ActType.NONE, res_bn=False, halo=0, stride=1, reader=0, gain=1.0, tail=True):
        super().__init__(storage)
        self.cin, self.mid, self.cout, self.h, self.w, self.kind = cin, mid, cout, h, w, kind
        self.act, self.mid_act, self.res_act, self.res_bn, self.halo, self.stride, self.reader, self.gain, self.tail = act, mid_act, res_act, res_bn, halo, stride, reader, gain, tail

    def define(self):
        h, w, s = self.h, self.w, self.stride
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(self.cin, h, w, self.cin))
        self.conv(1, "front", 1, self.cin, self.cin, h, w, 0, pad_out=self.halo)
        src = 1
        if self.kind == "batchnorm":
            bn = fa.GPULayerBuilder("bn").type(fa.LayerType.BATCHNORM).number(2).shape(self.cin, h, w, self.cin).deep()
            seed = self._next_seed()
            self._add(bn, lambda: np.concatenate([prng.uniform(seed, (self.cin,), 0.5, 1.5), prng.normal(seed + 1, (self.cin,), 0.0, 0.3)]))
            self._edges.append((1, 2, 0))
            src = 2
        if self.kind == "projection":
            self.conv(3, "projection", 1, self.cin, self.cout, h, w, 1, act=self.act)
        self.conv(4, "reduce", 1, self.cin, self.mid, h, w, src, act=self.act, pad_out=1)
        self._builders[-1].inputPadding(self.halo)
        self.conv(5, "spatial", 3, self.mid, self.mid, h, w, 4, stride=s, act=self.mid_act)
        res = 3 if self.kind == "projection" else None if self.kind == "none" or self.cin != self.cout else 1
        kw = {} if res is None else {"residual": res, "res_act": self.res_act, "res_pad": self.halo if res == 1 else 0}
        self.conv(6, "expand", 1, self.mid, self.cout, h // s, w // s, 5, act=ActType.RELU, **kw)
        if self.res_bn and res is not None:
            self._builders[-1].residual(self.res_act, True)
        last = 6
        if self.reader:   # something else reads the result of one of the layers in between
            rh, rw = (h, w) if self.reader == 4 else (h // s, w // s)
            self.conv(7, "side", 1, self.mid, 16, rh, rw, self.reader)
            self._builders[-1].inputPadding(1 if self.reader == 4 else 0)
            last = 7
        if self.tail:   # (a launch behind the block that clears the words of its tensors' value ranges)
            last += 1
            self.conv(last, "tail", 1, self.cout, self.cout, h // s, w // s, 6)
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.DOWNLOAD, "download").number(last + 1).shape(self.cout, h // s, w // s, self.cout).deep())
        self._edges.append((last if self.tail else 6, last + 1, 0))
        self.output_layer = last + 1

    def makeInput(self):
        return prng.uniform(991 + self.cin + self.h, (self.cin, self.h, self.w), -1.0, 1.0) * np.float32(self.gain)

    def setInput(self, x):
        self.layers[0].setInput(x, 0)


def run(net, reuse=True, passes=1):
    net.setup(reuseBuffers=reuse)
    x = net.makeInput()
    net.setInput(x)
    for _ in range(passes):
        net.forward()
    net.finish()
    out = net.getOutput(net.output_layer)
    infos = {lyr.name: lyr.kernelInfo() for lyr in net.layers}
    return x, out, infos


def together(infos):
    return infos["expand"].startswith("conv_b16") and all("launch of layer 6" in infos[n] for n in ("reduce", "spatial"))


CASES = [
    # (cin, mid, cout, h, w, kind, storages)
    (256, 64, 256, 56, 56, "identity", 2),
    (256, 64, 256, 12, 12, "batchnorm", 2),
    (64, 64, 256, 28, 28, "projection", 2),
    (256, 64, 256, 13, 11, "none", 2),        # ragged tiles
    (200, 48, 200, 5, 3, "identity", 2),      # channel counts between the compiled ones, less than two tiles
    (200, 48, 232, 9, 15, "batchnorm", 2),
    (40, 24, 72, 15, 9, "projection", 2),
    (256, 64, 256, 1, 1, "identity", 2),
    (256, 64, 256, 72, 100, "identity", 2),   # more than one round of workgroups
    (512, 128, 512, 28, 28, "identity", 1),   # (fp16 tensors only)
    (392, 104, 392, 7, 10, "batchnorm", 1),
]


@pytest.mark.parametrize(*combos(
    lambda case, storage: storage == fa.STORAGE_F16 or case[6] == 2,
    case=(CASES, lambda c: "%d_%d_%d_%dx%d_%s" % c[:6]), storage=([fa.STORAGE_F32, fa.STORAGE_F16], lambda st: "f32" if st == fa.STORAGE_F32 else "f16")))
def test_bottleneck_in_one_launch(case, storage, monkeypatch):
    cin, mid, cout, h, w, kind, _ = case
    if kind == "batchnorm":   # (a form of the 1x1 layer that takes the batch-norm layer in front)
        monkeypatch.setenv("FYNHIP_FORCE_KR16_CONV", "1")
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")

    def make():
        return Block(storage, cin, mid, cout, h, w, kind=kind, res_bn=h % 2 == 0)
    net = make()
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    print("  ", infos["expand"][:200], flush=True)
    assert together(infos)
    if kind == "batchnorm":
        assert "batch-norm layer in front" in infos["expand"] and "no launch of its own" in infos["bn"]
    if kind == "projection":
        assert "projection 3" in infos["expand"] and "launch of layer 6" in infos["projection"]
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    err = rel_l2(got, ref)
    monkeypatch.delenv("FYNHIP_FORCE_BLOCK_FUSION")
    monkeypatch.setenv("FYNHIP_NO_BLOCK_FUSION", "1")
    twin = make()
    _, apart, infos2 = run(twin)
    twin.cleanup()
    assert "conv_b16" not in infos2["expand"] and "launch of layer 6" not in infos2["reduce"]
    print("   rel_l2=%.3e, against the layers apart %.3e" % (err, rel_l2(got, apart)), flush=True)
    assert err <= TOL[storage] and rel_l2(got, apart) <= AGREE[storage]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("what", ["leaky", "none", "res_relu", "halo", "large", "small"])
def test_bottleneck_variants(what, storage, monkeypatch):
    """Activations other than ReLU, a ReLU on the residual, an input with a halo, and magnitudes far from 1: every tensor in
    between has to keep its own scale (fp32 tensors)."""
    if what in ("large", "small") and storage == fa.STORAGE_F16:
        gain = {"large": 64.0, "small": 1.0 / 64}[what]
    else:
        gain = {"large": 3e6, "small": 3e-8}.get(what, 1.0)
    kw = {"leaky": {"act": ActType.LEAKY_RELU, "mid_act": ActType.LEAKY_RELU}, "none": {"act": ActType.NONE, "mid_act": ActType.NONE}, "res_relu": {"res_act": ActType.RELU, "res_bn": True},
          "halo": {"halo": 2}}.get(what, {})
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    net = Block(storage, 256, 64, 256, 10, 18, gain=gain, **kw)
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    assert together(infos)
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    err = rel_l2(got, ref)
    print("   rel_l2=%.3e" % err, flush=True)
    assert err <= TOL[storage]


@pytest.mark.parametrize("why", ["step", "second_reader", "middle_reader", "no_reuse", "wide_fp32", "ranges"])
def test_bottleneck_keeps_its_launches_when_it_has_to(why, monkeypatch):
    """A step in the 3x3 layer, another reader of a tensor in between, a network without buffer reuse, a shape that no
    variant is compiled for, or value-range words that only the block's first launches can clear: three launches."""
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    mid, cin = (128, 512) if why == "wide_fp32" else (64, 256)
    net = Block(fa.STORAGE_F32, cin, mid, cin, 12, 12, kind="none" if why in ("step", "ranges") else "identity", stride=2 if why == "step" else 1, reader={"second_reader": 4, "middle_reader": 5}.get(why, 0),
                tail=(why != "ranges"), gain=3e6 if why == "ranges" else 1.0)
    x, got, infos = run(net, reuse=(why != "no_reuse"))
    desc = net.describe()
    net.cleanup()
    assert "conv_b16" not in infos["expand"] and "launch of layer 6" not in infos["reduce"]
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    assert rel_l2(got, ref) <= 1e-4


def test_bottleneck_weights_loaded_again_and_timed_apart(monkeypatch):
    """New weights on a network that is set up, a replayed graph behind them, and a pass that times its layers one by one."""
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    net = Block(fa.STORAGE_F32, 64, 64, 256, 12, 20, kind="projection")
    x, first, _ = run(net)
    for name in ("reduce", "spatial", "expand", "projection"):
        lyr = net.layers[name]
        lyr.loadWeightsAndBiases(lyr.weights * np.float32(0.75))
    net.useGraph(True)
    outs = []
    for _ in range(3):
        net.forward()
        outs.append(net.getOutput(net.output_layer).copy())
    desc = net.describe()
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    assert all(np.array_equal(o, outs[0]) for o in outs) and rel_l2(outs[0], ref) <= TOL[fa.STORAGE_F32] and rel_l2(outs[0], first) > 1e-2
    net.useGraph(False)
    net.enableTimings(True)
    net.forward()
    apart = net.getOutput(net.output_layer)
    net.cleanup()
    assert rel_l2(apart, ref) <= AGREE[fa.STORAGE_F32]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("kind", ["identity", "projection"])
def test_nan_stays_in_its_window(kind, storage, monkeypatch):
    """What a NaN does not reach (one position around it, by the 3x3 layer) is as it is without it, also where no activation
    drops it in between."""
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    cin = 256 if kind == "identity" else 64
    net = Block(storage, cin, 64, 256, 14, 11, kind=kind, act=ActType.NONE, mid_act=ActType.NONE)
    x, want, infos = run(net)
    assert together(infos)
    y = x.copy()
    y[0, 6, 5] = np.nan
    net.setInput(y)
    net.forward()
    net.finish()
    got = net.getOutput(net.output_layer)
    net.cleanup()
    mask = np.ones(got.shape[1:], bool)
    mask[5:8, 4:7] = False
    assert not np.array_equal(got, want) and rel_l2(got[:, mask], want[:, mask]) <= TOL[storage]


class Chain(Block):
    """upload -> 1x1 -> 3x3 -> 1x1 -> 3x3 -> 1x1 [-> 3x3 -> 1x1 ...] -> tail -> download: every 1x1 layer in the middle could end a
    block and begin one."""

    def __init__(self, storage, channels, h, w, blocks):
        super().__init__(storage, channels, channels, channels, h, w)
        self.blocks = blocks

    def define(self):
        h, w, c = self.h, self.w, self.cin
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(c, h, w, c))
        self.conv(1, "front", 1, c, c, h, w, 0)
        self.conv(2, "p0", 1, c, c, h, w, 1, act=ActType.RELU, pad_out=1)
        last = 2
        for i in range(1, self.blocks + 1):
            self.conv(last + 1, "s%d" % i, 3, c, c, h, w, last, act=ActType.RELU)
            self.conv(last + 2, "p%d" % i, 1, c, c, h, w, last + 1, act=ActType.RELU, pad_out=1 if i < self.blocks else 0)
            last += 2
        self.conv(last + 1, "tail", 1, c, c, h, w, last)
        self.conv(last + 2, "tail2", 1, c, c, h, w, last + 1)
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.DOWNLOAD, "download").number(last + 3).shape(c, h, w, c).deep())
        self._edges.append((last + 2, last + 3, 0))
        self.output_layer = last + 3


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("channels,h,w", [(64, 9, 14), (32, 12, 12)])
@pytest.mark.parametrize("blocks", [2, 3])
def test_blocks_that_share_a_layer(blocks, channels, h, w, storage, monkeypatch):
    """A 1x1 layer that ends one block does not begin the next one: its launch is what writes the tensor between them."""
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    net = Chain(storage, channels, h, w, blocks)
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    joined = [n for n in infos if infos[n].startswith("conv_b16")]
    inside = [n for n in infos if "no launch of its own" in infos[n]]
    print("  ", joined, inside, flush=True)
    assert (joined, inside) == ((["p1"], ["p0", "s1"]) if blocks == 2 else (["p1", "p3"], ["p0", "s1", "p2", "s3"]))
    err = rel_l2(got, O.run_network(desc, {net.input_key: x})[net.output_layer])
    print("   rel_l2=%.3e" % err, flush=True)
    assert err <= AGREE[storage]   # (a 3x3 layer runs by itself; nine roundings to 11 bits, 3e-4 each, add up to 1e-3)


class Scores(Block):
    """upload -> two 1x1 layers -> 1x1 -> 3x3 -> 1x1 scores -> arg-max: a segmentation head that ends as a block does."""

    def __init__(self, storage, channels, classes, h, w):
        super().__init__(storage, channels, channels, classes, h, w)
        self.output_layer, self.argmax_layer = 5, 6

    def define(self):
        h, w, c = self.h, self.w, self.cin
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(c, h, w, c))
        self.conv(1, "first", 1, c, c, h, w, 0)
        self.conv(2, "front", 1, c, c, h, w, 1)
        self.conv(3, "reduce", 1, c, c, h, w, 2, act=ActType.RELU, pad_out=1)
        self.conv(4, "spatial", 3, c, c, h, w, 3, act=ActType.RELU)
        self.conv(5, "scores", 1, c, self.cout, h, w, 4, act=ActType.RELU)
        self._add(fa.ArgMaxLayerBuilder("labels").number(6).shape(2, h, w, self.cout).deep())
        self._edges.append((5, 6, 0))


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("forced", [True, False], ids=["streaming", "general"])
@pytest.mark.parametrize("channels,classes,h,w", [(64, 21, 128, 128), (32, 21, 18, 13)])
def test_argmax_behind_a_block(channels, classes, h, w, forced, storage, monkeypatch):
    """Where the last layer also computes the arg-max layer behind it, it keeps its launch; elsewhere the arg-max layer runs behind
    the block.  Labels and best values are those of this frame's scores."""
    monkeypatch.setenv("FYNHIP_FORCE_BLOCK_FUSION", "1")
    monkeypatch.setenv("FYNHIP_FORCE_S16_CONV" if forced else "FYNHIP_NO_S16_CONV", "1")
    net = Scores(storage, channels, classes, h, w)
    net.setup()
    infos = {lyr.name: lyr.kernelInfo() for lyr in net.layers}
    assert ("conv_s16" if forced else "conv_b16") in infos["scores"].split("; apart")[0], infos["scores"]
    assert ("no launch of its own" in infos["labels"]) == forced
    for gain in (1.0, -1.0):   # (another frame, another answer)
        x = net.makeInput() * np.float32(gain)
        net.setInput(x)
        net.forward()
        labels, best = net.getArgMax(net.argmax_layer)
        scores = net.getOutput(net.output_layer)
        ref = O.run_network(net.describe(), {net.input_key: x})
        assert rel_l2(scores, ref[net.output_layer]) <= AGREE[storage]
        assert np.array_equal(labels, scores.argmax(axis=0)) and np.array_equal(best, scores.max(axis=0))
    net.cleanup()


@pytest.mark.parametrize("channels,mid,more", [(512, 128, False), (256, 64, True)])
def test_no_memory_for_blocks_that_no_variant_computes(channels, mid, more, monkeypatch):
    """The block's input keeps its buffer until the last layer has run only where that layer's launch may read it."""
    monkeypatch.setenv("FYNHIP_AUTOTUNE", "0")
    with_blocks = device_bytes(Block(fa.STORAGE_F32, channels, mid, channels, 24, 24, kind="none"))
    monkeypatch.setenv("FYNHIP_NO_BLOCK_FUSION", "1")
    without = device_bytes(Block(fa.STORAGE_F32, channels, mid, channels, 24, 24, kind="none"))
    assert with_blocks > without if more else with_blocks == without


def test_block_on_an_input_beyond_32_bit_offsets(monkeypatch):
    """A few positions in a halo so wide that the tensor has more than 2^30 values: the layers run by themselves."""
    outs = []
    for switch in ("FYNHIP_FORCE_BLOCK_FUSION", "FYNHIP_NO_BLOCK_FUSION"):
        monkeypatch.setenv(switch, "1")
        net = Block(fa.STORAGE_F16, 256, 64, 256, 4, 4, kind="none", halo=1024)
        _, got, infos = run(net)
        net.cleanup()
        assert "conv_b16" not in infos["expand"]
        outs.append(got)
        monkeypatch.delenv(switch)
    assert np.any(outs[0]) and rel_l2(*outs) <= TOL[fa.STORAGE_F16]


@pytest.mark.parametrize("storage,channels,mid,side,one", [
    (fa.STORAGE_F32, 64, 32, 64, True), (fa.STORAGE_F32, 64, 32, 68, False), (fa.STORAGE_F32, 128, 64, 68, True), (fa.STORAGE_F32, 128, 64, 84, False), (fa.STORAGE_F16, 64, 32, 68, True),
    (fa.STORAGE_F16, 64, 32, 84, False)])
def test_blocks_that_nothing_is_timed_for(storage, channels, mid, side, one, monkeypatch):
    """One launch in a single round of 256 workgroups, and in up to 400 where the layers are wide enough or the tensors fp16."""
    monkeypatch.setenv("FYNHIP_AUTOTUNE", "0")
    net = Block(storage, channels, mid, channels, side, side)
    net.setup()
    infos = {lyr.name: lyr.kernelInfo() for lyr in net.layers}
    net.cleanup()
    assert together(infos) == one, infos["expand"]
