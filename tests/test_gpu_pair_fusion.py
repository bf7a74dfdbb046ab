"""Two 3x3 layers between tensors of few channels as one launch (a residual block of a small style net, the middle of a
decoder).  Parity against the oracle, agreement with the layers' own launches, and the conditions under which the engine
keeps them apart.  Tolerances: fp32 storage 3e-6 (two convolutions of 22-bit operands and fp32 sums, 3e-7 each), fp16
storage 2e-3."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng
from fyusenet_amd.builders import ActType, ConvLayerBuilder, LayerType, UpDownLayerBuilder
from oracle import oracle as O
from util import combos, device_bytes, rel_l2

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 3e-6, fa.STORAGE_F16: 2e-3}
# (the layers apart: on fp32 tensors one of them may run the form whose correction terms are fp8 products, 1e-5 by itself)
AGREE = {fa.STORAGE_F32: 2e-5, fa.STORAGE_F16: 2e-3}


class Pair(networks._StreamNet):
    """upload -> 1x1 front -> 3x3 first -> 3x3 second (+ front) -> 1x1 tail -> download; unpadded shallow layers repeat the
    frame's edge, deep ones read zeros outside."""
    config_id = 6
    input_key = (0, 0)

    def __init__(self, storage, c, cout, h, w, clamp, residual=True, act=ActType.RELU, mid_act=ActType.RELU, res_act=ActType.NONE, gain=1.0, reader=False, tail=True, mid=None):
        super().__init__(storage)
        self.c, self.cout, self.h, self.w, self.clamp, self.residual = c, cout, h, w, clamp, residual
        self.act, self.mid_act, self.res_act, self.gain, self.reader, self.tail, self.mid = act, mid_act, res_act, gain, reader, tail, mid or c

    def _three(self, no, name, cin, cout, src, act, pad_out, residual=None):
        b = ConvLayerBuilder(3, name).type(LayerType.CONVOLUTION2D).number(no).shape(cout, self.h, self.w, cin).prefixAct(act)
        if not self.clamp:
            b.deep().inputPadding(1).outputPadding(pad_out)
        if residual is not None:
            b.residual(self.res_act).residualPadding(0 if self.clamp else 1)
            self._edges.append((residual, no, 1))
        seed = self._next_seed()
        self._add(b, lambda: networks.conv_block(seed, cout, 3, cin))
        self._edges.append((src, no, 0))

    def define(self):
        h, w = self.h, self.w
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(self.c, h, w, self.c))
        self.conv(1, "front", 1, self.c, self.c, h, w, 0, pad_out=0 if self.clamp else 1)
        self._three(2, "first", self.c, self.mid, 1, self.act, 1)
        self._three(3, "second", self.mid, self.cout, 2, self.mid_act, 0, residual=1 if self.residual else None)
        last = 3
        if self.reader:
            self._three(4, "side", self.mid, 8, 2, ActType.NONE, 0)
            last = 4
        out = 3
        if self.tail:   # (a launch behind the pair that clears the words of its tensors' value ranges)
            last += 1
            self.conv(last, "tail", 1, self.cout, self.cout, h, w, 3)
            out = last
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.DOWNLOAD, "download").number(last + 1).shape(self.cout, h, w, self.cout).deep())
        self._edges.append((out, last + 1, 0))
        self.output_layer = last + 1

    def makeInput(self):
        return prng.uniform(571 + self.c + self.h, (self.c, self.h, self.w), -1.0, 1.0) * np.float32(self.gain)

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
    return infos["second"].startswith("conv_c16") and "launch of layer 3" in infos["first"]


SIZES = [(1, 1), (2, 16), (3, 17), (6, 32), (7, 15), (13, 50), (24, 33), (64, 48)]


@pytest.mark.parametrize(*combos(
    lambda c, size, rows, clamp, storage: (c != 48 or size in ((7, 15), (24, 33))) and (rows != 4 or size[0] > 4),
    c=([40, 48], str), size=(SIZES, lambda s: "%dx%d" % s), rows=([2, 4, 6], lambda r: "rows%d" % r), clamp=([False, True], lambda c: "edge" if c else "zeros"),
    storage=([fa.STORAGE_F32, fa.STORAGE_F16], lambda st: "f32" if st == fa.STORAGE_F32 else "f16")))
def test_pair_in_one_launch(c, size, rows, clamp, storage, monkeypatch):
    monkeypatch.setenv("FYNHIP_FORCE_PAIR_FUSION", "1")
    monkeypatch.setenv("FYNHIP_PAIR_ROWS", str(rows))
    h, w = size
    kw = dict(residual=h % 2 == 1, res_act=ActType.RELU if h == 3 else ActType.NONE)
    net = Pair(storage, c, c if kw["residual"] else 20, h, w, clamp, **kw)
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    assert together(infos) and "%dx16" % rows in infos["second"], infos["second"]
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    err = rel_l2(got, ref)
    monkeypatch.delenv("FYNHIP_FORCE_PAIR_FUSION")
    monkeypatch.setenv("FYNHIP_NO_PAIR_FUSION", "1")
    twin = Pair(storage, c, c if kw["residual"] else 20, h, w, clamp, **kw)
    _, apart, infos2 = run(twin)
    twin.cleanup()
    assert "conv_c16" not in infos2["second"] and "launch of layer 3" not in infos2["first"]
    print("   rel_l2=%.3e, against the layers apart %.3e" % (err, rel_l2(got, apart)), flush=True)
    assert err <= TOL[storage] and rel_l2(got, apart) <= AGREE[storage]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("what", ["leaky", "none", "large", "small", "rounds", "channels"])
def test_pair_variants(what, storage, monkeypatch):
    """Activations other than ReLU, magnitudes far from 1 (the tensor in between keeps a scale of its own), several rounds of
    workgroups, and channel counts between whole groups of eight."""
    gain = {"large": 3e6, "small": 3e-8}.get(what, 1.0) if storage == fa.STORAGE_F32 else {"large": 64.0, "small": 1.0 / 64}.get(what, 1.0)
    act = {"leaky": ActType.LEAKY_RELU, "none": ActType.NONE}.get(what, ActType.RELU)
    h, w = (200, 330) if what == "rounds" else (21, 40)
    monkeypatch.setenv("FYNHIP_FORCE_PAIR_FUSION", "1")
    net = Pair(storage, 38 if what == "channels" else 40, 38 if what == "channels" else 40, h, w, what in ("none", "large", "rounds"), act=act, mid_act=act, gain=gain)
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    assert together(infos), infos
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    err = rel_l2(got, ref)
    print("   rel_l2=%.3e" % err, flush=True)
    assert err <= TOL[storage]


@pytest.mark.parametrize("why", ["second_reader", "no_reuse", "ranges", "channels"])
def test_pair_keeps_its_launches_when_it_has_to(why, monkeypatch):
    """Another reader of the tensor in between, a network without buffer reuse, value-range words that only the first launch
    can clear, or another number of channels in between: two launches."""
    monkeypatch.setenv("FYNHIP_FORCE_PAIR_FUSION", "1")
    net = Pair(fa.STORAGE_F32, 40, 40, 12, 20, True, residual=why != "ranges", reader=why == "second_reader", tail=why != "ranges", gain=3e6 if why == "ranges" else 1.0, mid=24 if why == "channels" else None)
    x, got, infos = run(net, reuse=why != "no_reuse")
    desc = net.describe()
    net.cleanup()
    assert "conv_c16" not in infos["second"] and "launch of layer 3" not in infos["first"]
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    assert rel_l2(got, ref) <= 1e-4


def test_pair_weights_loaded_again_and_timed_apart(monkeypatch):
    """New weights on a network that is set up, a replayed graph behind them, and a pass that times its layers one by one."""
    monkeypatch.setenv("FYNHIP_FORCE_PAIR_FUSION", "1")
    net = Pair(fa.STORAGE_F32, 40, 40, 12, 20, True)
    x, first, _ = run(net)
    for name in ("first", "second"):
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
@pytest.mark.parametrize("rows", [2, 4, 6])
def test_nan_stays_in_its_window(rows, storage, monkeypatch):
    """What a NaN does not reach (two positions around it) is as it is without it, also where no activation drops it in
    between."""
    monkeypatch.setenv("FYNHIP_FORCE_PAIR_FUSION", "1")
    monkeypatch.setenv("FYNHIP_PAIR_ROWS", str(rows))
    net = Pair(storage, 40, 40, 24, 33, False, act=ActType.NONE, mid_act=ActType.NONE)
    x, want, infos = run(net)
    assert together(infos)
    y = x.copy()
    y[0, 12, 16] = np.nan
    net.setInput(y)
    net.forward()
    net.finish()
    got = net.getOutput(net.output_layer)
    net.cleanup()
    mask = np.ones(got.shape[1:], bool)
    mask[10:15, 14:19] = False
    assert not np.array_equal(got, want) and rel_l2(got[:, mask], want[:, mask]) <= TOL[storage]


@pytest.mark.parametrize("channels,more", [(24, False), (40, True)])
def test_no_memory_for_pairs_that_no_variant_computes(channels, more, monkeypatch):
    """The pair's input keeps its buffer until the second layer has run only where that layer's launch may read it."""
    monkeypatch.setenv("FYNHIP_AUTOTUNE", "0")
    with_pairs = device_bytes(Pair(fa.STORAGE_F32, channels, channels, 96, 96, True, residual=False))
    monkeypatch.setenv("FYNHIP_NO_PAIR_FUSION", "1")
    without = device_bytes(Pair(fa.STORAGE_F32, channels, channels, 96, 96, True, residual=False))
    assert with_pairs > without if more else with_pairs == without
