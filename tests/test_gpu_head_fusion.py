"""A 9x9 layer on an image and the 3x3 layer with a step of two behind it as one launch (the first layers of a style net).
Parity against the oracle, agreement with the layers' own launches, and the conditions under which the engine keeps them
apart.  Tolerances: fp32 storage 2e-5 (the first layer's correction terms are fp8 products, 1e-5 by itself), fp16 storage
2e-3."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng
from fyusenet_amd.builders import ActType, ConvLayerBuilder, LayerType, UpDownLayerBuilder
from oracle import oracle as O
from util import combos, rel_l2

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 2e-5, fa.STORAGE_F16: 2e-3}


class Head(networks._StreamNet):
    """upload -> 9x9 first -> 3x3 second with a step of two -> 1x1 or 3x3 tail -> 1x1 tail -> download"""
    config_id = 6
    input_key = (0, 0)

    def __init__(self, storage, size, cin=3, mid=32, cout=64, act=ActType.NONE, mid_act=ActType.RELU, gain=1.0, reader=False, bn=True, pads=(4, 1, 0), tail=True, edge=False):
        super().__init__(storage)
        (self.h, self.w), self.cin, self.mid, self.cout = size, cin, mid, cout
        self.act, self.mid_act, self.gain, self.reader, self.bn, self.pads, self.tail, self.edge = act, mid_act, gain, reader, bn, (0, 0, 0) if edge else pads, tail, edge

    def _head(self, no, name, k, cin, cout, src, stride, act, pad_out):
        """(edge: a shallow layer, which repeats the frame's edge)"""
        if not self.edge:
            self.conv(no, name, k, cin, cout, self.h, self.w, src, stride=stride, act=act, pad_out=pad_out, bn=self.bn)
            return
        b = ConvLayerBuilder(k, name).type(LayerType.CONVOLUTION2D).number(no).shape(cout, self.h, self.w, cin).prefixAct(act).downsample(stride)
        seed = self._next_seed()
        self._add(b, lambda: networks.conv_block(seed, cout, k, cin))
        self._edges.append((src, no, 0))

    def define(self):
        h, w, (pin, pmid, pout) = self.h, self.w, self.pads
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(self.cin, h, w, self.cin).outputPadding(pin))
        self._head(1, "first", 9, self.cin, self.mid, 0, 1, self.act, pmid)
        self._head(2, "second", 3, self.mid, self.cout, 1, 2, self.mid_act, pout)
        last, h2, w2 = 3, h // 2, w // 2
        if self.reader:
            self.conv(3, "side", 3, self.mid, 8, h, w, 1)
            last = 4
        self.conv(last, "tail", 2 * pout + 1, self.cout, self.cout, h2, w2, 2)
        last += 1
        if self.tail:   # (a launch that clears the word of the second layer's value range)
            self.conv(last, "tail2", 1, self.cout, self.cout, h2, w2, last - 1)
            last += 1
        last -= 1
        self._add(UpDownLayerBuilder(UpDownLayerBuilder.DOWNLOAD, "download").number(last + 1).shape(self.cout, h2, w2, self.cout).deep())
        self._edges.append((last, last + 1, 0))
        self.output_layer = last + 1

    def makeInput(self):
        return prng.uniform(877 + self.cin + self.h, (self.cin, self.h, self.w), -1.0, 1.0) * np.float32(self.gain)

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
    return infos["second"].startswith("conv_a16") and "launch of layer 2" in infos["first"]


@pytest.fixture
def forced(monkeypatch):
    monkeypatch.setenv("FYNHIP_FORCE_HEAD_FUSION", "1")
    monkeypatch.setenv("FYNHIP_FORCE_P16_CONV", "1")   # (the first layer in its small-input form at these sizes too)
    monkeypatch.setenv("FYNHIP_P16_TILE", "4,16")
    return monkeypatch


# (tiles of 4 x 31 positions of the second layer's output, an odd last row or column of the first layer's)
SIZES = [(2, 2), (8, 62), (9, 63), (10, 64), (7, 125), (17, 30), (31, 131), (64, 48)]
STORAGE = ([fa.STORAGE_F32, fa.STORAGE_F16], lambda st: "f32" if st == fa.STORAGE_F32 else "f16")


@pytest.mark.parametrize(*combos(
    lambda size, channels, edge, storage: channels != (1, 8, 8) or not edge,
    size=(SIZES, lambda s: "%dx%d" % s), channels=([(3, 32, 64), (4, 20, 24), (3, 12, 20), (1, 8, 8)], lambda c: "%d_%d_%d" % c),
    edge=([False, True], lambda e: "edge" if e else "zeros"), storage=STORAGE))
def test_head_in_one_launch(size, channels, edge, storage, forced):
    cin, mid, cout = channels
    kw = dict(cin=cin, mid=mid, cout=cout, edge=edge, pads=(4, 1, 0) if cin == 3 else (4, 1, 1), bn=cin != 4)
    net = Head(storage, size, **kw)
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    assert together(infos), infos
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    forced.delenv("FYNHIP_FORCE_HEAD_FUSION")
    forced.setenv("FYNHIP_NO_HEAD_FUSION", "1")
    twin = Head(storage, size, **kw)
    _, apart, infos2 = run(twin)
    twin.cleanup()
    assert "conv_a16" not in infos2["second"] and "launch of layer 2" not in infos2["first"]
    print("   rel_l2=%.3e, against the layers apart %.3e" % (rel_l2(got, ref), rel_l2(got, apart)), flush=True)
    assert rel_l2(got, ref) <= TOL[storage] and rel_l2(got, apart) <= TOL[storage]


@pytest.mark.parametrize("storage", STORAGE[0], ids=STORAGE[1])
@pytest.mark.parametrize("what", ["leaky", "none", "prefix", "large", "small", "rounds", "few", "few_leaky"])
def test_head_variants(what, storage, forced):
    """Activations on either input, magnitudes far from 1 (the tensor in between has a scale of its own, tile by tile), and several
    tiles a workgroup."""
    gain = {"large": 3e6, "small": 3e-8}.get(what, 1.0) if storage == fa.STORAGE_F32 else {"large": 64.0, "small": 1.0 / 64}.get(what, 1.0)
    mid_act = {"leaky": ActType.LEAKY_RELU, "few_leaky": ActType.LEAKY_RELU, "none": ActType.NONE}.get(what, ActType.RELU)
    net = Head(storage, (260, 700) if what in ("rounds", "few") else (21, 140), mid=12 if "few" in what else 32, cout=20 if "few" in what else 64, edge="few" in what, mid_act=mid_act, act=ActType.LEAKY_RELU if what == "prefix" else ActType.NONE, gain=gain, bn=what != "small")
    x, got, infos = run(net, passes=2)
    desc = net.describe()
    net.cleanup()
    assert together(infos), infos
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    print("   rel_l2=%.3e" % rel_l2(got, ref), flush=True)
    assert rel_l2(got, ref) <= TOL[storage]


@pytest.mark.parametrize("why", ["second_reader", "ranges", "exact"])
def test_head_keeps_its_launches_when_it_has_to(why, forced):
    """Another reader of the tensor in between, value-range words that only the first launch can clear, or correction terms in
    fp16 asked for."""
    if why == "exact":
        forced.setenv("FYNHIP_EXACT_SPLIT", "1")
    net = Head(fa.STORAGE_F32, (24, 70), reader=why == "second_reader", tail=why != "ranges")
    x, got, infos = run(net)
    desc = net.describe()
    net.cleanup()
    assert "conv_a16" not in infos["second"] and "launch of layer 2" not in infos["first"]
    ref = O.run_network(desc, {net.input_key: x})[net.output_layer]
    assert rel_l2(got, ref) <= TOL[fa.STORAGE_F32]


@pytest.mark.parametrize(*combos(
    lambda size, channels, edge, storage: True,
    size=([(2, 3), (9, 63), (24, 70), (33, 125)], lambda s: "%dx%d" % s), channels=([(3, 32, 64), (4, 20, 24), (3, 12, 20)], lambda c: "%d_%d_%d" % c), edge=([False, True], lambda e: "edge" if e else "zeros"), storage=STORAGE))
def test_head_writes_the_tensor_in_between_where_all_stay_readable(size, channels, edge, storage, forced):
    """Without buffer reuse the launch writes the first layer's tensor too, its odd last row and column and its frame of zeros
    included, and the second layer's is the same to the bit as with reuse."""
    outs = []
    for reuse in (True, False):
        net = Head(storage, size, *channels, edge=edge)
        x, got, infos = run(net, reuse=reuse, passes=2)
        assert (together(infos)), infos
        outs.append(got)
        if not reuse:
            ref = O.run_network(net.describe(), {net.input_key: x})
            for no in (1, 2):
                assert rel_l2(net.getOutput(no), ref[no]) <= TOL[storage]
            tiled = net.getOutput(1, fa.ORDER_GPU_DEEP)   # (tiles and the zeros around them)
            inside = net.getOutput(1)
            assert np.count_nonzero(tiled) <= inside.size
        net.cleanup()
    assert np.array_equal(*outs)


def test_head_weights_loaded_again_and_timed_apart(forced):
    """New weights on a network that is set up, a replayed graph behind them, and a pass that times its layers one by one."""
    net = Head(fa.STORAGE_F32, (24, 70))
    x, first, infos = run(net)
    assert together(infos)
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
    assert rel_l2(apart, ref) <= TOL[fa.STORAGE_F32]


@pytest.mark.parametrize("reuse", [True, False], ids=["reuse", "keep"])
@pytest.mark.parametrize("channels", [(4, 32, 64), (4, 12, 20)], ids=["32_64", "12_20"])
def test_head_keeps_the_bits_of_small_values_under_large_weights(channels, reuse, forced):
    """A colour channel that is dark in the frame, under weights 2^24 times the others': the tensor in between is far smaller than
    its weights would allow and is split by what it holds.  Weights are powers of two and pixels multiples of 1/64, so that
    the first layer's products are exact; what is left are 22-bit operands and fp32 sums, 3e-7 a layer."""
    net = Head(fa.STORAGE_F32, (30, 140), *channels)
    net.setup(reuseBuffers=reuse)
    lyr = net.layers["first"]
    cin, mid, _ = channels
    blk = np.array(lyr.weights, np.float32)
    w = blk[mid:mid + mid * 81 * cin].reshape(mid, 9, 9, cin)
    w[...] = np.sign(w) * np.exp2(np.clip(np.round(np.log2(np.abs(w) + 1e-9)), -6, -2))
    w[..., cin - 1] = 0.0
    w[:, 4, 4, cin - 1] = 2.0 ** 22
    lyr.loadWeightsAndBiases(blk)
    x = np.round(net.makeInput() * 64) / np.float32(64)
    x[cin - 1] = 0.0
    net.setInput(x)
    net.forward()
    got = net.getOutput(net.output_layer)
    infos = {layer.name: layer.kernelInfo() for layer in net.layers}
    desc = net.describe()
    net.cleanup()
    assert together(infos), infos
    err = rel_l2(got, O.run_network(desc, {net.input_key: x})[net.output_layer])
    print("   rel_l2=%.3e" % err, flush=True)
    assert err <= 3e-6


def test_head_is_timed_in_the_form_that_will_run(monkeypatch, tmp_path):
    """Without buffer reuse the launch writes the tensor in between too: that form is measured, and its choice noted, by itself."""
    notes = tmp_path / "choices"
    monkeypatch.setenv("FYNHIP_AUTOTUNE", "1")
    monkeypatch.setenv("FYNHIP_TUNE_CACHE", str(notes))
    found = []
    for reuse in (True, False):
        net = Head(fa.STORAGE_F32, (618, 516))
        net.setup(reuseBuffers=reuse)
        info = net.layers["first"].kernelInfo()
        net.cleanup()
        assert "tw=16" in info, info   # (the form that the launch is made for)
        found.append({line.split()[0] for line in notes.read_text().splitlines() if line.startswith("head:")})
    assert found[0] == {"head:0:3to32to64:618x516:e0:k0"} and found[1] - found[0] == {"head:0:3to32to64:618x516:e0:k1"}
