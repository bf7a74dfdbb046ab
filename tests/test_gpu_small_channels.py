"""Convolutions between tensors of few channels: the form that gathers 3x3 windows from the tensor (conv_g16), at the
edges of its 16-position tiles, channel groups and fragments, for every edge rule, step and source step; and a sigmoid or
tanh layer that the convolution in front of it applies to what it stores.  The streaming 1x1 form (conv_s16) at the edges of
its trips, chunks and fragments, with the arg-max layer behind it.  Tolerances: rel-L2 <= 1e-4 (fp32 storage),
<= 2e-3 (fp16 storage)."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng, samples
from fyusenet_amd.builders import ActType, ConvLayerBuilder, LayerType
from oracle import oracle as O
from util import conv_block, oracle_single, rel_l2, run_single

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 1e-4, fa.STORAGE_F16: 2e-3}

# cin, cout, h, w, stride, deep, act, residual, fragments per wave (0: the engine's choice)
CASES = [
    (16, 16, 5, 3, 1, False, ActType.NONE, None, 0),            # fewer positions than a tile
    (16, 20, 24, 34, 2, False, ActType.RELU, None, 1),          # steps over the input, ragged fragment, a wave per fragment
    (12, 20, 33, 47, 1, False, ActType.RELU, None, 2),          # channels behind the count, odd rows
    (24, 12, 16, 16, 1, True, ActType.LEAKY_RELU, None, 1),     # zero padding, a leak
    (24, 40, 31, 65, 2, True, ActType.CLIP, None, 3),
    (32, 64, 9, 129, 1, True, ActType.NONE, ActType.RELU, 4),
    (40, 40, 78, 41, 1, False, ActType.RELU, ActType.NONE, 3),  # several tiles per wave
    (40, 36, 20, 20, 1, False, ActType.NONE, ActType.RELU, 1),
    (48, 32, 40, 23, 1, True, ActType.RELU, None, 2),
    (64, 16, 17, 50, 2, True, ActType.RELU, None, 1),
]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dto%d_%dx%d_s%d_%s" % (c[0], c[1], c[2], c[3], c[4], "deep" if c[5] else "shallow"))
def test_gathered_windows(monkeypatch, case, storage):
    cin, cout, h, w, stride, deep, act, residual, frags = case
    monkeypatch.setenv("FYNHIP_FORCE_G16_CONV", "1")
    if frags:
        monkeypatch.setenv("FYNHIP_G16_FRAGS", str(frags))
    b = ConvLayerBuilder(3, "conv").type(LayerType.CONVOLUTION2D).number(1).shape(cout, h, w, cin).prefixAct(act).downsample(stride)
    if act == ActType.LEAKY_RELU:
        b.leakyReLU(0.2)
    if act == ActType.CLIP:
        b.clip(-0.5, 0.75)
    if deep:
        b.deep().inputPadding(1).outputPadding(1)
    inputs = [prng.normal(41 + cin, (cin, h, w))]
    if residual is not None:
        b.residual(residual)
        if deep:
            b.residualPadding(1)
        inputs.append(prng.normal(43 + cin, (cout, h // stride, w // stride)))
    weights = conv_block(47 + cin, cout, 3, cin)
    got, info = run_single(b, storage, inputs, weights)
    assert "conv_g16" in info, info
    want = oracle_single(b, storage, inputs, weights)
    assert rel_l2(got, want) <= TOL[storage]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("cin,cout,h,w,step,stride", [(40, 20, 13, 16, 0.5, 2), (20, 12, 12, 19, 0.25, 2), (16, 16, 7, 9, 0.5, 1)])
def test_gathered_windows_of_repeated_pixels(monkeypatch, storage, cin, cout, h, w, step, stride):
    monkeypatch.setenv("FYNHIP_FORCE_G16_CONV", "1")
    b = ConvLayerBuilder(3, "conv").type(LayerType.FRACCONVOLUTION2D).number(1).shape(cout, h, w, cin).prefixAct(ActType.RELU).downsample(stride).sourceStep(step)
    x, weights = prng.normal(61, (cin, h, w)), conv_block(67, cout, 3, cin)
    got, info = run_single(b, storage, [x], weights)
    assert "conv_g16" in info, info
    assert rel_l2(got, oracle_single(b, storage, [x], weights)) <= TOL[storage]


# cin, cout, h, w, stride, deep, act, residual, rows of a tile
WINDOWED = [
    (16, 16, 2, 3, 1, False, ActType.NONE, None, 2),             # fewer positions than a row
    (12, 20, 24, 34, 2, False, ActType.RELU, None, 4),           # steps over the input, a ragged fragment, a window's even and odd columns
    (16, 20, 25, 33, 2, True, ActType.LEAKY_RELU, None, 2),      # zero padding, a leak
    (20, 40, 31, 65, 2, False, ActType.RELU, None, 2),
    (24, 48, 16, 18, 2, True, ActType.CLIP, None, 4),
    (40, 40, 11, 17, 1, False, ActType.RELU, ActType.NONE, 5),   # a row and a column behind the last whole tile
    (40, 36, 20, 20, 1, True, ActType.NONE, ActType.RELU, 2),
    (40, 12, 30, 47, 2, True, ActType.RELU, None, 4),
    (48, 33, 40, 23, 1, True, ActType.RELU, None, 5),            # channels behind the output's count
    (64, 64, 9, 33, 1, True, ActType.RELU, ActType.RELU, 2),     # two blocks of output channels
    (64, 88, 14, 20, 1, False, ActType.NONE, ActType.NONE, 5),   # three, the last with 24 channels (six fragments)
    (64, 20, 22, 30, 2, True, ActType.RELU, None, 2),
    (40, 64, 7, 18, 1, True, ActType.RELU, None, 5),             # four fragments, two a block
    (24, 8, 90, 1000, 1, False, ActType.RELU, None, 2),          # 2835 tiles: workgroups walk six
    (40, 40, 130, 400, 1, False, ActType.RELU, ActType.RELU, 5), # 650 tiles, the residual of a second tile
]


def _windowed(case):
    cin, cout, h, w, stride, deep, act, residual, _ = case
    b = ConvLayerBuilder(3, "conv").type(LayerType.CONVOLUTION2D).number(1).shape(cout, h, w, cin).prefixAct(act).downsample(stride)
    if act == ActType.LEAKY_RELU:
        b.leakyReLU(0.2)
    if act == ActType.CLIP:
        b.clip(-0.5, 0.75)
    if deep:
        b.deep().inputPadding(1).outputPadding(1)
    if residual is not None:
        b.residual(residual)
        if deep:
            b.residualPadding(1)
    return b


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("case", WINDOWED, ids=lambda c: "%dto%d_%dx%d_s%d_%s_th%d" % (c[0], c[1], c[2], c[3], c[4], "deep" if c[5] else "shallow", c[8]))
def test_windows_in_lds(monkeypatch, case, storage):
    cin, cout, h, w, stride, deep, act, residual, rows = case
    monkeypatch.setenv("FYNHIP_P16N_ROWS", str(rows))
    b = _windowed(case)
    inputs = [prng.normal(141 + cin, (cin, h, w))]
    if residual is not None:
        inputs.append(prng.normal(143 + cin, (cout, h // stride, w // stride)))
    weights = conv_block(147 + cin, cout, 3, cin)
    got, info = run_single(b, storage, inputs, weights)
    assert "conv_p16n" in info and "of %dx16" % rows in info, info
    # (fp32 tensors: three passes over 22-bit operands, as in the other exact forms)
    assert rel_l2(got, oracle_single(b, storage, inputs, weights)) <= (2e-6 if storage == fa.STORAGE_F32 else TOL[storage])


# ... and fewer fragments of output channels in a workgroup than there are: the last element is their number
WINDOWED_BLOCKS = [
    (40, 40, 12, 16, 1, False, ActType.RELU, ActType.RELU, 2, 1),    # the samples' layers on small frames: three blocks, the last with eight channels
    (40, 40, 23, 37, 1, True, ActType.RELU, None, 5, 1),
    (20, 20, 24, 34, 2, False, ActType.NONE, ActType.NONE, 4, 1),    # two blocks, the last with four
    (16, 32, 9, 17, 1, True, ActType.LEAKY_RELU, None, 2, 1),
    (24, 33, 31, 20, 2, True, ActType.CLIP, ActType.RELU, 2, 1),     # three, the last with one channel
    (48, 44, 18, 33, 1, False, ActType.RELU, ActType.NONE, 5, 1),
    (40, 96, 11, 18, 2, False, ActType.NONE, None, 4, 2),            # three blocks of two
    (12, 128, 10, 15, 1, True, ActType.NONE, ActType.RELU, 5, 2),    # four
    (64, 64, 17, 30, 1, True, ActType.RELU, ActType.RELU, 5, 1),     # four blocks of one
    (64, 36, 13, 22, 2, False, ActType.RELU, None, 2, 1),
    (40, 40, 90, 300, 1, False, ActType.NONE, ActType.RELU, 5, 1),   # 342 tiles x 3 blocks: workgroups walk two and three
]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("case", WINDOWED_BLOCKS, ids=lambda c: "%dto%d_%dx%d_s%d_%s_th%d_fr%d" % (c[0], c[1], c[2], c[3], c[4], "deep" if c[5] else "shallow", c[8], c[9]))
def test_windows_in_lds_with_blocks_of_output_channels(monkeypatch, case, storage):
    cin, cout, h, w, stride, deep, act, residual, rows, frags = case
    monkeypatch.setenv("FYNHIP_P16N_ROWS", "%d,%d" % (rows, frags))
    b = _windowed(case[:9])
    inputs = [prng.normal(151 + cin, (cin, h, w))]
    if residual is not None:
        inputs.append(prng.normal(153 + cin, (cout, h // stride, w // stride)))
    weights = conv_block(157 + cin, cout, 3, cin)
    got, info = run_single(b, storage, inputs, weights)
    assert "conv_p16n" in info and "of %dx16" % rows in info and "%d fragment(s)" % frags in info, info
    assert rel_l2(got, oracle_single(b, storage, inputs, weights)) <= (2e-6 if storage == fa.STORAGE_F32 else TOL[storage])   # (as in the test above)


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("cin,cout,h,w,step,stride", [(40, 20, 13, 16, 0.5, 2), (20, 12, 12, 19, 0.25, 2), (16, 16, 7, 9, 0.5, 1)])
def test_windows_in_lds_of_repeated_pixels(monkeypatch, storage, cin, cout, h, w, step, stride):
    monkeypatch.setenv("FYNHIP_FORCE_P16N_CONV", "1")
    b = ConvLayerBuilder(3, "conv").type(LayerType.FRACCONVOLUTION2D).number(1).shape(cout, h, w, cin).prefixAct(ActType.RELU).downsample(stride).sourceStep(step)
    x, weights = prng.normal(161, (cin, h, w)), conv_block(167, cout, 3, cin)
    got, info = run_single(b, storage, [x], weights)
    assert "conv_p16n" in info, info
    assert rel_l2(got, oracle_single(b, storage, [x], weights)) <= (2e-6 if storage == fa.STORAGE_F32 else TOL[storage])


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("kernel,width,height", [(3, 64, 48), (9, 100, 76)])
def test_function_layer_applied_by_the_convolution_in_front(monkeypatch, storage, kernel, width, height):
    """The samples' last two layers as one launch and as two: the same values, and the tensors in front keep theirs."""
    outs = []
    for fused in (True, False):
        if not fused:
            monkeypatch.setenv("FYNHIP_NO_FUNCTION_FUSION", "1")
        net = samples.StyleNetSample(kernel, width, height, storage)
        net.setup()
        x = net.makeInput()
        for _ in range(2):   # (a second pass over reused buffers)
            net.setInput(x)
            net.forward()
            net.finish()
        assert ("no launch of its own" in net.layers[net.SIGMOID].kernelInfo()) == fused
        outs.append(net.getOutput(net.SIGMOID))
        if fused:
            want = O.run_network(net.describe(), {net.input_key: x})[net.SIGMOID]
        net.cleanup()
    assert rel_l2(outs[0], outs[1]) <= (1e-6 if storage == fa.STORAGE_F32 else 1e-4)
    assert rel_l2(outs[0], want) <= TOL[storage]


# cin, cout, h, w, stride, pads (in, out), act, residual
STREAMED = [
    (8, 8, 3, 5, 1, (0, 0), ActType.NONE, None),                 # fewer positions than a trip, a quarter of a chunk
    (32, 21, 37, 29, 1, (0, 1), ActType.RELU, None),             # ragged fragment, halo behind
    (40, 16, 20, 66, 1, (1, 0), ActType.LEAKY_RELU, None),       # ragged second chunk, halo in front, a leak
    (96, 32, 31, 33, 1, (0, 0), ActType.RELU, ActType.RELU),
    (16, 64, 50, 130, 2, (0, 0), ActType.CLIP, None),            # steps over the input
    (128, 20, 16, 17, 1, (0, 0), ActType.NONE, ActType.NONE),
]


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("case", STREAMED, ids=lambda c: "%dto%d_%dx%d_s%d" % c[:5])
def test_streamed_pointwise(monkeypatch, case, storage):
    cin, cout, h, w, stride, (pad_in, pad_out), act, residual = case
    monkeypatch.setenv("FYNHIP_FORCE_S16_CONV", "1")
    b = ConvLayerBuilder(1, "conv").type(LayerType.CONVOLUTION2D).number(1).shape(cout, h, w, cin).prefixAct(act).downsample(stride)
    b.deep().inputPadding(pad_in).outputPadding(pad_out)
    if act == ActType.LEAKY_RELU:
        b.leakyReLU(0.2)
    if act == ActType.CLIP:
        b.clip(-0.5, 0.75)
    inputs = [prng.normal(71 + cin, (cin, h, w))]
    if residual is not None:
        b.residual(residual).residualPadding(pad_out)
        inputs.append(prng.normal(73 + cin, (cout, h // stride, w // stride)))
    weights = conv_block(79 + cin, cout, 1, cin)
    got, info = run_single(b, storage, inputs, weights)
    assert "conv_s16" in info, info
    assert rel_l2(got, oracle_single(b, storage, inputs, weights)) <= TOL[storage]


class Labels(networks._StreamNet):
    """upload -> 3x3 conv -> 1x1 conv to the classes -> arg-max."""
    config_id = 7
    input_key = (0, 0)

    def __init__(self, storage, w, h, classes, act):
        super().__init__(storage)
        self.w, self.h, self.classes, self.act = w, h, classes, act
        self.output_layer, self.argmax_layer = 2, 3

    def define(self):
        w, h = self.w, self.h
        self._add(fa.UpDownLayerBuilder(fa.UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(3, h, w, 3).outputPadding(1))
        self.conv(1, "front", 3, 3, 32, h, w, 0)
        self.conv(2, "scores", 1, 32, self.classes, h, w, 1, act=ActType.RELU, bn=False)
        self._add(fa.ArgMaxLayerBuilder("labels").number(3).shape(2, h, w, self.classes).prefixAct(self.act).deep())
        self._edges.append((2, 3, 0))

    def setInput(self, x):
        self.layers[0].setInput(x, 0)


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("w,h,classes,act", [(150, 130, 21, ActType.NONE), (129, 129, 5, ActType.RELU), (131, 140, 64, ActType.NONE)])
def test_argmax_computed_by_the_convolution_in_front(monkeypatch, storage, w, h, classes, act):
    """Labels and best values are those of the stored scores: with ReLU on fetch many positions tie at zero."""
    monkeypatch.setenv("FYNHIP_FORCE_S16_CONV", "1")
    if storage == fa.STORAGE_F32 and classes > 32:
        classes = 32
    x = prng.uniform(9, (3, h, w), -1.0, 1.0)
    net = Labels(storage, w, h, classes, act)
    net.setup()
    for _ in range(2):
        net.setInput(x)
        net.forward()
        labels, best = net.getArgMax(3)
    assert "no launch of its own" in net.layers[3].kernelInfo()
    scores = net.getOutput(2)
    net.cleanup()
    fetched = np.maximum(scores, 0) if act == ActType.RELU else scores
    assert np.array_equal(labels, fetched.argmax(axis=0))
    assert np.array_equal(best, fetched.max(axis=0))
