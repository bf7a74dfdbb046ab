"""Convolutions between tensors of few channels: the form that gathers 3x3 windows from the tensor (conv_g16), at the
edges of its 16-position tiles, channel groups and fragments, for every edge rule, step and source step; and a sigmoid or
tanh layer that the convolution in front of it applies to what it stores.  Tolerances: rel-L2 <= 1e-4 (fp32 storage),
<= 2e-3 (fp16 storage)."""
import pytest

import fyusenet_amd as fa
from fyusenet_amd import prng, samples
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
