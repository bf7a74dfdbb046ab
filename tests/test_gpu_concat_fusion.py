"""A concatenation in one launch, with the bilinear scale layers in front of it and the batch-norm layer behind it: parity
against the oracle, equality with the separate launches, and the networks in which the engine leaves the layers alone.
Tolerances: rel-L2 <= 1e-4 (fp32 storage), <= 2e-3 (fp16 storage)."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng
from oracle import oracle as O
from util import rel_l2

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 1e-4, fa.STORAGE_F16: 2e-3}
A = fa.ActType


class Join(networks._StreamNet):
    """upload -> 1x1 conv at full size and, behind a stride-2 convolution, one at half size -> scaled up -> concatenation
    (-> batch-norm) -> 1x1 conv.  second_reader: the scaled tensor is read by another layer as well."""
    config_id = 8
    input_key = (0, 0)

    def __init__(self, storage, w, h, c_full, c_half, bn=True, scale=fa.ScalingType.LINEAR, second_reader=False, bn_act=A.RELU):
        super().__init__(storage)
        self.w, self.h, self.c_full, self.c_half = w, h, c_full, c_half
        self.bn, self.scale, self.second_reader, self.bn_act = bn, scale, second_reader, bn_act

    def define(self):
        w, h, cf, ch = self.w, self.h, self.c_full, self.c_half
        total = cf + ch
        self._add(fa.UpDownLayerBuilder(fa.UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(3, h, w, 3).outputPadding(1))
        self.conv(1, "full", 3, 3, cf, h, w, 0)
        self.conv(2, "half", 3, 3, ch, h, w, 0, stride=2)
        up = fa.ScaleLayerBuilder("up").number(3).shape(ch, h // 2, w // 2, ch).scale(2.0).scaleType(self.scale).prefixAct(A.RELU)
        self._add(up.deep())
        self._edges.append((2, 3, 0))
        cat = fa.ConcatLayerBuilder("cat").number(4).deep().input(ch, 0).input(cf, 0)
        cat.size(w, h)
        cat.outputChannels_ = total
        self._add(cat)
        self._edges += [(3, 4, 0), (1, 4, 1)]
        last = 4
        if self.bn:
            b = fa.GPULayerBuilder("bn").type(fa.LayerType.BATCHNORM).number(5).shape(total, h, w, total).prefixAct(self.bn_act).deep()
            seed = self._next_seed()
            self._add(b, lambda: np.concatenate([prng.uniform(seed, (total,), 0.5, 1.5), prng.normal(seed + 1, (total,), 0.0, 0.1)]))
            self._edges.append((4, 5, 0))
            last = 5
        self.conv(6, "mix", 1, total, 16, h, w, last, act=A.RELU)
        self.output_layer = 6
        if self.second_reader:
            self.conv(7, "aside", 1, ch, 16, h, w, 3)
            self.conv(8, "sum", 1, 16, 16, h, w, 7, residual=6)
            self.output_layer = 8

    def setInput(self, x):
        self.layers[0].setInput(x, 0)


def run(net, x, passes=2):
    net.setup()
    for _ in range(passes):
        net.setInput(x)
        net.forward()
        net.finish()
    return net.getOutput(net.output_layer)


@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("w,h,c_full,c_half,kw,joined", [
    (36, 28, 48, 48, {}, (True, True)),
    (130, 6, 8, 24, {"bn_act": A.NONE}, (True, None)),            # (a batch-norm layer without activation may be the reader's)
    (20, 22, 4, 12, {"bn": False}, (True, None)),                  # vectors of four channels
    (24, 20, 16, 40, {"scale": fa.ScalingType.NEAREST}, (False, True)),
    (24, 20, 16, 16, {"second_reader": True}, (False, True)),
    (24, 20, 6, 10, {}, (False, False)),                           # no whole vectors
])
def test_concat_with_neighbours(monkeypatch, storage, w, h, c_full, c_half, kw, joined):
    x = prng.uniform(5, (3, h, w), -1.0, 1.0)
    net = Join(storage, w, h, c_full, c_half, **kw)
    got = run(net, x)
    assert ("no launch of its own" in net.layers[3].kernelInfo()) == joined[0]
    if joined[1] is not None:
        assert ("no launch of its own" in net.layers[4].kernelInfo()) == joined[1]
    want = O.run_network(net.describe(), {net.input_key: x})[net.output_layer]
    net.cleanup()
    assert rel_l2(got, want) <= TOL[storage]
    monkeypatch.setenv("FYNHIP_NO_CONCAT_FUSION", "1")
    apart = Join(storage, w, h, c_full, c_half, **kw)
    again = run(apart, x)
    assert "no launch of its own" not in apart.layers[3].kernelInfo()
    apart.cleanup()
    assert rel_l2(got, again) <= (1e-6 if storage == fa.STORAGE_F32 else 5e-4)
