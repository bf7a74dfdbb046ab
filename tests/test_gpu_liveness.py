"""Layers computed inside a neighbour's launch in networks whose branches interleave: a launch that writes a later layer's
tensor early, beside one that reads an earlier layer's input late, where both tensors would share a buffer.  Every result
equals the oracle's, and that of the network with every layer in a launch of its own.  Tolerances: rel-L2 <= 1e-4 (fp32
storage), <= 2e-3 (fp16 storage)."""
import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import networks, prng
from oracle import oracle as O
from util import rel_l2

pytestmark = pytest.mark.gpu
TOL = {fa.STORAGE_F32: 1e-4, fa.STORAGE_F16: 2e-3}
A = fa.ActType
W, H = 24, 20


class Branches(networks._StreamNet):
    """Two branches over one frame; `kind` names the layer whose input is read late.  The other branch is a 1x1 layer and the
    depthwise (or arg-max) layer behind it, which the 1x1 layer's launch computes."""
    config_id = 10
    input_key = (0, 0)

    def __init__(self, storage, kind):
        super().__init__(storage)
        self.kind = kind

    def scale(self, no, c, src):
        up = fa.ScaleLayerBuilder("scale%d" % no).number(no).shape(c, H // 2, W // 2, c).scale(2.0).scaleType(fa.ScalingType.LINEAR).prefixAct(A.RELU)
        self._add(up.deep())
        self._edges.append((src, no, 0))

    def concat(self, no, parts):
        cat = fa.ConcatLayerBuilder("cat%d" % no).number(no).deep()
        for port, (src, c) in enumerate(parts):
            cat.input(c, 0)
            self._edges.append((src, no, port))
        cat.size(W, H)
        cat.outputChannels_ = sum(c for _, c in parts)
        self._add(cat)

    def batchnorm(self, no, c, h, w, src, act):
        b = fa.GPULayerBuilder("bn%d" % no).type(fa.LayerType.BATCHNORM).number(no).shape(c, h, w, c).prefixAct(act).deep()
        seed = self._next_seed()
        self._add(b, lambda: np.concatenate([prng.uniform(seed, (c,), 0.5, 1.5), prng.normal(seed + 1, (c,), 0.0, 0.1)]))
        self._edges.append((src, no, 0))

    def define(self):
        h, w = H // 2, W // 2
        self._add(fa.UpDownLayerBuilder(fa.UpDownLayerBuilder.UPLOAD, "upload").number(0).shape(3, H, W, 3).outputPadding(1))
        if self.kind == "scale":           # layer 2's tensor: read by 9 instead of 7, its buffer written by 8 instead of 10
            self.conv(1, "base", 3, 3, 16, H, W, 0, stride=2)
            self.conv(2, "x", 1, 16, 32, h, w, 1)
            self.conv(3, "full", 3, 3, 16, H, W, 0)
            self.scale(7, 32, 2)
            self.conv(8, "expand", 1, 16, 32, h, w, 1, pad_out=1)
            self.concat(9, [(7, 32), (3, 16)])
            self.conv(10, "dw", 3, 32, 32, h, w, 8, groups=32)
            self.conv(11, "a", 1, 32, 16, h, w, 10)
            self.conv(12, "b", 1, 48, 16, H, W, 9)
        elif self.kind == "concat":        # layer 1's: read by 9 (the batch-norm layer's launch) instead of 4, written by 5 instead of 10
            self.conv(1, "x", 3, 3, 32, H, W, 0)
            self.conv(2, "y", 3, 3, 16, H, W, 0)
            self.conv(3, "base", 1, 16, 16, H, W, 2)
            self.concat(4, [(1, 32), (2, 16)])
            self.conv(5, "expand", 1, 16, 32, H, W, 3, pad_out=1)
            self.batchnorm(9, 48, H, W, 4, A.RELU)
            self.conv(10, "dw", 3, 32, 32, H, W, 5, groups=32)
            self.conv(11, "a", 1, 32, 16, H, W, 10)
            self.conv(12, "b", 1, 48, 16, H, W, 9)
        elif self.kind == "argmax":        # layer 2's: read by 9 instead of 7, written by 8 (for the arg-max layer) instead of 10
            self.conv(1, "base", 3, 3, 16, H, W, 0, stride=2)
            self.conv(2, "x", 1, 16, 4, h, w, 1)
            self.conv(3, "full", 3, 3, 12, H, W, 0)
            self.scale(7, 4, 2)
            self.conv(8, "classes", 1, 16, 16, h, w, 1)
            self.concat(9, [(7, 4), (3, 12)])
            self._add(fa.ArgMaxLayerBuilder("best").number(10).shape(2, h, w, 16).deep())
            self._edges.append((8, 10, 0))
            self.conv(11, "a", 1, 2, 8, h, w, 10)
            self.conv(12, "b", 1, 16, 16, H, W, 9)
        elif self.kind == "depthwise":     # layer 2's: read by 9 instead of 5, written by 7 instead of 10
            self.conv(1, "base", 3, 3, 16, H, W, 0)
            self.conv(2, "x", 1, 16, 32, H, W, 1, stride=2, pad_out=1)
            self.conv(5, "dw1", 3, 32, 32, h, w, 2, groups=32)
            self.conv(7, "expand", 1, 16, 32, H, W, 1, pad_out=1)
            self.conv(9, "project", 1, 32, 16, h, w, 5)
            self.conv(10, "dw", 3, 32, 32, H, W, 7, stride=2, pad_out=1, groups=32)
            self.conv(11, "a", 3, 32, 16, h, w, 10)
            self.conv(12, "b", 1, 16, 16, h, w, 9)
        else:                              # layer 2's: read by 9 instead of 5, written by 7 instead of 10
            self.conv(1, "base", 3, 3, 16, H, W, 0)
            self.conv(2, "x", 1, 16, 32, H, W, 1)
            self.batchnorm(5, 32, H, W, 2, A.NONE)
            self.conv(7, "expand", 1, 16, 32, H, W, 1, pad_out=1)
            self.conv(9, "reader", 1, 32, 16, H, W, 5, act=A.RELU)
            self.conv(10, "dw", 3, 32, 32, H, W, 7, groups=32)
            self.conv(11, "a", 1, 32, 16, H, W, 10)
            self.conv(12, "b", 1, 16, 16, H, W, 9)

    def setInput(self, x):
        self.layers[0].setInput(x, 0)


def run(net, x):
    net.setup()
    for _ in range(2):
        net.setInput(x)
        net.forward()
        net.finish()
    return net.getOutput(11), net.getOutput(12)


def joined(net, layer):
    return "no launch of its own" in net.layers[layer].kernelInfo()


# (kind, the layer that may be computed by the launch in front of it, the layer whose work would move behind that launch)
@pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])
@pytest.mark.parametrize("kind,early,late", [("scale", 10, 7), ("concat", 10, 4), ("argmax", 10, 7), ("depthwise", 10, 5), ("batchnorm", 10, 5)])
def test_interleaved_branches(monkeypatch, kind, early, late, storage):
    monkeypatch.setenv("FYNHIP_FORCE_DW_FUSION", "1")
    monkeypatch.setenv("FYNHIP_FORCE_S16_CONV" if kind == "argmax" else "FYNHIP_FORCE_KR16_CONV", "1")
    x = prng.uniform(7, (3, H, W), -1.0, 1.0)
    net = Branches(storage, kind)
    got = run(net, x)
    print(kind, storage, [(b.number_, net.layers[b.number_].kernelInfo()) for b in net._builders], flush=True)
    one = joined(net, early), joined(net, late)
    net.cleanup()
    want = O.run_network(net.describe(), {net.input_key: x})
    for g, layer in zip(got, (11, 12)):
        if (kind, layer) != ("argmax", 11):     # (near ties: below, against the same scores)
            assert rel_l2(g, want[layer]) <= TOL[storage], layer
    assert one[0] != one[1]                     # (one of the two is joined, and not both)
    for switch in ("FYNHIP_NO_DW_FUSION", "FYNHIP_NO_CONCAT_FUSION", "FYNHIP_NO_ARGMAX_FUSION", "FYNHIP_NO_BN_FUSION"):
        monkeypatch.setenv(switch, "1")
    apart = Branches(storage, kind)
    again = run(apart, x)
    assert not joined(apart, early) and not joined(apart, late)
    apart.cleanup()
    for g, a in zip(got, again):
        assert rel_l2(g, a) <= (1e-5 if storage == fa.STORAGE_F32 else 1e-3)
