"""Host frames and results at the edges of the layout kernels and of the transfers' pieces (fyusenet/gpu/uploadlayer.cpp:92-186,
gpulayerbase.cpp:525-564): a copy layer hands back what was put in, through every host layout, into memory of the
library's and of the caller's own."""
import ctypes

import numpy as np
import pytest

import fyusenet_amd as fa
from fyusenet_amd import capi, prng, samples

STORAGES = pytest.mark.parametrize("storage", [fa.STORAGE_F32, fa.STORAGE_F16], ids=["f32", "f16"])


def _copy_net(c, h, w, storage, pad=0):
    class Net(fa.NeuralNetwork):
        def buildLayers(self, f):
            b = fa.ConcatLayerBuilder("copy").number(1).deep().input(c, 0).outputPadding(pad)
            b.size(w, h)
            b.outputChannels_ = c
            b.push(f)

        def connectLayers(self, layers, bm):
            pass

    net = Net(storage)
    net.setup()
    return net


@pytest.mark.gpu
@STORAGES
@pytest.mark.parametrize("c,h,w", [(1, 1, 1), (3, 1, 2), (3, 5, 7), (4, 1, 3), (2, 9, 4), (8, 33, 41), (70, 50, 61), (3, 701, 433), (4, 1201, 640), (260, 63, 65)])
def test_frames_come_back_as_they_went_in(c, h, w, storage):
    pad = 2
    net = _copy_net(c, h, w, storage, pad)
    lyr = net.layers[1]
    x = prng.uniform(500 + c * h, (c, h, w), -2.0, 2.0)
    want = x if storage == fa.STORAGE_F32 else x.astype(np.float16).astype(np.float32)
    orders = [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW]
    for order in orders:
        lyr.setInput(np.zeros_like(x), 0)
        lyr.setInput(x if order == fa.ORDER_CHANNELWISE else np.ascontiguousarray(x.transpose(1, 2, 0)), 0, order)
        net.forward()
        assert np.array_equal(net.getOutput(1), want), order
        own = np.full(x.shape, np.nan, np.float32)
        capi.check(capi.lib().fyn_net_get_output(net._h, 1, capi.fptr(own), fa.ORDER_CHANNELWISE))
        assert np.array_equal(own, want), order
    halo = lyr.copyResult(includePadding=True)
    assert np.array_equal(halo[:, pad:-pad, pad:-pad], want) and np.count_nonzero(halo) == np.count_nonzero(want)
    if c <= 4:
        pc = 4 if c == 3 else c
        own = np.full((h, w, pc), np.nan, np.float32)
        capi.check(capi.lib().fyn_net_get_output(net._h, 1, capi.fptr(own), fa.ORDER_GPU_SHALLOW))
        for got in (net.getOutput(1, fa.ORDER_GPU_SHALLOW), own):
            assert np.array_equal(got[..., :c].transpose(2, 0, 1), want) and not got[..., c:].any()
    net.cleanup()


@pytest.mark.gpu
@pytest.mark.parametrize("order", [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW], ids=["chw", "hwc"])
@pytest.mark.parametrize("width,height,depth", [(404, 300, 1), (404, 300, 2), (660, 500, 3)])
def test_overlapped_pipeline_matches_the_synchronous_path(width, height, depth, order):
    """Frames large enough for streams of their own: the upload of a frame runs beside the layers of the one before it,
    and its result leaves while the next is computed."""
    net = samples.StyleNetSample(3, width, height)
    net.setup()
    hwc = order == fa.ORDER_GPU_SHALLOW
    frames = [prng.uniform(3300 + i, (height, width, 3) if hwc else (3, height, width), 0.0, 1.0) for i in range(2 * depth + 3)]
    want = []
    for f in frames:
        net.layers[net.UPLOAD].setInput(f, 0, order)
        net.forward()
        want.append(net.getOutput(net.output_layer, order))
    assert not np.array_equal(want[0], want[1])
    net.asyncBegin(net.UPLOAD, net.output_layer, inOrder=order, outOrder=order, depth=depth)
    outs = [np.full_like(want[0], np.nan) for _ in frames]
    for i, (f, o) in enumerate(zip(frames, outs)):
        ticket = net.asyncSubmit(f, o)
        for k in range(i - depth + 1):
            assert np.array_equal(outs[k], want[k]), (i, k)
    net.asyncWait(ticket)
    for i in range(len(frames)):
        assert np.array_equal(outs[i], want[i]), i
    net.asyncEnd()
    net.cleanup()


@pytest.mark.gpu
@pytest.mark.parametrize("graph", [False, True], ids=["eager", "graph"])
@pytest.mark.parametrize("order", [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW], ids=["chw", "hwc"])
@pytest.mark.parametrize("depth", [1, 2, 4])
def test_overlapped_pipeline_computes_late_frames_again(monkeypatch, depth, order, graph):
    """Launches that give up at once on a frame that has not arrived (FYNHIP_FEED_GIVE_UP): every result is the frame's own."""
    monkeypatch.setenv("FYNHIP_FEED_GIVE_UP", "0")
    width, height = 660, 500
    net = samples.StyleNetSample(3, width, height)
    net.setup()
    net.useGraph(graph)
    hwc = order == fa.ORDER_GPU_SHALLOW
    frames = [prng.uniform(4100 + i, (height, width, 3) if hwc else (3, height, width), 0.0, 1.0) for i in range(3 * depth + 4)]
    want = []
    for f in frames:
        net.layers[net.UPLOAD].setInput(f, 0, order)
        net.forward()
        want.append(np.array(net.getOutput(net.output_layer, order)))
    for again in range(2):
        net.asyncBegin(net.UPLOAD, net.output_layer, inOrder=order, outOrder=order, depth=depth)
        outs = [np.full_like(want[0], np.nan) for _ in frames]
        tickets = [net.asyncSubmit(f, o) for f, o in zip(frames, outs)]
        if again:
            net.asyncEnd()
        else:
            for t, (got, w) in enumerate(zip(outs, want)):
                net.asyncWait(tickets[t])
                assert np.array_equal(got, w), t
            net.asyncEnd()
        for i, (got, w) in enumerate(zip(outs, want)):
            assert np.array_equal(got, w), (again, i)
    net.cleanup()


@pytest.mark.gpu
def test_results_belong_to_the_caller():
    """A result handed out stays what it was while later frames pass and after the network has gone; memory of results
    that nobody holds is used again."""
    net = _copy_net(4, 120, 160, fa.STORAGE_F32)
    kept = []
    for i in range(6):
        net.layers[1].setInput(np.full((4, 120, 160), i, np.float32), 0)
        net.forward()
        kept.append(net.getOutput(1))
    assert len({k.ctypes.data for k in kept}) == 6
    address = kept.pop(2).ctypes.data
    again = net.getOutput(1)
    assert again.ctypes.data == address and (again == 5).all()
    net.cleanup()
    for value, k in zip((0, 1, 3, 4, 5), kept):
        assert (k == value).all()

@pytest.mark.gpu
@STORAGES
@pytest.mark.parametrize("order", [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW], ids=["chw", "hwc"])
@pytest.mark.parametrize("c,h,w", [(1, 64, 300), (2, 63, 301), (3, 65, 302), (4, 66, 299)])
def test_results_at_any_place_of_a_block(c, h, w, order, storage):
    """A result that begins one, two or three floats into memory of the library's (fyn_host_acquire), with guards around it."""
    net = _copy_net(c, h, w, storage)
    x = prng.uniform(70 + c, (c, h, w), -2.0, 2.0)
    net.layers[1].setInput(x, 0)
    net.forward()
    want = x if storage == fa.STORAGE_F32 else x.astype(np.float16).astype(np.float32)
    pc = 4 if c == 3 else c
    n = h * w * (c if order == fa.ORDER_CHANNELWISE else pc)
    for offset in range(4):
        block = capi.result_array((n + 8,))
        assert type(block.base).__name__ == "_ResultBlock"
        block[:] = 77.0
        out = block[offset:offset + n]
        capi.check(capi.lib().fyn_net_get_output(net._h, 1, capi.fptr(out), order))
        got = out.reshape(c, h, w) if order == fa.ORDER_CHANNELWISE else out.reshape(h, w, pc)[..., :c].transpose(2, 0, 1)
        assert np.array_equal(got, want), offset
        assert (block[:offset] == 77.0).all() and (block[offset + n:] == 77.0).all(), offset
    net.cleanup()


@pytest.mark.gpu
@STORAGES
@pytest.mark.parametrize("order", [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW], ids=["chw", "hwc"])
@pytest.mark.parametrize("c,h,w", [(3, 5, 7), (3, 701, 433), (4, 1080, 1920)])
def test_a_frame_that_is_late_is_converted_again(monkeypatch, c, h, w, order, storage):
    """Launches that give up at the first pixel that is not there yet (FYNHIP_FEED_GIVE_UP, ticks; 4 s as a rule): the frame
    arrives all the same, every time."""
    monkeypatch.setenv("FYNHIP_FEED_GIVE_UP", "0")
    net = _copy_net(c, h, w, storage, 1)
    for i in range(6):
        x = prng.uniform(900 + i, (c, h, w), -2.0, 2.0)
        net.layers[1].setInput(x if order == fa.ORDER_CHANNELWISE else np.ascontiguousarray(x.transpose(1, 2, 0)), 0, order)
        net.forward()
        assert np.array_equal(net.getOutput(1), x if storage == fa.STORAGE_F32 else x.astype(np.float16).astype(np.float32)), i
    net.cleanup()


@pytest.mark.gpu
def test_a_late_frame_leaves_its_own_value_range(monkeypatch):
    """The value range that the first convolution scales by is the frame's, not that of what lay in the area before."""
    frames = [prng.uniform(40 + i, (3, 500, 660), 0.0, top) for i, top in enumerate((1.0, 1000.0, 1e-3, 1.0))]
    results = []
    for give_up in (None, "0"):
        if give_up is not None:
            monkeypatch.setenv("FYNHIP_FEED_GIVE_UP", give_up)
        net = samples.StyleNetSample(3, 660, 500)
        net.setup()
        got = []
        for f in frames:
            net.layers[net.UPLOAD].setInput(f, 0)
            net.forward()
            got.append(np.array(net.getOutput(net.output_layer)))
        net.cleanup()
        results.append(got)
    for i, (a, b) in enumerate(zip(*results)):
        assert np.array_equal(a, b), i
@pytest.mark.gpu
@STORAGES
@pytest.mark.parametrize("c,h,w", [(3, 303, 401), (3, 401, 302), (3, 16, 8191), (4, 257, 515), (2, 401, 501), (1, 701, 389)])
def test_overlapped_pipeline_on_odd_frames(c, h, w, storage):
    """The conversions between buffers in device memory: pixel counts that are no multiple of four, rows that end inside a
    thread's four pixels, every channel count of interleaved pixels; from both host layouts to both."""
    net = _copy_net(c, h, w, storage, pad=1)
    x = [prng.uniform(700 + i + c * w, (c, h, w), -2.0, 2.0) for i in range(3)]
    for in_order in (fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW):
        for out_order in (fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW):
            net.asyncBegin(1, 1, inOrder=in_order, outOrder=out_order, depth=2)
            pc = 4 if c == 3 else c
            outs = [np.full((c, h, w) if out_order == fa.ORDER_CHANNELWISE else (h, w, pc), np.nan, np.float32) for _ in x]
            for f, o in zip(x, outs):
                ticket = net.asyncSubmit(f if in_order == fa.ORDER_CHANNELWISE else np.ascontiguousarray(f.transpose(1, 2, 0)), o)
            net.asyncWait(ticket)
            net.asyncEnd()
            for f, o in zip(x, outs):
                want = f if storage == fa.STORAGE_F32 else f.astype(np.float16).astype(np.float32)
                if out_order == fa.ORDER_GPU_SHALLOW:
                    assert not o[..., c:].any()
                    o = o[..., :c].transpose(2, 0, 1)
                assert np.array_equal(o, want), (in_order, out_order)
    net.cleanup()


@pytest.mark.gpu
@pytest.mark.parametrize("order", [fa.ORDER_CHANNELWISE, fa.ORDER_GPU_SHALLOW], ids=["chw", "hwc"])
def test_page_locked_input_is_read_behind_the_default_stream(order):
    """A frame that the application's default stream is still writing into page-locked memory when it is handed over."""
    hip = ctypes.CDLL("libamdhip64.so")

    def call(name, *args):
        assert getattr(hip, name)(*args) == 0, name

    c, h, w = 3, 301, 500
    net = _copy_net(c, h, w, fa.STORAGE_F32)
    shape = (c, h, w) if order == fa.ORDER_CHANNELWISE else (h, w, c)
    nbytes, large = 4 * c * h * w, 1 << 30
    pinned, frame, a, b = (ctypes.c_void_p() for _ in range(4))
    call("hipHostMalloc", ctypes.byref(pinned), ctypes.c_size_t(nbytes), ctypes.c_uint(0))
    for p, n in ((frame, nbytes), (a, large), (b, large)):
        call("hipMalloc", ctypes.byref(p), ctypes.c_size_t(n))
    view = np.ctypeslib.as_array((ctypes.c_float * (c * h * w)).from_address(pinned.value)).reshape(shape)
    view[:] = 0
    for i in range(3):
        x = np.ascontiguousarray(prng.uniform(60 + i, shape, -2.0, 2.0))
        call("hipMemcpy", frame, x.ctypes.data_as(ctypes.c_void_p), ctypes.c_size_t(nbytes), ctypes.c_int(1))
        for _ in range(16):     # (milliseconds of work in front of the copy)
            call("hipMemcpyAsync", b, a, ctypes.c_size_t(large), ctypes.c_int(3), None)
        call("hipMemcpyAsync", pinned, frame, ctypes.c_size_t(nbytes), ctypes.c_int(2), None)
        net.layers[1].setInput(view, 0, order)
        net.forward()
        got = net.getOutput(1)
        assert np.array_equal(got, x if order == fa.ORDER_CHANNELWISE else x.transpose(2, 0, 1)), i
    net.cleanup()
    for p in (frame, a, b):
        call("hipFree", p)
    call("hipHostFree", pinned)


def _allocations(net):
    calls, nbytes = ctypes.c_size_t(0), ctypes.c_size_t(0)
    capi.check(capi.lib().fyn_net_device_allocations(net._h, ctypes.byref(calls), ctypes.byref(nbytes)))
    return calls.value, nbytes.value


@pytest.mark.gpu
@pytest.mark.parametrize("width,height,device_slots", [(64, 48, 0), (660, 500, 2)])
def test_allocations_count_every_area_in_use(width, height, device_slots):
    """The slots of a pipeline count when it is made, its frames do not; frames handed over one behind the other without
    waiting count up to four areas, frames one after the other a single one."""
    net = samples.StyleNetSample(3, width, height)
    net.setup()
    frame = prng.uniform(1, (3, height, width), 0.0, 1.0)
    result = np.empty((3, height, width), np.float32)
    begin = _allocations(net)
    for _ in range(5):
        net.layers[net.UPLOAD].setInput(frame, 0)
        net.forward()
        capi.check(capi.lib().fyn_net_get_output(net._h, net.output_layer, capi.fptr(result), fa.ORDER_CHANNELWISE))
    one = _allocations(net)
    assert one[0] - begin[0] == 2 and one[1] - begin[1] >= 2 * frame.nbytes   # (a frame in, a result out)
    for _ in range(12):
        net.layers[net.UPLOAD].setInput(frame, 0)
    net.finish()
    four = _allocations(net)
    assert four[0] - one[0] <= 3
    for again in range(2):
        before = _allocations(net)
        net.asyncBegin(net.UPLOAD, net.output_layer, depth=2)
        made = _allocations(net)
        assert made[0] - before[0] == 3 * ((0 if again else 2) + device_slots), again
        assert again or made[1] - before[1] >= 3 * 2 * frame.nbytes
        for _ in range(7):
            ticket = net.asyncSubmit(frame, result)
        net.asyncWait(ticket)
        assert _allocations(net) == made
        net.asyncEnd()
    net.cleanup()


def test_results_without_any_network_lie_in_ordinary_memory():
    capi.check(capi.lib().fyn_host_release(None))
    a = capi.result_array((64, 1024))
    a[:] = 1
    assert a.shape == (64, 1024) and a.dtype == np.float32
