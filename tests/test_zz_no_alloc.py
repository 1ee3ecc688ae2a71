"""jepa_amd_preprocess_frames_device_noalloc (no counterpart in the reference: preprocessing for callers
that cannot allocate device memory) against jepa_amd_preprocess_frames_device or the host function, bit for bit,
on two calls in a row with the second input smaller than the first, on a caller's stream (a torch stream of its own,
not the null stream) and on the null stream; the call captured into a HIP graph and replayed on new frames; and the
refusal of an input whose scratch would exceed the static array, before any device work. Both ways through it: the
tile kernel, one launch without tables or scratch, and the two kernels of large reductions, whose tables and
horizontal-pass image live in the static array."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _params(jlib, resize_short=256, crop=256, resample=0):
    p = jlib.PreprocessParams()
    for c, (m, sd) in enumerate(zip((0.485, 0.456, 0.406), (0.229, 0.224, 0.225))):
        p.mean[c], p.std[c] = m, sd
    p.resize_short, p.crop, p.resample, p.resize_mode, p.rescale, p.fused_norm = resize_short, crop, resample, 0, 1.0 / 255.0, True
    return p


def _run(jlib, fn, p, frames_dev, T, h, w, n_out, stream=None):
    out = torch.full((n_out,), float("nan"), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    oh, ow = C.c_int(0), C.c_int(0)
    args = [0, C.byref(p), frames_dev.data_ptr(), T, h, w, out.data_ptr(), out.numel(), C.byref(oh), C.byref(ow)]
    if fn == "jepa_amd_preprocess_frames_device_noalloc":
        args.append(stream)
    rc = getattr(jlib.lib(), fn)(*args)
    assert rc == 0, jlib.error_text()
    torch.cuda.synchronize()
    return out.cpu().numpy(), (oh.value, ow.value)


@pytest.mark.parametrize("use_own_stream", [True, False])
def test_noalloc_equals_allocating_entry_point(jlib, use_own_stream):
    rng = np.random.default_rng(7)
    side = torch.cuda.Stream() if use_own_stream else None
    stream = side.cuda_stream if use_own_stream else None
    if use_own_stream:
        assert stream, "a torch side stream must not be the null stream"
    # first a larger input, then a smaller one (both through the tile kernel)
    for (T, h, w, resample) in [(4, 720, 1280, 1), (2, 300, 400, 0)]:
        frames = torch.from_numpy(rng.integers(0, 256, (T, h, w, 3), dtype=np.uint8)).cuda()
        p = _params(jlib, resample=resample)
        n_out = 3 * T * 256 * 256
        want, shape_a = _run(jlib, "jepa_amd_preprocess_frames_device", p, frames, T, h, w, n_out)
        got, shape_b = _run(jlib, "jepa_amd_preprocess_frames_device_noalloc", p, frames, T, h, w, n_out, stream)
        assert shape_a == shape_b == (256, 256)
        assert np.isfinite(want).all()
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


def test_noalloc_graph_capture_and_replay(jlib):
    """The call (the tile kernel) captured on a side stream into a HIP graph (there is no host copy and no stream
    synchronisation to break the capture), then replayed three times on new frames written into the same input buffer between replays, each
    replay bit for bit against the allocating entry point on those frames."""
    rng = np.random.default_rng(11)
    T, h, w = 3, 480, 640
    p = _params(jlib, resample=1)
    n_out = 3 * T * 256 * 256
    frames = torch.from_numpy(rng.integers(0, 256, (T, h, w, 3), dtype=np.uint8)).cuda()
    out = torch.full((n_out,), float("nan"), dtype=torch.float32, device="cuda")
    side = torch.cuda.Stream()
    oh, ow = C.c_int(0), C.c_int(0)
    fn = jlib.lib().jepa_amd_preprocess_frames_device_noalloc
    args = lambda st: [0, C.byref(p), frames.data_ptr(), T, h, w, out.data_ptr(), out.numel(), C.byref(oh), C.byref(ow), st]
    torch.cuda.synchronize()
    # one eager call first: the per-device scratch address is looked up outside the capture
    with torch.cuda.stream(side):
        assert fn(*args(side.cuda_stream)) == 0, jlib.error_text()
    side.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        rc = fn(*args(side.cuda_stream))
    assert rc == 0, jlib.error_text()
    for rep in range(3):
        new = rng.integers(0, 256, (T, h, w, 3), dtype=np.uint8)
        frames.copy_(torch.from_numpy(new).cuda())
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        want, _ = _run(jlib, "jepa_amd_preprocess_frames_device", p, frames, T, h, w, n_out)
        assert np.isfinite(want).all()
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32), err_msg=f"replay {rep}")
    del g


# reductions by about 30 with the wide filter: more LDS than a tile may have
UNTILED = [(4, 900, 1000, 30, 32), (2, 700, 640, 24, 24)]


def _captured(jlib, p, frames, T, h, w, out, side):
    """The call captured on stream `side`: the graph, and how many nodes it has."""
    L = jlib.lib()
    g, n = C.c_void_p(), C.c_size_t(0)
    assert L.hipStreamBeginCapture(C.c_void_p(side.cuda_stream), 1) == 0     # thread-local
    rc = L.jepa_amd_preprocess_frames_device_noalloc(0, C.byref(p), frames.data_ptr(), T, h, w, out.data_ptr(), out.numel(), None, None, side.cuda_stream)
    assert L.hipStreamEndCapture(C.c_void_p(side.cuda_stream), C.byref(g)) == 0
    assert rc == 0, jlib.error_text()
    assert L.hipGraphGetNodes(g, None, C.byref(n)) == 0
    return g, n.value


@pytest.mark.parametrize("use_own_stream", [True, False])
def test_noalloc_two_kernels_share_the_scratch(jlib, use_own_stream):
    """A larger input, then a smaller one, through the two kernels: the second call must not see the first one's tables
    or image in the static array."""
    rng = np.random.default_rng(17)
    side = torch.cuda.Stream() if use_own_stream else None
    for T, h, w, short, crop in UNTILED + UNTILED[:1]:
        u8 = rng.integers(0, 256, (T, h, w, 3), dtype=np.uint8)
        p = _params(jlib, short, crop, 1)
        got, shape = _run(jlib, "jepa_amd_preprocess_frames_device_noalloc", p, torch.from_numpy(u8).cuda(), T, h, w, 3 * T * crop * crop,
                          side.cuda_stream if side else None)
        want = jlib.preprocess_frames(p, list(u8)).reshape(-1)
        assert shape == (crop, crop)
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


def test_noalloc_two_kernels_capture_and_replay(jlib):
    """The two kernels captured: their tables travel as kernel arguments, so the graph holds them, and a call of another
    geometry between replays, which writes the same static array, does not change a replay. The capture has several
    nodes; the tile kernel's has one."""
    rng = np.random.default_rng(19)
    L = jlib.lib()
    side = torch.cuda.Stream()
    T, h, w, short, crop = UNTILED[0]
    p = _params(jlib, short, crop, 1)
    frames = torch.zeros((T, h, w, 3), dtype=torch.uint8, device="cuda")
    out = torch.zeros(3 * T * crop * crop, device="cuda")
    _run(jlib, "jepa_amd_preprocess_frames_device_noalloc", p, frames, T, h, w, out.numel(), side.cuda_stream)
    g, nodes = _captured(jlib, p, frames, T, h, w, out, side)
    assert nodes >= 3
    exe = C.c_void_p()
    assert L.hipGraphInstantiate(C.byref(exe), g, None, None, C.c_size_t(0)) == 0
    T2, h2, w2, short2, crop2 = UNTILED[1]
    other = torch.from_numpy(rng.integers(0, 256, (T2, h2, w2, 3), dtype=np.uint8)).cuda()
    for rep in range(3):
        u8 = rng.integers(0, 256, (T, h, w, 3), dtype=np.uint8)
        frames.copy_(torch.from_numpy(u8).cuda())
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        assert L.hipGraphLaunch(exe, C.c_void_p(side.cuda_stream)) == 0
        side.synchronize()
        want = jlib.preprocess_frames(p, list(u8)).reshape(-1)
        np.testing.assert_array_equal(out.cpu().numpy().view(np.uint32), want.view(np.uint32), err_msg=f"replay {rep}")
        _run(jlib, "jepa_amd_preprocess_frames_device_noalloc", _params(jlib, short2, crop2, 1), other, T2, h2, w2, 3 * T2 * crop2 * crop2, None)
    assert L.hipGraphExecDestroy(exe) == 0 and L.hipGraphDestroy(g) == 0
    small = torch.zeros((2, 300, 400, 3), dtype=torch.uint8, device="cuda")
    out2 = torch.zeros(3 * 2 * 256 * 256, device="cuda")
    torch.cuda.synchronize()
    g, nodes = _captured(jlib, _params(jlib), small, 2, 300, 400, out2, side)
    assert nodes == 1
    assert L.hipGraphDestroy(g) == 0


def test_noalloc_refuses_oversized_scratch(jlib):
    # 64 frames of 1080 x 1920 cropped to 256: the two kernels' horizontal pass alone is 64 * 1080 * 256 * 3
    # bytes, over the 32 MiB static array; refused on the host, before any device work, also where, as here, the tile
    # kernel would not need it (the limit is the entry point's contract)
    # (the buffers have the sizes the call describes, so nothing could go out of bounds either way)
    p = _params(jlib)
    frames = torch.zeros((64, 1080, 1920, 3), dtype=torch.uint8, device="cuda")
    out = torch.zeros(3 * 64 * 256 * 256, dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    jlib.lib().jepa_error_reset()
    rc = jlib.lib().jepa_amd_preprocess_frames_device_noalloc(0, C.byref(p), frames.data_ptr(), 64, 1080, 1920, out.data_ptr(),
                                                             out.numel(), None, None, None)
    assert rc == -1
    assert "scratch" in jlib.error_text()
