"""Library-owned GEMM workspaces are per (device, stream): two streams in flight at once on one GPU each get their own
split-K partials and pre-pass buffers, so every result equals the same call made serially (the reference keeps these
buffers thread_local, src/kernels/gemm.cu:3258-3368). So do two host threads that call on one stream."""
import ctypes
import sys
import threading

import pytest
import torch

from qengine_amd import call, ops, synth
from test_gemm_gpu import SPLIT_SHAPE, setup

pytestmark = pytest.mark.gpu

KIND = {"split": 0, "i8": 1, "h16": 2}


def _run(path, w, x):
    if path == "i8":
        return ops.gemm_w4_i8(w, x, G=64)
    if path == "h16":
        return ops.gemm_w4h(w, x)
    return ops.gemm_w4_choice(w, x, cfg=0, ks=2)[0]


@pytest.mark.parametrize("path", ["i8", "h16", "split"])
def test_two_streams_keep_their_own_workspace(dev, path):
    n, k, t = SPLIT_SHAPE if path == "split" else (4096, 2048, 700)
    w, _, _ = setup(n, k, 1, seed=n + t)
    xs = [synth.to_dev(synth.x_host(t, k, seed=s)) for s in (1, 2)]
    want = [_run(path, w, x) for x in xs]  # serial, default stream
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:  # size each stream's buffers with an eager call before the overlapped ones
        with torch.cuda.stream(s):
            _run(path, w, xs[0])
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(8):  # the two streams' calls interleaved, nothing waits in between
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i].append(_run(path, w, xs[i]))
    torch.cuda.synchronize()
    iv = torch.int16 if want[0].dtype == torch.bfloat16 else torch.int32
    for i in range(2):
        for r, y in enumerate(got[i]):
            assert torch.equal(y.view(iv), want[i].view(iv)), (path, i, r)
    assert call("qe_workspace_count", KIND[path]) >= 3  # the default stream's and one per stream


# one case per buffer: the 9..16-row slice sums, the 33..64-row and 17..32-row tail parts, the split-K partials, the
# W4A8 and fp16 pre-pass buffers
PATHS = {"decode_12": (5120, 13824, 12), "decode_48": (5120, 3712, 48), "decode_24": (17408, 2560, 24),
         "prefill": (1040, 2176, 100), "i8": (1040, 2176, 100), "h16": (1040, 2176, 100)}
_MADE = {}


def _case(path):
    if path not in _MADE:
        n, k, m = PATHS[path]
        w, _, _ = setup(n, k, 1, seed=n + m)
        f = {"i8": lambda x, y=None: ops.gemm_w4_i8(w, x, G=64, y=y), "h16": lambda x, y=None: ops.gemm_w4h(w, x, y=y)}
        _MADE[path] = f.get(path, lambda x, y=None: ops.matmul_w4(w, x, y=y)), \
            [synth.to_dev(synth.x_host(m, k, seed=s)) for s in (1, 2)]
    return _MADE[path]


@pytest.mark.parametrize("path", list(PATHS))
def test_two_threads_on_one_stream(dev, path):
    """a call's launches stay together on the stream: no other thread's launch writes its buffer in between"""
    run, xs = _case(path)
    want = [run(x) for x in xs]
    torch.cuda.synchronize()
    got = [[torch.empty_like(want[i]) for _ in range(60)] for i in range(2)]
    gate = threading.Barrier(2)

    def calls(i):
        gate.wait()
        for y in got[i]:
            run(xs[i], y)

    threads = [threading.Thread(target=calls, args=(i,)) for i in range(2)]
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1e-6)
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    finally:
        sys.setswitchinterval(interval)
    torch.cuda.synchronize()
    for i in range(2):
        for r, y in enumerate(got[i]):
            assert torch.equal(y, want[i]), (path, i, r)


@pytest.mark.parametrize("path", list(PATHS))
def test_two_streams_in_flight(dev, path):
    """calls of two streams interleaved, nothing waits in between: each the bits of the serial call"""
    run, xs = _case(path)
    want = [run(x) for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    got = [[torch.empty_like(want[i]) for _ in range(20)] for i in range(2)]
    for r in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                run(xs[i], got[i][r])
    torch.cuda.synchronize()
    for i in range(2):
        for r, y in enumerate(got[i]):
            assert torch.equal(y, want[i]), (path, i, r)


def _graph(run, x, y, stream):
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=stream):
        run(x, y)
    return g


@pytest.mark.parametrize("path", list(PATHS))
def test_two_graphs_of_one_stream_replayed_at_once(dev, path):
    """a graph's calls use buffers of the graph's own: two captured on one stream and replayed on two, beside eager calls
    on the stream of the capture, nothing waiting in between, all give the eager bits"""
    run, xs = _case(path)
    want = [run(x) for x in xs]
    cap = torch.cuda.Stream()
    cap.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(cap):
        run(xs[0])  # (the split and the pre-passes need their stream sized before a capture)
    outs = [torch.empty_like(want[i]) for i in range(2)]
    graphs = [_graph(run, xs[i], outs[i], cap) for i in range(2)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    got, eager = [[], []], []
    for _ in range(20):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                graphs[i].replay()
                got[i].append(outs[i].clone())
        with torch.cuda.stream(cap):
            eager.append(run(xs[1]))
    torch.cuda.synchronize()
    for r in range(20):
        assert torch.equal(eager[r], want[1]), (path, r)
        for i in range(2):
            assert torch.equal(got[i][r], want[i]), (path, i, r)


@pytest.mark.parametrize("path,kind", [("decode_12", 4), ("decode_48", 3), ("decode_24", 3)])
def test_decode_captured_without_preparation(dev, path, kind):
    """decode under capture on a stream that never ran it: the kernels of the eager call, hence its bits; the graph's
    buffer goes back with the graph and serves the next one"""
    run, xs = _case(path)
    want = run(xs[0])
    y = torch.empty_like(want)
    torch.cuda.synchronize()
    counts = []
    for _ in range(3):
        before = call("qe_workspace_count", kind)
        g = _graph(run, xs[0], y, torch.cuda.Stream())
        counts.append(call("qe_workspace_count", kind) - before)
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want), path
        g.reset()
        del g
        torch.cuda.synchronize()
        counts.append(call("qe_workspace_count", kind) - before)
    assert counts == [1, 0] * 3, counts


def _fresh_stream():
    """a non-blocking stream that no call was made on (torch hands out 32 of its own in turn)"""
    hip = ctypes.CDLL("libamdhip64.so")
    raw = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(raw), 1) == 0
    return torch.cuda.ExternalStream(raw.value)


@pytest.mark.parametrize("G", [32, 64, 128])
def test_w4a8_captured_after_its_reserve(dev, G):
    """qe_gemm_i8_reserve_s is all that a W4A8 capture needs: the split of the eager call, hence its bits"""
    n, k, t = 1040, 2176, 100
    w, _, _ = setup(n, k, 1, seed=n + t)
    x = synth.to_dev(synth.x_host(t, k, seed=1))
    want = ops.gemm_w4_i8(w, x, G=G)
    call("qe_gemm_set_sk_maxparts", 1)
    try:
        unsplit = ops.gemm_w4_i8(w, x, G=G)
    finally:
        call("qe_gemm_set_sk_maxparts", 0)
    assert not torch.equal(unsplit, want)  # (the eager call splits)
    st = _fresh_stream()
    call("qe_gemm_i8_reserve_s", k, t, ctypes.c_void_p(st.cuda_stream))
    y = torch.empty_like(want)
    g = _graph(lambda a, b: ops.gemm_w4_i8(w, a, G=G, y=b), x, y, st)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("path", list(PATHS))
def test_first_call_beside_a_capture(dev, path):
    """a stream's first call, which allocates its buffer, while another thread captures in the default (global) mode: both
    give the eager bits"""
    run, xs = _case(path)
    want = [run(x) for x in xs]
    y, z = torch.empty_like(want[0]), torch.empty_like(want[1])
    fresh = _fresh_stream()
    failed = []

    def first_call():
        try:
            with torch.cuda.stream(fresh):
                run(xs[1], z)
        except Exception as e:  # noqa: BLE001  (reported by the main thread, whose capture has to end first)
            failed.append(e)

    cap = torch.cuda.Stream()
    with torch.cuda.stream(cap):
        run(xs[0], y)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=cap):
        t = threading.Thread(target=first_call)
        t.start()
        t.join()
        run(xs[0], y)
    torch.cuda.synchronize()
    assert not failed, failed
    assert torch.equal(z, want[1]), path
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[0]), path
