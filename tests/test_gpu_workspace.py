"""The device workspaces that calls keep for the next ones: several streams and threads, the bound and giving back."""
import ctypes
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from helpers import random_rotations, random_spectrum

pytestmark = pytest.mark.gpu

DEV = "cuda"


def nx():
    import noa_amd.xform as m
    return m


def _call(n, b, volume, rot, out):
    nx().extract_central_slices_3d("h2h", volume, None, (1, n, n, n), out, None, (b, 1, n, n), None, rot)


@pytest.mark.parametrize("n,b", [(32, 200), (96, 400)])
def test_streams_and_threads_do_not_share_a_workspace_in_use(n, b):
    """Each thread extracts from its own volume on its own stream (every call copies the volume into a workspace); every
    result is the one of the call made alone."""
    print(f"case workspace threads n={n}", flush=True)
    rng = np.random.default_rng(7)
    rot = nx().Mat33Array(random_rotations(b, rng), DEV)
    jobs = []
    for _ in range(3):
        volume = torch.from_numpy(random_spectrum((1, n, n, n // 2 + 1), rng)).to(DEV)
        want = torch.empty((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        _call(n, b, volume, rot, want)
        jobs.append((volume, want))
    torch.cuda.synchronize()
    failed = []

    def work(volume, want):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                out = torch.zeros_like(want)
                _call(n, b, volume, rot, out)
                if not torch.equal(torch.view_as_real(out), torch.view_as_real(want)):
                    failed.append(1)
        stream.synchronize()

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed


def test_threads_on_one_stream_do_not_share_a_workspace_in_use():
    """Two threads enqueue on the same stream: their calls take turns there, each with its own workspace while its call
    is being enqueued; every result is the one of the call made alone."""
    print("case workspace threads on one stream", flush=True)
    rng = np.random.default_rng(9)
    n, b = 64, 300
    rot = nx().Mat33Array(random_rotations(b, rng), DEV)
    jobs = []
    for _ in range(2):
        volume = torch.from_numpy(random_spectrum((1, n, n, n // 2 + 1), rng)).to(DEV)
        want = torch.empty((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        _call(n, b, volume, rot, want)
        jobs.append((volume, want, [torch.empty_like(want) for _ in range(20)]))
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()

    def work(volume, _, outs):
        with torch.cuda.stream(stream):
            for out in outs:
                _call(n, b, volume, rot, out)

    threads = [threading.Thread(target=work, args=j) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    stream.synchronize()
    for _, want, outs in jobs:
        assert all(torch.equal(torch.view_as_real(out), torch.view_as_real(want)) for out in outs)


def test_a_destroyed_stream_leaves_its_workspaces_usable():
    """A workspace outlives the stream it was last used on: a new stream, which may have the old one's handle, takes it
    or another one, and trimming gives all of them back."""
    print("case workspace destroyed stream", flush=True)
    rng = np.random.default_rng(10)
    n, b = 64, 300
    hip = ctypes.CDLL("libamdhip64.so")
    volume = torch.from_numpy(random_spectrum((1, n, n, n // 2 + 1), rng)).to(DEV)
    rot = nx().Mat33Array(random_rotations(b, rng), DEV)
    want = torch.empty((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
    _call(n, b, volume, rot, want)
    out = torch.empty_like(want)
    for _ in range(3):
        handle = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
        out.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
            _call(n, b, volume, rot, out)
        torch.cuda.synchronize()
        assert hip.hipStreamDestroy(handle) == 0
        assert torch.equal(torch.view_as_real(out), torch.view_as_real(want))
    assert nx().workspace_trim() > 0


def _cycles(seconds):
    """Cycles that keep a stream busy for about `seconds`."""
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    torch.cuda._sleep(1000)
    begin.record()
    torch.cuda._sleep(1000000)
    end.record()
    end.synchronize()
    return int(1e6 * 1e3 * seconds / begin.elapsed_time(end))


def _independent_streams(cycles):
    """Two streams on different hardware queues: work on the second ends while the first is busy."""
    first = torch.cuda.Stream()
    probe, x = torch.cuda.Event(), torch.zeros(16, device=DEV)
    for second in [torch.cuda.Stream() for _ in range(4)]:
        if second == first:
            continue
        torch.cuda.synchronize()
        with torch.cuda.stream(first):
            torch.cuda._sleep(cycles)
            probe.record()
        with torch.cuda.stream(second):
            x.add_(1)
        second.synchronize()
        if not probe.query():
            torch.cuda.synchronize()
            return first, second
    pytest.skip("no two streams that run side by side")


def test_a_full_store_does_not_order_streams(monkeypatch):
    """Two streams whose workspaces (block copies of a 512^3 volume, 553 MB each) exceed the bound together: the second
    one's call neither waits on the host nor on the GPU for the first one's, which still has its workspace in use; once
    it has ended, its workspace makes room. Results as alone, and never more than the bound is kept."""
    print("case workspace bound", flush=True)
    n, b, limit = 512, 4, 1 << 30
    monkeypatch.setenv("NOA_HIP_EXTRACT_LAYOUT", "bricks")
    volume = torch.view_as_complex(torch.randn((1, n, n, n // 2 + 1, 2), device=DEV))
    rot = nx().Mat33Array(random_rotations(b, np.random.default_rng(11)), DEV)
    want, out_a, out_b = (torch.zeros((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=DEV) for _ in range(3))
    nx().workspace_trim()
    _call(n, b, volume, rot, want)
    torch.cuda.synchronize()
    assert 0 < 2 * nx().workspace_trim() - limit < limit
    cycles = _cycles(0.5)
    first, second = _independent_streams(cycles // 10)
    ended = torch.cuda.Event()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(cycles)
        _call(n, b, volume, rot, out_a)
        ended.record()
    with torch.cuda.stream(second):
        _call(n, b, volume, rot, out_b)
    host_free = not ended.query()
    second.synchronize()
    gpu_free = not ended.query()
    torch.cuda.synchronize()
    assert host_free and gpu_free
    assert torch.equal(torch.view_as_real(out_a), torch.view_as_real(want))
    assert torch.equal(torch.view_as_real(out_b), torch.view_as_real(want))
    out_b.zero_()
    with torch.cuda.stream(second):
        _call(n, b, volume, rot, out_b)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(out_b), torch.view_as_real(want))
    kept = nx().workspace_trim()
    assert 0 < kept <= limit
    assert nx().workspace_trim() == 0


def test_trim_gives_the_workspaces_back():
    print("case workspace trim", flush=True)
    rng = np.random.default_rng(8)
    n, b = 64, 300
    volume = torch.from_numpy(random_spectrum((1, n, n, n // 2 + 1), rng)).to(DEV)
    rot = nx().Mat33Array(random_rotations(b, rng), DEV)
    first, second = (torch.empty((b, 1, n, n // 2 + 1), dtype=torch.complex64, device=DEV) for _ in range(2))
    _call(n, b, volume, rot, first)
    assert 0 < nx().workspace_trim() <= 1 << 30
    assert nx().workspace_trim() == 0
    _call(n, b, volume, rot, second)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(first), torch.view_as_real(second))
