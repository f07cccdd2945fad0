"""The device workspaces that calls keep for the next ones: several streams and threads, the bound and giving back."""
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
