"""The tiled rasterisation (LDS accumulators per box of the volume, each box visited by the slices whose plane
crosses it, one device-wide atomic flush per work item).

It takes launches into a cubic volume with FP32 values and weights, Mat33<f32> or
Quaternion<f32> rotations, Mat22 inverse scalings or none, no Ewald curvature and cutoff <= 0.5; NOA_HIP_RASTERIZE_LAYOUT=direct selects the other path. Bars: rel-L2 1e-6 of values and weights
against the oracle (noa's per-pixel scatter; the sums are regrouped, by LDS and device atomics in both paths) and
against the one-lane-per-pixel kernel.
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle as O
from helpers import random_rotations, random_spectrum, rel_l2

pytestmark = pytest.mark.gpu

DEV = "cuda"


def nx():
    import noa_amd.xform as m
    return m


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def axis_poses():
    m = nx()
    poses = [np.eye(3)]
    for fn in (m.rotate_z, m.rotate_y, m.rotate_x):
        for deg in (90, 180, 270):
            poses.append(fn(np.deg2rad(deg)))
    return np.round(np.stack(poses)).astype(np.float32)


def gpu(layout, monkeypatch, remap, sl, w, b, n, rot, out_dtype=torch.complex64, wvol=True, cutoff=0.5, start=None,
        wstart=None):
    monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", layout)
    wr = n // 2 + 1
    vol = dev(start) if start is not None else torch.zeros((1, n, n, wr), dtype=out_dtype, device=DEV)
    wv = None
    if wvol:
        wv = dev(wstart) if wstart is not None else torch.zeros((1, n, n, wr), dtype=torch.float32, device=DEV)
    opts = nx().RasterizeCentralSlicesOptions(fftfreq_cutoff=cutoff)
    nx().rasterize_central_slices_3d(remap, sl, w, (b, 1, n, n), vol, wv, (1, n, n, n), None, rot, opts)
    torch.cuda.synchronize()
    return vol.cpu().numpy(), (wv.cpu().numpy() if wvol else None)


def oracle(remap, sl, w, b, n, rot, out_dtype=np.complex64, wvol=True, cutoff=0.5, start=None, wstart=None):
    wr = n // 2 + 1
    vol = start.copy() if start is not None else np.zeros((1, n, n, wr), out_dtype)
    wv = None
    if wvol:
        wv = wstart.copy() if wstart is not None else np.zeros((1, n, n, wr), np.float32)
    O.rasterize_central_slices_3d(remap, sl, w, (b, 1, n, n), vol, wv, (1, n, n, n), None, rot,
                                  fftfreq_cutoff=cutoff, n_threads=8)
    return vol, wv


@pytest.mark.parametrize("remap,n,b,cutoff", [
    ("h2h", 64, 300, 0.5),
    ("hc2hc", 64, 300, 0.5),
    ("hc2h", 33, 120, 0.5),        # odd size
    ("h2hc", 48, 200, 0.31),       # smaller cutoff
    ("hc2hc", 128, 96, 0.5),
])
def test_tiles_match_the_oracle_and_the_direct_kernel(monkeypatch, remap, n, b, cutoff):
    print(f"case rasterize tiles {remap} n={n} b={b} cutoff={cutoff}", flush=True)
    rng = np.random.default_rng(1700 + n)
    sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
    w = rng.uniform(0.1, 1.0, (b, 1, n, n // 2 + 1)).astype(np.float32)
    rot = random_rotations(b, rng)
    rot[: len(axis_poses())] = axis_poses()     # taps exactly on lattice points, tile faces and the x = 0 plane
    want_v, want_w = oracle(remap, sl, w, b, n, rot, cutoff=cutoff)
    got_v, got_w = gpu("tiles", monkeypatch, remap, dev(sl), dev(w), b, n, dev(rot), cutoff=cutoff)
    assert rel_l2(got_v, want_v) < 1e-6
    assert rel_l2(got_w, want_w) < 1e-6
    ref_v, ref_w = gpu("direct", monkeypatch, remap, dev(sl), dev(w), b, n, dev(rot), cutoff=cutoff)
    assert rel_l2(got_v, ref_v) < 1e-6
    assert rel_l2(got_w, ref_w) < 1e-6


def test_tiles_axis_poses_per_voxel(monkeypatch):
    """Axis poses only: every pixel lands on a lattice point (fraction 0), so each voxel receives whole values and
    the x = 0 duplicates carry the conjugate; checked per voxel, where a misplaced tap cannot hide in a norm."""
    print("case rasterize tiles axis poses", flush=True)
    rng = np.random.default_rng(1710)
    n = 32
    rot = np.concatenate([axis_poses()] * 7)                  # 70 slices: the tiled path by default
    b = rot.shape[0]
    sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
    w = rng.uniform(0.1, 1.0, (b, 1, n, n // 2 + 1)).astype(np.float32)
    for remap in ("h2h", "hc2hc"):
        want_v, want_w = oracle(remap, sl, w, b, n, rot)
        got_v, got_w = gpu("tiles", monkeypatch, remap, dev(sl), dev(w), b, n, dev(rot))
        np.testing.assert_allclose(got_v, want_v, rtol=0, atol=2e-6 * np.abs(want_v).max())
        np.testing.assert_allclose(got_w, want_w, rtol=0, atol=2e-6 * np.abs(want_w).max())


@pytest.mark.parametrize("kind", ["real", "c2r", "value", "no_weights", "weight_value"])
def test_tiles_value_types_and_weights(monkeypatch, kind):
    print(f"case rasterize tiles {kind}", flush=True)
    rng = np.random.default_rng(1720)
    n, b = 48, 128
    rot = random_rotations(b, rng)
    spec = random_spectrum((b, 1, n, n // 2 + 1), rng)
    wts = rng.uniform(0.1, 1.0, (b, 1, n, n // 2 + 1)).astype(np.float32)
    out_np, out_t, wvol = np.complex64, torch.complex64, True
    sl_np, sl_dev, w_np, w_dev = spec, dev(spec), wts, dev(wts)
    if kind == "real":
        sl_np = rng.standard_normal((b, 1, n, n // 2 + 1)).astype(np.float32)
        sl_dev, out_np, out_t = dev(sl_np), np.float32, torch.float32
    elif kind == "c2r":
        out_np, out_t = np.float32, torch.float32
    elif kind == "value":
        sl_np = sl_dev = 2.5
        out_np, out_t = np.float32, torch.float32
    elif kind == "no_weights":
        w_np = w_dev = None
        wvol = False
    elif kind == "weight_value":
        w_np = w_dev = 0.75
    want_v, want_w = oracle("hc2hc", sl_np, w_np, b, n, rot, out_dtype=out_np, wvol=wvol)
    got_v, got_w = gpu("tiles", monkeypatch, "hc2hc", sl_dev, w_dev, b, n, dev(rot), out_dtype=out_t, wvol=wvol)
    assert rel_l2(got_v, want_v) < 1e-6
    if wvol:
        assert rel_l2(got_w, want_w) < 1e-6


def test_tiles_strided_slices_accumulate_and_keep_voxels_beyond_the_cutoff(monkeypatch):
    """Slices cut from wider rows, a volume that already holds values (rasterisation adds to it), and voxels that no
    tap reaches keep their value."""
    print("case rasterize tiles strided/accumulate", flush=True)
    rng = np.random.default_rng(1730)
    n, b = 64, 150
    wide = random_spectrum((b, 1, n, n // 2 + 7), rng)
    sl = wide[..., : n // 2 + 1]
    rot = random_rotations(b, rng)
    start = random_spectrum((1, n, n, n // 2 + 1), rng)
    wstart = rng.uniform(0, 1, (1, n, n, n // 2 + 1)).astype(np.float32)
    want_v, want_w = oracle("h2h", sl, None, b, n, rot, cutoff=0.4, start=start, wstart=wstart)
    gs = torch.from_numpy(wide).to(DEV)[..., : n // 2 + 1]
    got_v, got_w = gpu("tiles", monkeypatch, "h2h", gs, None, b, n, dev(rot), cutoff=0.4, start=start, wstart=wstart)
    assert rel_l2(got_v, want_v) < 1e-6
    assert rel_l2(got_w, want_w) < 1e-6
    untouched = (want_v == start) & (want_w == wstart)
    np.testing.assert_array_equal(got_v[untouched], start[untouched])


def test_tiles_with_a_degenerate_transform(monkeypatch):
    """A singular matrix collapses the plane: every pixel of that slice is a candidate of every tile, and each is
    still rasterised once."""
    print("case rasterize tiles degenerate transform", flush=True)
    rng = np.random.default_rng(1740)
    n, b = 32, 70
    sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
    rot = random_rotations(b, rng)
    rot[3] = np.array([[0.3, 0.5, 0.5], [0.1, 0.5, 0.5], [0.2, -0.5, -0.5]], np.float32)
    rot[5] = np.zeros((3, 3), np.float32)
    want_v, want_w = oracle("h2h", sl, None, b, n, rot)
    got_v, got_w = gpu("tiles", monkeypatch, "h2h", dev(sl), None, b, n, dev(rot))
    assert rel_l2(got_v, want_v) < 1e-6
    assert rel_l2(got_w, want_w) < 1e-6


def test_default_selection_by_slice_count(monkeypatch):
    """Without the switch, calls of at most 16 slices with fewer than 2^14 pixels take the direct kernel and larger ones the
    boxes; on both sides of the line (7 slices of 64^2 have 14,784 pixels, 8 have 16,896) and well above it."""
    print("case rasterize default selection", flush=True)
    monkeypatch.delenv("NOA_HIP_RASTERIZE_LAYOUT", raising=False)
    rng = np.random.default_rng(1750)
    n = 64
    for b in (7, 8, 17, 64):
        sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
        rot = random_rotations(b, rng)
        vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        nx().rasterize_central_slices_3d("hc2hc", dev(sl), None, (b, 1, n, n), vol, None, (1, n, n, n), None, dev(rot))
        torch.cuda.synchronize()
        want, _ = oracle("hc2hc", sl, None, b, n, rot, wvol=False)
        assert rel_l2(vol.cpu().numpy(), want) < 1e-6


@pytest.mark.parametrize("remap,n,b", [("h2h", 64, 200), ("hc2hc", 48, 96)])
def test_tiles_take_quaternions(monkeypatch, remap, n, b):
    """Quaternion<f32> rotations on the tiled path (the plane geometry from their matrix, noa's quaternion rotation
    per pixel): against the oracle with the same quaternions and against the direct kernel, rel-L2 1e-6."""
    print(f"case rasterize tiles quaternions {remap} n={n} b={b}", flush=True)
    rng = np.random.default_rng(1800 + n)
    sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
    w = rng.uniform(0.1, 1.0, (b, 1, n, n // 2 + 1)).astype(np.float32)
    rot = random_rotations(b, rng)
    rot[: len(axis_poses())] = axis_poses()
    q = nx().quaternion_from_matrix(rot.astype(np.float64)).astype(np.float32)
    want_v = np.zeros((1, n, n, n // 2 + 1), np.complex64)
    want_w = np.zeros((1, n, n, n // 2 + 1), np.float32)
    O.rasterize_central_slices_3d(remap, sl, w, (b, 1, n, n), want_v, want_w, (1, n, n, n), None, q, quaternion=True,
                                  n_threads=8)
    got_v, got_w = gpu("tiles", monkeypatch, remap, dev(sl), dev(w), b, n, nx().Quaternions(dev(q)))
    dir_v, dir_w = gpu("direct", monkeypatch, remap, dev(sl), dev(w), b, n, nx().Quaternions(dev(q)))
    assert rel_l2(got_v, want_v) < 1e-6 and rel_l2(got_w, want_w) < 1e-6
    assert rel_l2(got_v, dir_v) < 1e-6 and rel_l2(got_w, dir_w) < 1e-6


def _scalings(b, rng):
    """Anisotropic inverse scalings (magnification 0.9-1.1 along a random in-plane axis): R(t) diag(s) R(-t)."""
    t = rng.uniform(0, np.pi, b)
    s = rng.uniform(0.9, 1.1, (b, 2))
    c, d = np.cos(t), np.sin(t)
    rt = np.stack([np.stack([c, -d], -1), np.stack([d, c], -1)], -2)
    return np.ascontiguousarray(rt @ (s[:, :, None] * np.transpose(rt, (0, 2, 1)))).astype(np.float32)


@pytest.mark.parametrize("remap,n,b,quat", [("h2h", 64, 200, False), ("hc2hc", 48, 96, False), ("h2h", 64, 120, True)])
def test_tiles_take_inverse_scalings(monkeypatch, remap, n, b, quat):
    """Mat22 inverse scalings on the tiled path (the plane's pixel columns scaled, noa's general expression per
    pixel without Ewald curvature): against the oracle with the same scalings and against the direct kernel,
    rel-L2 1e-6."""
    print(f"case rasterize tiles scalings {remap} n={n} b={b} quat={quat}", flush=True)
    rng = np.random.default_rng(1900 + n + b)
    sl = random_spectrum((b, 1, n, n // 2 + 1), rng)
    w = rng.uniform(0.1, 1.0, (b, 1, n, n // 2 + 1)).astype(np.float32)
    rot = random_rotations(b, rng)
    rot[: len(axis_poses())] = axis_poses()
    scale = _scalings(b, rng)
    if quat:
        rot = nx().quaternion_from_matrix(rot.astype(np.float64)).astype(np.float32)
    want_v = np.zeros((1, n, n, n // 2 + 1), np.complex64)
    want_w = np.zeros((1, n, n, n // 2 + 1), np.float32)
    O.rasterize_central_slices_3d(remap, sl, w, (b, 1, n, n), want_v, want_w, (1, n, n, n), scale, rot,
                                  quaternion=quat, n_threads=8)
    got, direct = {}, {}
    for layout, out in (("tiles", got), ("direct", direct)):
        monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", layout)
        vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        wv = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=DEV)
        r = nx().Quaternions(dev(rot)) if quat else dev(rot)
        nx().rasterize_central_slices_3d(remap, dev(sl), dev(w), (b, 1, n, n), vol, wv, (1, n, n, n), dev(scale), r,
                                         nx().RasterizeCentralSlicesOptions())
        torch.cuda.synchronize()
        out["v"], out["w"] = vol.cpu().numpy(), wv.cpu().numpy()
    assert np.abs(want_v).max() > 0
    assert rel_l2(got["v"], want_v) < 1e-6 and rel_l2(got["w"], want_w) < 1e-6
    assert rel_l2(got["v"], direct["v"]) < 1e-6 and rel_l2(got["w"], direct["w"]) < 1e-6


def _tilt_series(b, rng):
    tilt = np.deg2rad(np.linspace(-60, 60, b))
    return np.stack([nx().rotate_z(0.4) @ nx().rotate_y(t) for t in tilt]).astype(np.float32)


@pytest.mark.parametrize("n,b,kind,per_item", [
    (16, 1, "plain", None),         # the smallest size; fewer positions than a box
    (17, 64, "plain", 3),           # the most slices without the items kernel
    (40, 65, "quat", 2),            # the fewest with it
    (41, 257, "scaled", 5),         # one slice past a scan of the items kernel
    (24, 5, "strided", None),       # real slices with a pitch and a batch gap
    (64, 300, "tilt", 7),           # boxes on the tilt axis: every slice, many items
    (766, 1, "plain", None),        # the largest size
])
def test_boxes_match_the_oracle(monkeypatch, n, b, kind, per_item):
    """Every pixel is rasterised once whatever the split into items: against the oracle, rel-L2 1e-6 (sums of at most a
    few hundred FP32 terms in another order: 2^-24 times the square root of their number, about 1e-6 at the worst)."""
    print(f"case rasterize boxes n={n} b={b} {kind} per_item={per_item}", flush=True)
    rng = np.random.default_rng(2000 + n + b)
    monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", "tiles")      # also the calls that the default leaves to a lane per pixel
    if per_item is not None:
        monkeypatch.setenv("NOA_HIP_RASTERIZE_PAIRS", str(per_item))
    wr = n // 2 + 1
    real = kind == "strided"
    sl = random_spectrum((b, 1, n, wr), rng)
    sl = sl.real.copy() if real else sl
    w = rng.uniform(0.1, 1.0, (b, 1, n, wr)).astype(np.float32)
    rot = _tilt_series(b, rng) if kind == "tilt" else random_rotations(b, rng)
    scale = _scalings(b, rng) if kind == "scaled" else None
    if kind == "quat":
        rot = nx().quaternion_from_matrix(rot.astype(np.float64)).astype(np.float32)
    gsl = dev(sl)
    if real:
        room = torch.zeros((b, 2, n, wr + 3), dtype=torch.float32, device=DEV)
        room[:, :1, :, :wr] = gsl
        gsl = room[:, :1, :, :wr]
    gw, grot = dev(w), (nx().Quaternions(dev(rot)) if kind == "quat" else nx().Mat33Array(dev(rot), DEV))
    vol = torch.zeros((1, n, n, wr), dtype=gsl.dtype, device=DEV)
    wv = torch.zeros((1, n, n, wr), dtype=torch.float32, device=DEV)

    def call():
        vol.zero_()
        wv.zero_()
        nx().rasterize_central_slices_3d("h2h", gsl, gw, (b, 1, n, n), vol, wv, (1, n, n, n),
                                         None if scale is None else dev(scale), grot)

    if n > 300:     # the lane-per-pixel kernel, itself checked against the oracle at the sizes above
        monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", "direct")
        call()
        want_v, want_w = vol.clone(), wv.clone()
        monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", "tiles")
    else:
        want_v, want_w = np.zeros((1, n, n, wr), sl.dtype), np.zeros((1, n, n, wr), np.float32)
        O.rasterize_central_slices_3d("h2h", sl, w, (b, 1, n, n), want_v, want_w, (1, n, n, n), scale, rot,
                                      quaternion=kind == "quat", n_threads=8)
        want_v, want_w = dev(want_v), dev(want_w)

    def check():
        for got, want in ((vol, want_v), (wv, want_w)):
            assert float(torch.linalg.vector_norm(got - want) / torch.linalg.vector_norm(want)) < 1e-6

    call()
    check()
    if scale is None and kind != "quat":         # captured: nothing is allocated, the items scan for their slices
        stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call()
        for _ in range(3):
            vol.fill_(1)
            graph.replay()
            check()


@pytest.mark.parametrize("b", [7, 100])
def test_first_call_of_a_size_can_be_captured(b, monkeypatch):
    """A size and cutoff that no call had before, in a graph: the boxes are not resident and nothing may be uploaded
    then, so the lane-per-pixel kernel serves the call. Replays against an eager call, rel-L2 1e-6 (other sums)."""
    print(f"case rasterize first call captured b={b}", flush=True)
    monkeypatch.delenv("NOA_HIP_RASTERIZE_LAYOUT", raising=False)
    n, cutoff = 44, 0.40625 + 0.0001 * b
    rng = np.random.default_rng(b)
    sl, rot = dev(random_spectrum((b, 1, n, n // 2 + 1), rng)), nx().Mat33Array(random_rotations(b, rng), DEV)
    vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
    wv = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=DEV)
    opts = nx().RasterizeCentralSlicesOptions(fftfreq_cutoff=cutoff)

    def call():
        vol.zero_()
        wv.zero_()
        nx().rasterize_central_slices_3d("h2h", sl, None, (b, 1, n, n), vol, wv, (1, n, n, n), None, rot, opts)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    call()
    torch.cuda.synchronize()
    want_v, want_w = vol.cpu().numpy(), wv.cpu().numpy()
    for _ in range(3):
        vol.fill_(1)
        graph.replay()
        torch.cuda.synchronize()
        assert rel_l2(vol.cpu().numpy(), want_v) < 1e-6 and rel_l2(wv.cpu().numpy(), want_w) < 1e-6


@pytest.mark.parametrize("n,length,ratio", [(512, 100.0, 1e3), (512, 100.0, 1.5e3), (700, 20.0, 1.5e3), (512, 9.0, 900.0),
                                            (512, 1.0, 900.0), (512, 0.5, 5e3)])
def test_boxes_find_the_pixels_of_sheared_scalings(monkeypatch, n, length, ratio):
    """Inverse scalings that make a slice's axes nearly parallel and long: the plane's normal and the coordinates round in
    proportion, and no pixel may fall between the boxes. Against the lane-per-pixel kernel; the voxels around the origin
    sum some 10,000 terms in another order, which 1e-5 rel-L2 holds (2^-24 times the square root of their number)."""
    print(f"case rasterize sheared scalings n={n} {length} {ratio}", flush=True)
    rng = np.random.default_rng(int(ratio))
    b = 20
    turn = lambda t: np.stack([np.stack([np.cos(t), -np.sin(t)], -1), np.stack([np.sin(t), np.cos(t)], -1)], -2)
    scale = turn(rng.uniform(0, np.pi, b)) @ np.diag([length, length / ratio]) @ turn(rng.uniform(0, np.pi, b))
    scale = dev(scale.astype(np.float32))
    sl, rot = dev(random_spectrum((b, 1, n, n // 2 + 1), rng)), nx().Mat33Array(dev(random_rotations(b, rng)), DEV)
    got = {}
    for layout in ("direct", "tiles"):
        monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", layout)
        vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        wv = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=DEV)
        nx().rasterize_central_slices_3d("h2h", sl, None, (b, 1, n, n), vol, wv, (1, n, n, n), scale, rot)
        torch.cuda.synchronize()
        got[layout] = vol, wv
    for a, want in zip(got["tiles"], got["direct"]):
        assert float(torch.linalg.vector_norm(a - want) / torch.linalg.vector_norm(want)) < 1e-5


def test_boxes_keep_what_is_not_a_number(monkeypatch):
    """A matrix of no numbers gives voxels that are not numbers, the same ones with both kernels, and no others."""
    print("case rasterize non-finite matrix", flush=True)
    n, b = 64, 20
    rng = np.random.default_rng(3)
    sl, m = dev(random_spectrum((b, 1, n, n // 2 + 1), rng)), random_rotations(b, rng)
    m[7] = np.nan
    rot, got = nx().Mat33Array(dev(m), DEV), {}
    for layout in ("direct", "tiles"):
        monkeypatch.setenv("NOA_HIP_RASTERIZE_LAYOUT", layout)
        vol = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.complex64, device=DEV)
        wv = torch.zeros((1, n, n, n // 2 + 1), dtype=torch.float32, device=DEV)
        nx().rasterize_central_slices_3d("h2h", sl, None, (b, 1, n, n), vol, wv, (1, n, n, n), None, rot)
        torch.cuda.synchronize()
        got[layout] = vol, wv
    assert bool(torch.isnan(got["direct"][1]).any())
    for a, want in zip(got["tiles"], got["direct"]):
        a, want = (torch.view_as_real(t) if t.is_complex() else t for t in (a, want))
        assert torch.equal(torch.isnan(a), torch.isnan(want))
        a, want = torch.nan_to_num(a), torch.nan_to_num(want)
        assert float(torch.linalg.vector_norm(a - want) / torch.linalg.vector_norm(want)) < 1e-6
