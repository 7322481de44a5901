"""The filters' fast forms against the float64 oracle where they can go wrong: the direct Gaussian's
32 x 32 tiles (sizes about their edges, one row or column past them, radii from 3 to the largest,
36), the box path that keeps no image (long frames, a last box of one pixel, radii past the frame),
CLAHE's tables by a wave (levels below, at and above 64), and a pixel that is not finite."""
import numpy as np
import pytest

from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _raw(n, h, w, seed):
    rng = np.random.default_rng(seed)
    r, c = np.meshgrid(np.arange(h), np.arange(w), indexing="ij")
    hump = 300 * np.exp(-((r - 0.4 * h) ** 2 + (c - 0.6 * w) ** 2) / (2 * (0.5 * w) ** 2))
    return np.maximum(hump + 200 + 60 * np.cos(0.3 * r + 0.2 * c) + rng.normal(0, 8, (n, h, w)), 0).astype(np.float32)


def _call(raw, mask, forced_global=False, **kw):
    import torch
    from zebsdsolve_amd import _native as nat, engine
    lib = nat.load()
    n, h, w = raw.shape
    o = nat.PrepOpts()
    for k, v in kw.items():
        setattr(o, k, v)
    kind = {"float32": 2, "uint16": 1, "uint8": 0}[raw.dtype.name]
    dev = torch.from_numpy(raw.astype(np.int32) if kind == 1 else raw).cuda()
    dev = dev.to(torch.uint16) if kind == 1 else dev
    out = torch.full((n, h, w), float("nan"), device="cuda")
    m = (nat.ctypes.c_float * 3)(*[float(x) for x in mask])
    prev = lib.zb_knob_set(b"prep_global", int(forced_global))
    try:
        need = int(lib.zb_prep_workspace(n, h, w, nat.ctypes.byref(o)))
        ws = torch.empty((max(need, 8),), dtype=torch.uint8, device="cuda")
        nat.check(lib.zb_prep_work(dev.data_ptr(), kind, n, h, w, m, nat.ctypes.byref(o), ws.data_ptr(), ws.numel(), out.data_ptr(),
                                   engine.stream_ptr()), "prep")
        return out.cpu().numpy()
    finally:
        lib.zb_knob_set(b"prep_global", prev)


@pytest.mark.parametrize("forced_global", [False, True])
@pytest.mark.parametrize("h,w,sigma", [(2, 2, 1.0), (5, 7, 2.3), (31, 33, 0.7), (32, 32, 11.9), (33, 65, 9.0), (64, 64, 11.99), (65, 40, 4.0),
                                       (97, 96, 8.0), (129, 128, 11.0), (60, 60, 9.0), (160, 141, 6.0)])
def test_direct_gaussian_about_the_tiles_edges(h, w, sigma, forced_global):
    from oracle import pipeline as op
    print(f"direct {h}x{w} sigma {sigma} global {forced_global}", flush=True)
    raw = _raw(3, h, w, h * 1000 + w)
    mask = op.frame(np.eye(3), h, w)["mask"]
    got = _call(raw, mask, forced_global, dynamic=1, dynamic_sigma=sigma)
    for b in range(3):
        ref = op.prep(raw[b], mask, dynamic="subtract", dynamic_sigma=sigma / w)
        # float32 sums of up to 73 x 2 taps of values to 560 and their difference with the pixel, which
        # is a hundredth of them where the frame is nearly flat: 2e-5 of the largest value, 1e-4 for the
        # frames of a few pixels (a difference of 1 in 500)
        err = np.abs(got[b] - ref).max() / np.abs(ref).max()
        assert err < (2e-5 if h * w > 64 else 1e-4), (b, err)


@pytest.mark.parametrize("h,w,sigma,dtype", [(81, 83, 12.45, np.float32), (80, 80, 12.0, np.uint8), (24, 200, 30.0, np.uint16), (145, 97, 14.55, np.float32),
                                             (128, 129, 18.0, np.uint16), (301, 203, 30.5, np.uint16), (40, 40, 60.0, np.float32)])
def test_boxes_without_the_image(h, w, sigma, dtype):
    from oracle import pipeline as op
    print(f"boxes {h}x{w} sigma {sigma} {np.dtype(dtype).name}", flush=True)
    raw = _raw(3, h, w, h * 1000 + w)
    raw = (raw / 4 if dtype == np.uint8 else raw).astype(dtype)
    mask = op.frame(np.eye(3), h, w)["mask"]
    for dyn, name in ((1, "subtract"), (2, "divide")):
        got = _call(raw, mask, dynamic=dyn, dynamic_sigma=sigma)
        for b in range(3):
            ref = op.prep(raw[b], mask, dynamic=name, dynamic_sigma=sigma / w)
            err = np.abs(got[b] - ref).max() / np.abs(ref).max()
            assert err < 2e-5, (name, b, err)


@pytest.mark.parametrize("forced_global", [False, True])
@pytest.mark.parametrize("bins,grid", [(16, 3), (64, 4), (65, 5), (256, 8)])
def test_clahe_tables_by_a_wave(bins, grid, forced_global):
    from oracle import pipeline as op
    print(f"clahe bins {bins} grid {grid} global {forced_global}", flush=True)
    raw = _raw(3, 61, 75, bins)
    mask = op.frame(np.eye(3), 61, 75)["mask"]
    got = _call(raw, mask, forced_global, clahe=1, clahe_grid=grid, clahe_bins=bins, clahe_clip=2.5)
    for b in range(3):
        ref = op.prep(raw[b], mask, clahe_opts=(grid, bins, 2.5))
        # a pixel on a level's edge may count to either level: 1 of a tile's pixels, on few pixels
        err = np.abs(got[b] - ref) / np.abs(ref).max()
        assert np.median(err) < 2e-5 and (err > 2e-4).mean() < 0.02, (b, np.median(err), (err > 2e-4).mean())


@pytest.mark.parametrize("value", [np.nan, np.inf, 3e38])
def test_a_pixel_that_is_not_finite_stays_within_its_radius(value):
    """A corner's dead pixel farther than the taps reach from the mask changes nothing under it."""
    print(f"dead pixel {value}", flush=True)
    raw = _raw(2, 60, 60, 3)
    mask = (29.5, 29.5, 12.0 ** 2)
    clean = _call(raw, mask, dynamic=1, dynamic_sigma=3.0)
    raw[:, 0, 0] = value
    got = _call(raw, mask, dynamic=1, dynamic_sigma=3.0)
    r, c = np.meshgrid(np.arange(60.0), np.arange(60.0), indexing="ij")
    inside = (r - mask[0]) ** 2 + (c - mask[1]) ** 2 <= mask[2]
    assert np.isfinite(got[:, inside]).all()
    assert np.abs(got - clean)[:, inside].max() < 2e-5 * np.abs(clean).max()
