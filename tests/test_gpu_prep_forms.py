"""The filters' forms give the same bits: whatever the alignment of the workspace, the kernel that a size and a
chain of filters take, and the switches that force another."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.test_gpu_prep_tiles import _raw

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

CHAINS = {"direct": dict(dynamic=1, dynamic_sigma=4.0), "boxes": dict(dynamic=1, dynamic_sigma=14.5), "divided boxes": dict(dynamic=2, dynamic_sigma=12.5),
          "clahe": dict(clahe=1, clahe_grid=4, clahe_bins=64, clahe_clip=2.0),
          "all": dict(dynamic=2, dynamic_sigma=9.3, clahe=1, clahe_grid=3, clahe_bins=65, clahe_clip=2.5, bandpass=1, bp_fine=1.5, bp_coarse=6.0),
          "all by boxes": dict(dynamic=2, dynamic_sigma=13.0, clahe=1, clahe_grid=5, clahe_bins=32, clahe_clip=1.5, bandpass=1, bp_fine=12.0, bp_coarse=16.0),
          "band pass": dict(bandpass=1, bp_fine=0.0, bp_coarse=13.0)}


def _call(raw, chain, shift=0, background=False, **knobs):
    """The patterns through zb_prep_work, the workspace `shift` bytes past 256, with the knobs set; and the
    workspace's bytes that the call wrote."""
    import torch
    from zebsdsolve_amd import _native as nat, engine
    lib = nat.load()
    n, h, w = raw.shape
    o = nat.PrepOpts()
    for k, v in CHAINS[chain].items():
        setattr(o, k, v)
    kind = {"float32": 2, "uint16": 1, "uint8": 0}[raw.dtype.name]
    dev = torch.from_numpy(raw.view(np.int16) if kind == 1 else raw).cuda()
    bg = torch.from_numpy(raw.astype(np.float64).mean(0).astype(np.float32)).cuda()
    o.background = bg.data_ptr() if background else None
    out = torch.full((n, h, w), float("nan"), device="cuda")
    m = (nat.ctypes.c_float * 3)((h - 1) / 2, (w - 1) / 2, (min(h, w) / 2) ** 2)
    before = {k: lib.zb_knob_set(k.encode(), v) for k, v in knobs.items()}
    assert min(before.values(), default=0) >= 0
    try:
        need = int(lib.zb_prep_workspace(n, h, w, nat.ctypes.byref(o)))
        ws = torch.full((max(need, 8) + shift,), 171, dtype=torch.uint8, device="cuda")
        nat.check(lib.zb_prep_work(dev.data_ptr(), kind, n, h, w, m, nat.ctypes.byref(o), ws.data_ptr() + shift, ws.numel() - shift, out.data_ptr(),
                                   engine.stream_ptr()), "prep")
        return out.cpu().numpy(), int((ws != 171).sum())
    finally:
        for k, v in before.items():
            lib.zb_knob_set(k.encode(), v)


@pytest.mark.parametrize("chain", ["direct", "all", "all by boxes"])
@pytest.mark.parametrize("h,w", [(60, 60), (44, 64), (120, 120)])
def test_a_workspace_of_eight_bytes_alignment(chain, h, w):
    print(f"prep workspace alignment {chain} {h}x{w}", flush=True)
    raw = _raw(5, h, w, h + w)
    want, _ = _call(raw, chain, 0, prep_global=1)
    for shift in (8, 16, 24):
        got, wrote = _call(raw, chain, shift, prep_global=1)
        assert wrote > 0 and np.array_equal(got, want), shift


@pytest.mark.parametrize("chain", list(CHAINS))
@pytest.mark.parametrize("h,w,dtype", [(60, 60, np.uint8), (75, 83, np.float32), (120, 120, np.uint16)])
def test_prep_global_goes_through_global_memory(chain, h, w, dtype):
    """With the knob prep_global every chain's image lies in the workspace, and every pixel is the same."""
    print(f"prep forced global {chain} {h}x{w} {np.dtype(dtype).name}", flush=True)
    raw = _raw(5, h, w, h + w)
    raw = (raw / 4 if dtype == np.uint8 else raw).astype(dtype)
    want, _ = _call(raw, chain, background=True, prep_global=0)
    got, wrote = _call(raw, chain, background=True, prep_global=1)
    assert wrote > 0
    assert np.array_equal(got, want)


SIZES = [(2, 2), (5, 7), (8, 64), (31, 33), (32, 32), (33, 65), (44, 64), (60, 60), (64, 48), (75, 83), (97, 96), (120, 120), (129, 128), (240, 320)]


@pytest.mark.parametrize("chain", list(CHAINS))
@pytest.mark.parametrize("forced", [0, 1])
def test_the_fast_forms_give_the_general_kernels_bits(chain, forced):
    """Every pixel of k_prep_tiles and k_prep_box is that of k_prep and k_prep_g: their sums run in the same order."""
    for k, (h, w) in enumerate(SIZES):
        dtype = (np.uint8, np.uint16, np.float32)[k % 3]
        print(f"prep forms {chain} {h}x{w} {np.dtype(dtype).name} global {forced}", flush=True)
        raw = _raw(4, h, w, 100 * h + w)
        raw = (raw / 4 if dtype == np.uint8 else raw).astype(dtype)
        for background in (False, True):
            want, _ = _call(raw, chain, background=background, prep_global=forced, prep_loops=1)
            got, _ = _call(raw, chain, background=background, prep_global=forced)
            assert np.isfinite(want).all()
            assert np.array_equal(got, want), (h, w, background, np.abs(got - want).max())


@pytest.mark.parametrize("sigma", [0.3, 0.7, 2.0, 5.5, 9.0, 11.99, 12.0, 17.3, 30.5, 60.0])
@pytest.mark.parametrize("dynamic", [1, 2])
def test_every_deviation_gives_the_general_kernels_bits(sigma, dynamic, monkeypatch):
    monkeypatch.setitem(CHAINS, "one", dict(dynamic=dynamic, dynamic_sigma=sigma))
    for h, w in ((40, 40), (61, 90), (128, 129)):
        print(f"prep forms sigma {sigma} dynamic {dynamic} {h}x{w}", flush=True)
        raw = _raw(4, h, w, h * w)
        want, _ = _call(raw, "one", prep_loops=1)
        got, _ = _call(raw, "one")
        assert np.array_equal(got, want), (h, w, np.abs(got - want).max())


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, 3e38, 1e-42, -0.0])
@pytest.mark.parametrize("chain", list(CHAINS))
def test_odd_pixels_give_the_general_kernels_bits(value, chain):
    print(f"prep forms {chain} a pixel of {value}", flush=True)
    raw = _raw(3, 60, 60, 9)
    raw[0, 0, 0] = raw[1, 30, 31] = raw[2, 59, 59] = value
    want, _ = _call(raw, chain, prep_loops=1)
    got, _ = _call(raw, chain)
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("chain", ["none", "clahe", "one tap", "boxes"])
@pytest.mark.parametrize("n", [3, 513])
def test_either_side_of_the_general_kernels_sizes(chain, n, monkeypatch):
    """The pixels do not depend on the kernel that the size, the taps and the count choose: sizes about each line."""
    monkeypatch.setitem(CHAINS, "none", {})
    monkeypatch.setitem(CHAINS, "one tap", dict(dynamic=1, dynamic_sigma=0.5))
    sizes = {"none": [(48, 48), (48, 49), (49, 49), (64, 64), (64, 65), (100, 102), (101, 102), (230, 200)], "clahe": [(64, 64), (64, 65), (101, 101), (102, 102)],
             "one tap": [(42, 42), (43, 43), (44, 44)], "boxes": [(18, 18), (19, 19), (26, 26), (27, 27)]}[chain]
    for h, w in sizes:
        print(f"prep lines {chain} {h}x{w} n {n}", flush=True)
        raw = np.repeat(_raw(3, h, w, h + w), n // 3, 0).astype(np.uint8)
        want, _ = _call(raw, chain, background=True, prep_loops=1)
        got, _ = _call(raw, chain, background=True)
        assert np.array_equal(got, want)
