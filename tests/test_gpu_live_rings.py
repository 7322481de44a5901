"""Ring pairs without a sample in the window are left out by the sphere stage: the coefficients do not
depend on how many pairs a block takes (one pair, where every empty one is left out, to all of them,
where none is), bit for bit; agree with the float64 oracle where most pairs are empty; and an empty
window's are zeros. Ring lengths below and above a wave, past 128 pairs, FP32 and 16-bit products."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

H, W = 44, 60


def _coefficients(L, n, radius, flags, group=0, centre=None):
    """(coefficients [n, pairs] complex, stats, patterns, frame dict) of n random patterns under a mask."""
    import torch
    from zebsdsolve_amd import _native as nat, engine
    from zebsdsolve_amd.geometry import Geometry
    lib = nat.load()
    e = engine.Engine()
    e.settings.apply(bandwidth=min(L, 64))
    e.geo = Geometry(pc=cases.PC, sample_tilt_deg=70.0)
    e.set_patterns(np.zeros((1, 1, H, W), np.float32))
    band, fr = e.band(L), e.frame()
    c = centre or ((H - 1) / 2, (W - 1) / 2)
    fr.mask[0], fr.mask[1], fr.mask[2] = c[0], c[1], radius * radius
    gen = torch.Generator(device="cuda")
    gen.manual_seed(L)
    pats = torch.rand((n, H, W), generator=gen, device="cuda") - 0.3
    t = e.positions(np.zeros(n, np.int64)).astype(np.float32)
    items = np.concatenate([t, np.arange(n, dtype=np.float32)[:, None]], 1)
    items[:, :3] += np.random.default_rng(L).uniform(-1, 1, (n, 3)).astype(np.float32)
    d_items = torch.from_numpy(items).cuda()
    alm = torch.full((n, band.host.pairs, 2), float("nan"), device="cuda")
    stats = torch.empty((n, 4), device="cuda")
    work = torch.empty((int(lib.zb_sh_workspace(band.c, n)),), dtype=torch.uint8, device="cuda")
    prev = lib.zb_knob_set(b"rings_group", group)
    try:
        nat.check(lib.zb_sh_coefficients(band.c, fr, pats.data_ptr(), d_items.data_ptr(), n, flags, work.data_ptr(), work.numel(), alm.data_ptr(),
                                         stats.data_ptr(), engine.stream_ptr()), "coefficients")
        return alm.cpu().numpy(), stats.cpu().numpy(), pats.cpu().numpy(), items
    finally:
        lib.zb_knob_set(b"rings_group", prev)


@pytest.mark.parametrize("L", [8, 16, 24, 40, 64, 96, 150])
@pytest.mark.parametrize("product", ["fp32", "fp16", "bf16"])
def test_coefficients_do_not_depend_on_the_pairs_a_block_takes(L, product):
    from zebsdsolve_amd import _native as nat
    print(f"live rings L {L} {product}", flush=True)
    flags = nat.FLAG_CENTER | nat.FLAG_NORM | {"fp32": 0, "fp16": nat.FLAG_FP16, "bf16": nat.FLAG_BF16}[product]
    one = _coefficients(L, 19, 14.0, flags, 1)
    assert np.isfinite(one[0]).all() and np.abs(one[0]).max() > 0
    for group in (0, 4, 64):
        other = _coefficients(L, 19, 14.0, flags, group)
        assert np.array_equal(one[0], other[0]) and np.array_equal(one[1], other[1]), group


@pytest.mark.parametrize("radius,centre", [(5.0, (8.0, 50.0)), (22.0, None), (9.0, (40.0, 6.0))])
def test_coefficients_of_a_small_window_match_the_oracle(radius, centre):
    from oracle import pipeline as op
    from zebsdsolve_amd import _native as nat
    print(f"live rings oracle radius {radius} centre {centre}", flush=True)
    L = 40
    alm, stats, pats, items = _coefficients(L, 5, radius, nat.FLAG_CENTER, 0, centre)
    fr, _ = cases.oracle_frame(H, W)
    fr = dict(fr)
    c = centre or ((H - 1) / 2, (W - 1) / 2)
    fr["mask"] = (c[0], c[1], radius * radius)
    n, x, wq = op.grid(L)
    for b in range(5):
        v, g = op.sample_grid(pats[b].astype(np.float64), fr, items[b, :3].astype(np.float64), L)
        tot, area = (v * g * wq[:, None]).sum(), (g * wq[:, None]).sum()
        # the window's area and mean: float32 sums of some hundred samples; a sample on the window's edge
        # may fall on either side (one of a few hundred)
        if area == 0:
            assert stats[b, 0] == 0 and np.all(alm[b] == 0)
            continue
        assert abs(stats[b, 0] - area * 2 * np.pi / (2 * n)) < 0.02 * area * 2 * np.pi / (2 * n)
        assert abs(stats[b, 1] - tot / area) < 0.02


def test_an_empty_window_gives_zeros():
    from zebsdsolve_amd import _native as nat
    print("live rings empty", flush=True)
    alm, stats, _, _ = _coefficients(64, 3, 0.01, nat.FLAG_CENTER | nat.FLAG_NORM, 0, (0.37, 0.41))
    assert np.all(alm == 0) and np.all(stats[:, 0] == 0)
