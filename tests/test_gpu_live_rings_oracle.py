"""The sphere stage leaves out the ring pairs without a sample in the window: for windows of few pairs, in the
frame's middle and off it, every coefficient is the float64 oracle's, in FP32 and 16-bit products. One pair
dropped from the oracle's own samples moves them past the FP32 and FP16 bounds twice over at least."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import gpu_available
from tests.test_gpu_live_rings import H, W, _coefficients

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]

N = 4


def _items(L):
    """The items' detector positions that _coefficients makes for L, in float64."""
    from zebsdsolve_amd import engine
    from zebsdsolve_amd.geometry import Geometry
    e = engine.Engine()
    e.geo = Geometry(pc=cases.PC, sample_tilt_deg=70.0)
    e.shape = (1, 1, H, W)
    t = e.positions(np.zeros(N, np.int64)).astype(np.float32)
    return (t + np.random.default_rng(L).uniform(-1, 1, (N, 3)).astype(np.float32)).astype(np.float64)


def _margin(t, fr, L, centre, radius):
    """How near a grid point's pixel comes to the window's edge or the frame's (pixels)."""
    from oracle import pipeline as op
    n, x, _ = op.grid(L)
    phi = op.TAU * np.arange(2 * n) / (2 * n)
    st = np.sqrt(np.maximum(1 - x * x, 0))
    d = np.stack(np.broadcast_arrays(st[:, None] * np.cos(phi), st[:, None] * np.sin(phi), x[:, None]), -1)
    nd = d @ fr["c2"]
    hv = ((fr["c2"] @ t) / np.where(nd > 1e-4, nd, 1))[..., None] * d - t
    row, col = (hv @ fr["c0"])[nd > 1e-4], (hv @ fr["c1"])[nd > 1e-4]
    edge = np.abs(np.hypot(row - centre[0], col - centre[1]) - radius).min()
    near = np.hypot(row - centre[0], col - centre[1]) < radius + 1
    for v, last in ((row[near], H - 1), (col[near], W - 1)):
        edge = min(edge, np.abs(v).min(initial=9.0), np.abs(v - last).min(initial=9.0))
    return edge


@pytest.mark.parametrize("L,radius,centre", [(16, 9.0, (21.5, 29.5)), (24, 7.0, (9.0, 45.0)), (40, 5.0, (8.0, 50.0)), (40, 9.0, (40.0, 6.0)), (64, 3.0, (30.0, 12.0)),
                                             (64, 8.0, (21.5, 29.5)), (96, 4.0, (20.0, 52.0)), (150, 1.5, (38.0, 20.0))])
def test_coefficients_of_few_ring_pairs_are_the_oracles(L, radius, centre):
    from oracle import pipeline as op, sh as osh
    from zebsdsolve_amd import _native as nat
    fr, _ = cases.oracle_frame(H, W)
    ts = _items(L)
    # (a radius that no grid point's pixel comes within a thousandth of a pixel of, fifty times the float32 rounding
    # of a position, so that both sides count the same samples)
    for k in range(400):
        r = float(np.float32(radius + 0.003 * k))
        if min(_margin(t, fr, L, centre, r) for t in ts) > 1e-3:
            break
    else:
        raise AssertionError("no radius clear of every sample")
    fr = dict(fr, mask=(centre[0], centre[1], float(np.float32(r * r))))
    n, x, wq = op.grid(L)
    weight = np.where(osh.pairs(L)[0] == 0, 1, 2)
    for product, bound in (("fp32", 2e-4), ("fp16", 2e-3), ("bf16", 1.5e-2)):
        # FP32: a position's rounding (2e-5 pixels) times a random pattern's slope against its deviation; 16-bit operands
        # without their low halves: 2^-11 and 2^-8 a product, times four
        print(f"few ring pairs L {L} radius {r:.2f} centre {centre} {product}", flush=True)
        flags = nat.FLAG_CENTER | nat.FLAG_NORM | {"fp32": 0, "fp16": nat.FLAG_FP16, "bf16": nat.FLAG_BF16}[product]
        alm, stats, pats, items = _coefficients(L, N, r, flags, 0, centre)
        assert np.abs(items[:, :3] - ts).max() < 1e-6
        for b in range(N):
            t, pat = items[b, :3].astype(np.float64), pats[b].astype(np.float64)
            ref, _ = op.coefficients(pat, fr, t, L)
            got = alm[b, :, 0] + 1j * alm[b, :, 1]
            assert np.linalg.norm(got - ref) < bound * np.linalg.norm(ref), (product, b)
            if product == "bf16":
                continue
            # the oracle without its first or its last pair of rings in the window
            val, win = op.sample_grid(pat, fr, t, L)
            live = np.flatnonzero(win.sum(1)[:n // 2] + win.sum(1)[::-1][:n // 2])
            assert 0 < len(live) < n // 2
            mean = (val * win * wq[:, None]).sum() / (win * wq[:, None]).sum()
            f = (val - mean) * win
            for y in (live[0], live[-1]):
                cut = f.copy()
                cut[[y, n - 1 - y]] = 0
                less = osh.analyze(cut, L, x, wq)
                less /= np.sqrt(np.sum(weight * np.abs(less) ** 2))
                assert np.linalg.norm(less - ref) > 2 * bound * np.linalg.norm(ref), (product, b, y)
