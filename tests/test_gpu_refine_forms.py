"""The refinement's launch forms at the frames where they change: 2, 3 or 4 waves a block with the
pixels held in registers (to 24, 36 and 48 steps of 64 masked pixels), 2, 4 or 8 waves with the
list read again in each pass (the waves by the number of items), 16 waves over tiles (past 65 536
pixels). Against the oracle at the recorded orientation, and one batch against another of a
different size (the records do not depend on the form)."""
import ctypes

import numpy as np
import pytest

from tests import cases
from tests.conftest import NI, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _setup(h, w, n, seed):
    import torch
    from oracle import pipeline as op
    from zebsdsolve_amd import _native as nat, engine
    from zebsdsolve_amd.geometry import Geometry
    e = engine.Engine()
    e.settings.apply(static_background="none", dynamic_background="none", mask=False)
    e.geo = Geometry(pc=cases.PC, sample_tilt_deg=70.0)
    e.add_phase(NI)
    e.set_patterns(np.zeros((1, 1, h, w), np.float32))
    R = op.bruker_R(70.0, 0.0)
    fr = op.frame(R, h, w, mask_on=False)
    t = op.translation(R, cases.PC, float(h), float(w))
    rng = np.random.default_rng(h * 1000 + w + seed)
    truth = cases.random_quaternions(rng, n)
    lib, st = nat.load(), engine.stream_ptr()
    poses = torch.zeros((n, 8), dtype=torch.float32)
    poses[:, :3] = torch.from_numpy(np.tile(t.astype(np.float32), (n, 1)))
    poses[:, 4:] = torch.from_numpy(truth.astype(np.float32))
    poses = poses.cuda()
    _, (sheets, grad, host) = e.baked(0)
    side = e.phases[0].master.side
    raw = torch.empty((n, h, w), device="cuda")
    nat.check(lib.zb_project(sheets.data_ptr(), side, e.frame(), poses.data_ptr(), n, raw.data_ptr(), st), "project")
    pats = torch.empty_like(raw)
    mask = (ctypes.c_float * 3)(*e.mask_tuple())
    nat.check(lib.zb_normalize(raw.data_ptr(), 2, n, h, w, mask, pats.data_ptr(), st), "normalize")
    axis = rng.normal(size=(n, 3))
    axis /= np.linalg.norm(axis, axis=1, keepdims=True)
    half = np.radians(0.7) / 2
    turn = np.concatenate([np.full((n, 1), np.cos(half)), axis * np.sin(half)], 1)
    seeds = np.stack([op.qmul(turn[i], truth[i]) for i in range(n)]).astype(np.float32)
    items = torch.from_numpy(np.concatenate([np.tile(t.astype(np.float32), (n, 1)), np.arange(n, dtype=np.float32)[:, None]], 1)).cuda()
    return dict(op=op, nat=nat, lib=lib, st=st, e=e, fr=fr, t=t, truth=truth, sheets=sheets, grad=grad, side=side, pats=pats, seeds=seeds, items=items)


def _refine(c, n, iters=8):
    import torch
    nat = c["nat"]
    seeds = torch.from_numpy(c["seeds"]).cuda()
    opts = nat.RefineOpts(iters, float(np.radians(2.0)), 1.0, 0.02, 1e4, 16, 9)
    rec = torch.full((n, 8), np.nan, dtype=torch.float32, device="cuda")
    nat.check(c["lib"].zb_refine(c["sheets"].data_ptr(), c["e"].grad_half(0).data_ptr(), c["side"], c["e"].frame(), c["pats"].data_ptr(),
                                 c["items"].data_ptr(), seeds.data_ptr(), 4, n, opts, rec.data_ptr(), 0, c["st"]), "refine")
    return rec.cpu().numpy()


@pytest.mark.parametrize("h,w", [(8, 8), (9, 7), (48, 32), (48, 33), (48, 48), (47, 50), (64, 48), (65, 48), (80, 77), (192, 160), (256, 256), (257, 256)])
def test_records_at_the_forms_edges(h, w):
    """The recorded NCC is the oracle's at the recorded orientation (float32 sums over at most
    65 792 pixels against float64: 1e-5), no worse than the seed's (to the half-precision field's
    1e-3), and on frames of at least 1 500 pixels the noise-free pattern's orientation is found."""
    from oracle import pipeline as op
    from zebsdsolve_amd import sym
    n = 5
    print(f"refine form {h}x{w}", flush=True)
    c = _setup(h, w, n, 1)
    r = _refine(c, n)
    assert np.all(r[:, 7] == 9.0)
    g = c["grad"].cpu().numpy().reshape(-1, 4)
    p = c["pats"].cpu().numpy().astype(np.float64)
    for b in range(n):
        _, at, _ = op.refine(g, c["side"], c["fr"], p[b], c["t"], r[b, :4].astype(np.float64), iters=0)
        _, before, _ = op.refine(g, c["side"], c["fr"], p[b], c["t"], c["seeds"][b].astype(np.float64), iters=0)
        assert abs(at - r[b, 4]) < 1e-5, (b, at, r[b, 4])
        assert r[b, 4] > before - 1e-3, (b, before, r[b, 4])
    if h * w >= 1500:
        d = np.degrees(sym.disorientation(r[:, :4].astype(np.float64), c["truth"], c["e"].phases[0].master.rotations))
        assert d.max() < 0.1, d


@pytest.mark.parametrize("h,w", [(56, 56), (70, 70), (130, 128)])
def test_records_do_not_depend_on_the_batch(h, w):
    """The list forms take 8, 4 or 2 waves a block by the number of items: the same items in
    batches of 3, 300 and 600 give the same records bit for bit."""
    print(f"refine batches {h}x{w}", flush=True)
    c = _setup(h, w, 600, 2)
    whole = _refine(c, 600, iters=4)
    for n in (3, 300):
        assert np.array_equal(_refine(c, n, iters=4), whole[:n]), n
