"""zb_fit6 (the whole fit in two launches a turn, the items in the order of the master regions they
look up) against the same fit turn by turn through zb_fit6_step / PoseNcc / zb_fit6_keep: item
counts about a wave of 64, a flat pattern's item, the rotation alone, no turn at all."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.test_gpu_fit import fitcase  # noqa: F401 (fixture)

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _turn_by_turn(field, poses0, iters, unknowns, tol):
    import torch
    from zebsdsolve_amd import _native as nat, fit
    from zebsdsolve_amd.engine import stream_ptr
    lib = nat.load()
    poses = torch.as_tensor(poses0, dtype=torch.float32, device="cuda").clone().contiguous()
    n = len(poses)
    flags = fit.ROTATION_ONLY if unknowns == 3 else 0
    local = fit.local_with_autograd(field, poses, flags)
    lam = torch.full((n,), 1e-3, dtype=torch.float64, device="cuda")
    cur = torch.zeros((n, 2), dtype=torch.float64, device="cuda")
    state = torch.zeros((n,), dtype=torch.int32, device="cuda")
    trial = torch.empty_like(poses)
    scored = n
    for _ in range(iters):
        nat.check(lib.zb_fit6_step(poses.data_ptr(), local.data_ptr(), lam.data_ptr(), n, unknowns, float(np.radians(2.0)), 2.0, trial.data_ptr(),
                                   cur.data_ptr(), state.data_ptr(), stream_ptr()), "step")
        tl = fit.local_with_autograd(field, trial, flags, state)
        scored += int((state == 0).sum())
        nat.check(lib.zb_fit6_keep(trial.data_ptr(), tl.data_ptr(), n, tol, cur.data_ptr(), poses.data_ptr(), local.data_ptr(), lam.data_ptr(),
                                   state.data_ptr(), stream_ptr()), "keep")
    return poses, torch.where(local[:, 1] > 0.5, local[:, 0], torch.zeros_like(local[:, 0])), state, scored


@pytest.mark.parametrize("n,iters,unknowns", [(1, 5, 6), (63, 8, 6), (64, 8, 3), (65, 8, 6), (130, 0, 6), (130, 12, 6)])
def test_fit6_is_the_fit_turn_by_turn(fitcase, n, iters, unknowns):  # noqa: F811
    import torch
    from zebsdsolve_amd import fit
    print(f"fit6 turns n {n} iters {iters} unknowns {unknowns}", flush=True)
    field = fitcase["field"]
    rng = np.random.default_rng(n + iters)
    base = np.asarray(fitcase["poses"], np.float32)
    poses = base[rng.integers(0, len(base), n)].copy()
    poses[:, :3] += rng.normal(0, 0.05, (n, 3)).astype(np.float32)
    poses[:, 4:8] *= rng.uniform(0.98, 1.02, (n, 1)).astype(np.float32)  # not quite unit
    flip = rng.random(n) < 0.3
    poses[flip, 4:8] *= -1
    counts = {}
    a = fit.fit6(field, poses, iters=iters, unknowns=unknowns, tol=1e-5, counts=counts)
    b = _turn_by_turn(field, poses, iters, unknowns, 1e-5)
    # the same operations in the same order: the sums are equal, the float64 steps to their rounding
    assert torch.equal(a[2], b[2])
    assert int(counts["scored"]) == b[3]
    assert (a[0] - b[0]).abs().max() < 1e-5
    assert (a[1] - b[1]).abs().max() < 1e-9


def test_fit6_of_a_flat_master_is_state_2(fitcase):  # noqa: F811
    import copy
    import torch
    from zebsdsolve_amd import fit
    print("fit6 flat", flush=True)
    field = copy.copy(fitcase["field"])
    field.grad = torch.zeros_like(field.grad)
    poses, ncc, state = fit.fit6(field, fitcase["poses"], iters=3)
    assert (state == 2).all() and (ncc == 0).all()
    assert torch.equal(poses.cpu(), torch.as_tensor(np.asarray(fitcase["poses"], np.float32)))
