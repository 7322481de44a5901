"""fit6 of a field with a local model of its own: the plain field's result where that model is the plain one, and
the model's own word where it is not."""
import copy

import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.test_gpu_fit import fitcase  # noqa: F401 (fixture)

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _as(field, cls):
    f = copy.copy(field)
    f.__class__ = cls
    return f


@pytest.mark.parametrize("unknowns", [6, 3])
def test_a_model_handed_on_gives_the_plain_fit(fitcase, unknowns):  # noqa: F811
    from zebsdsolve_amd import fit
    print(f"fit overrides unknowns {unknowns}", flush=True)

    class Same(fit.PoseField):
        def local6(self, poses, flags=0, state=None):
            return super().local6(poses, flags, state)

    poses = np.asarray(fitcase["poses"], np.float32).copy()
    poses[:, :3] += np.random.default_rng(4).normal(0, 0.05, (len(poses), 3)).astype(np.float32)
    ca, cb = {}, {}
    a = fit.fit6(fitcase["field"], poses, iters=9, unknowns=unknowns, tol=1e-5, counts=ca)
    b = fit.fit6(_as(fitcase["field"], Same), poses, iters=9, unknowns=unknowns, tol=1e-5, counts=cb)
    # the same operations, the float64 steps to their rounding
    assert (a[2] == b[2]).all() and int(ca["scored"]) == int(cb["scored"])
    assert (a[0] - b[0]).abs().max() < 1e-5 and (a[1] - b[1]).abs().max() < 1e-9


def test_a_model_of_nothing_moves_nothing(fitcase):  # noqa: F811
    import torch
    from zebsdsolve_amd import fit
    print("fit overrides flat", flush=True)

    class Flat(fit.PoseField):
        def sums(self, poses, flags=0, state=None):
            return torch.zeros_like(super().sums(poses, flags, state))

    poses, ncc, state = fit.fit6(_as(fitcase["field"], Flat), fitcase["poses"], iters=3)
    assert (state == 2).all() and (ncc == 0).all()
    assert torch.equal(poses.cpu(), torch.as_tensor(np.asarray(fitcase["poses"], np.float32)))


@pytest.mark.parametrize("n,iters", [(0, 4), (5, 0), (65, 1), (130, 6), (130, 14)])
def test_last_local_is_the_last_turns_model(fitcase, n, iters):  # noqa: F811
    import torch
    from tests.test_gpu_fit_turns import _turn_by_turn
    from zebsdsolve_amd import fit
    print(f"fit last local n {n} iters {iters}", flush=True)
    base = np.asarray(fitcase["poses"], np.float32)
    rng = np.random.default_rng(n)
    poses = base[rng.integers(0, len(base), n)].copy()
    poses[:, :3] += rng.normal(0, 0.05, (n, 3)).astype(np.float32)
    one, two = copy.copy(fitcase["field"]), copy.copy(fitcase["field"])
    _, ncc, state = fit.fit6(one, poses, iters=iters, tol=1e-4)
    a = one.last_local
    assert a.shape == (n, fit.LOCAL) and a.dtype == torch.float64
    if n == 0:
        return
    _turn_by_turn(two, poses, iters, 6, 1e-4)
    b = two.last_local
    # the same rows scored; their models to the trials' float32 rounding
    assert torch.equal(a[:, 1], b[:, 1]) and (a[a[:, 1] == 0] == 0).all()
    assert ((a - b).abs() <= 1e-4 * b.abs().amax(0)).all()
    if iters == 0:
        assert torch.equal(a[:, 0], ncc)
    if iters == 14:
        assert (a[:, 1] == 0).any()  # some had converged before
