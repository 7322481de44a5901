"""Arguments that do not fit are refused on the host, before any launch: a kernel takes its counts and
indices as they come. No GPU: the engine's device side is replaced by stand-ins that note a call."""
import ctypes
import types

import numpy as np
import pytest

from zebsdsolve_amd import engine


class Launched(Exception):
    """A stand-in for the device was reached."""


def _engine(rows=2, cols=3, h=8, w=8):
    """An engine of a host scan that has no device."""
    e = engine.Engine.__new__(engine.Engine)
    e.shape = (rows, cols, h, w)
    e.patterns = np.arange(rows * cols * h * w, dtype=np.float32).reshape(e.shape)
    e._device = lambda: "cpu"
    return e


@pytest.mark.parametrize("n,shape", [(3, (4, 4)), (3, (8, 4)), (3, (2, 2, 4)), (5, (7, 4)), (3, (2, 4, 3)), (0, (1, 4)), (3, (0, 4))])
def test_nmi_at_refuses_orientations_that_do_not_fit_the_cells(n, shape, monkeypatch):
    e = _engine()

    def raw(cells):
        raise Launched

    e._raw_for = raw
    monkeypatch.setattr(engine.nat, "load", lambda: types.SimpleNamespace())
    with pytest.raises(ValueError):
        e.nmi_at(0, np.arange(n), np.zeros(shape, np.float32))


@pytest.mark.parametrize("n,shape,launched,result", [(3, (3, 4), 3, (3,)), (1, (4,), 1, (1,)), (3, (12,), 3, (3,)), (3, (8, 3, 4), 24, (8, 3)), (3, (1, 3, 4), 3, (1, 3)),
                                                     (6, (2, 3, 4), 6, (6,))])
def test_nmi_at_launches_an_item_an_orientation(n, shape, launched, result, monkeypatch):
    import torch
    e = _engine()
    e.settings = {"refine": False, "nmi_bins": 8}
    e.phases = [types.SimpleNamespace(master=types.SimpleNamespace(side=5))]
    e.mask_tuple = lambda: (0.0, 0.0, 0.0)
    e.prep_into = lambda *a: None
    e.refine_opts = lambda: types.SimpleNamespace(iters=1, stamp=1)
    e.positions = lambda cells: np.zeros((len(cells), 3), np.float32)
    e.baked = lambda pi: (None, (torch.zeros(1), None, None))
    e.grad_half = lambda pi: torch.zeros(1)
    e.frame = lambda: None
    seen = []

    def refine(*a):
        seen.append(a[8])
        (ctypes.c_float * (8 * a[8])).from_address(a[10])[7::8] = [1.0] * a[8]  # the records' stamps
        return 0

    monkeypatch.setattr(engine.nat, "load", lambda: types.SimpleNamespace(zb_refine=refine))
    monkeypatch.setattr(engine, "stream_ptr", lambda: None)
    out = e.nmi_at(0, np.arange(n), np.zeros(shape, np.float32))
    assert seen == [launched] and out.shape == result


@pytest.mark.parametrize("shape", [(5, 7), (8,), (5, 9), (2, 5, 8), ()])
def test_fit6_refuses_poses_that_are_not_rows_of_eight(shape, monkeypatch):
    import torch
    from zebsdsolve_amd import fit

    def launched(*a):
        raise Launched

    monkeypatch.setattr(fit.nat, "load", lambda: types.SimpleNamespace(zb_fit6=launched, zb_fit6_workspace=launched))
    field = types.SimpleNamespace(pats=torch.zeros((1, 4, 4)))
    with pytest.raises(ValueError):
        fit.fit6(field, np.zeros(shape, np.float32))


@pytest.mark.parametrize("cells", [[6], [5, 6], [0, 9, 2], [-7, 0], [3, -8, 1]])
@pytest.mark.parametrize("resident", [True, False])
def test_cells_outside_the_map_are_refused(cells, resident):
    import torch
    e = _engine(2, 3)
    # (a tensor on the meta device checks no index, as one on a GPU before its kernel runs)
    e._resident = torch.empty(e.shape, device="meta") if resident else None
    e._device = lambda: torch.device("meta" if resident else "cpu")
    with pytest.raises(IndexError):
        e._raw_for(cells)


@pytest.mark.parametrize("cells", [[5], [0, 1, 2], [4, 0, 5], [-1], [-2, -1], [-1, 0, 1], [-6, 3], []])
@pytest.mark.parametrize("resident", [True, False])
def test_cells_of_the_map_give_their_patterns(cells, resident):
    import torch
    e = _engine(2, 3)
    e._resident = torch.from_numpy(e.patterns) if resident else None
    got = e._raw_for(cells)
    assert np.array_equal(got.numpy(), e.patterns.reshape(6, 8, 8)[np.asarray(cells, np.int64)])
