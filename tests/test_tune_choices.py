"""Solver.tune times a launch-shape value only where it changes the launches (no GPU: every trial takes the
same time, so none is kept)."""
import re
import time
import types

import pytest

from zebsdsolve_amd import Solver, _native, rings_group, sh


def _tried(monkeypatch, L, refine_queue=0):
    """The values tune sets each of the library's knobs to, and not the ones it puts back."""
    import torch
    knobs = {"refine_queue": refine_queue, "rings_group": 0}
    sets = {k: [] for k in knobs}

    def put(name, v):
        old, knobs[name.decode()] = knobs[name.decode()], v
        sets[name.decode()].append(v)
        return old

    ticks = iter(range(10 ** 6))
    monkeypatch.setattr(time, "perf_counter", lambda: float(next(ticks)))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(_native, "load", lambda: types.SimpleNamespace(zb_knob_get=lambda n: knobs[n.decode()], zb_knob_set=put))
    s = Solver.__new__(Solver)
    s._chance = s._chance_key = s._pending = None
    s._gen, s._cancel, s._events, s._step_cells = 0, False, [], 16384
    s._e = types.SimpleNamespace(phases=[object()], shape=(4, 8, 8, 8), spec_budget=1 << 30, index_lanes=1, batch_items=1 << 14,
                                 corr_chunk=lambda k, L, mb=0: k, index_cells=lambda c, L: None,
                                 settings=types.SimpleNamespace(as_dict=lambda: {"bandwidth": L}))
    s.tune()
    return {k: v[::2] for k, v in sets.items()}  # (each value tried is put back)


@pytest.mark.parametrize("L,values", [(16, [4, 8]), (32, [4, 8, 32]), (64, [8, 16, 32]), (96, [8, 16, 32])])
def test_tune_times_the_ring_groups_that_differ_from_the_default(monkeypatch, L, values):
    assert _tried(monkeypatch, L)["rings_group"] == values


def test_the_default_group_is_the_librarys():
    """The lengths and groups that csrc/common.h pads for (fft_shift, fft_lines)."""
    text = open(_native.__file__.replace("_native.py", "csrc/common.h")).read()
    shift = re.search(r"fft_shift\(int log2n\) \{ return log2n == (\d+) \? (\d+) : (\d+); \}", text)
    lines = re.search(r"fft_lines\(int log2n\) \{ return (\d+) >> \(log2n - fft_shift\(log2n\)\); \}", text)
    at, one, other = (int(x) for x in shift.groups())
    for log2n in (7, 8, 9):
        n = (1 << log2n) // 2
        assert rings_group(0, n) == int(lines.group(1)) >> (log2n - (one if log2n == at else other))
    for L in (8, 16, 200, 256):
        n = sh.fft_size(L)
        assert rings_group(0, n) == max(1, min(2048 // (2 * n), n // 2))


@pytest.mark.parametrize("present,values", [(0, [1]), (1, [0]), (2, [0])])
def test_tune_times_the_two_refinement_forms(monkeypatch, present, values):
    """refine_queue 2 is the form 1 is."""
    assert _tried(monkeypatch, 64, present)["refine_queue"] == values
