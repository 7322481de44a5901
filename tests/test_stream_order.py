"""What a batch on a stream of its own reads is made before that stream starts (no GPU: stand-ins
note the order of the calls)."""
import types

import numpy as np
import pytest

from zebsdsolve_amd import engine


class Stop(Exception):
    pass


@pytest.mark.parametrize("background", ["average", "file", "none"])
def test_a_lane_waits_after_the_static_background_is_made(background, monkeypatch):
    import torch
    calls = []
    e = engine.Engine.__new__(engine.Engine)
    e.settings = {"static_background": background, "bandwidth": 8}
    e.phases = [object()]
    e.spec_budget, e.batch_items = 1 << 20, 64
    e._device = lambda: "cpu"
    e.band = lambda L: types.SimpleNamespace(c=None, host=types.SimpleNamespace(pairs=36))
    e.frame = lambda: None
    e.mask_tuple = lambda: (0.0, 0.0, 0.0)
    e.refine_opts = lambda: None
    e.phase_band = lambda pi, L: types.SimpleNamespace(c=None)
    e.use_mfma = lambda L, pi: False
    e.rden = lambda pi, L: None
    e.baked = lambda pi: (None, (None, None, None))
    e.grad_half = lambda pi: None

    def made():
        calls.append("background")
        return types.SimpleNamespace(record_stream=lambda st: calls.append("kept for the lane"))

    def wait(stream):
        calls.append("wait")

    def buf(*a):
        raise Stop

    e.static_background = made
    lane = types.SimpleNamespace(stream=types.SimpleNamespace(wait_stream=wait, cuda_stream=0), buf=buf)
    monkeypatch.setattr(engine.nat, "load", lambda: types.SimpleNamespace(zb_so3_workspace=lambda *a: 8, zb_sh_workspace=lambda *a: 8))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: None)
    with pytest.raises(Stop):
        e.run_batch(torch.zeros((2, 4, 4)), torch.zeros((2, 4)), lane=lane)
    assert calls == (["wait"] if background == "none" else ["background", "wait", "kept for the lane"])
