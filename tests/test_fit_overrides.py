"""fit6 of a field with sums or a local model of its own takes them (no GPU: the library's steps are stand-ins
that note a call)."""
import types

import pytest

from zebsdsolve_amd import engine, fit


class WholeFit(Exception):
    pass


def _field(cls):
    import torch
    f = cls.__new__(cls)
    f.pats = torch.zeros((1, 4, 4))
    f.grad, f.side, f.frame = torch.zeros(1), 2, None
    return f


def _lib(calls):
    def whole(*a):
        raise WholeFit

    def note(name):
        def call(*a):
            calls.append(name)
            return 0
        return call

    return types.SimpleNamespace(zb_fit6=whole, zb_fit6_workspace=lambda n: 8 * fit.LOCAL * n, zb_fit6_step=note("step"), zb_fit6_keep=note("keep"),
                                 zb_local6=note("local6"), zb_sums=note("sums"), zb_sums_active=note("sums"))


def _model(self, poses, flags=0, state=None):
    import torch
    self.calls.append("own")
    return torch.zeros((len(poses), fit.LOCAL), dtype=torch.float64)


def _sums(self, poses, flags=0, state=None):
    import torch
    self.calls.append("own")
    return torch.zeros((len(poses), fit.N_SUMS))


@pytest.mark.parametrize("how", ["local6", "sums", "on the object", "on the class"])
def test_fit6_takes_a_fields_own_model(how, monkeypatch):
    import torch
    calls = []
    monkeypatch.setattr(fit.nat, "load", lambda: _lib(calls))
    monkeypatch.setattr(engine, "stream_ptr", lambda: None)
    if how == "on the object":
        f = _field(fit.PoseField)
        f.local6 = types.MethodType(_model, f)
    elif how == "on the class":
        monkeypatch.setattr(fit.PoseField, "local6", _model)
        f = _field(fit.PoseField)
    else:
        f = _field(type("Own", (fit.PoseField,), {"local6": _model} if how == "local6" else {"sums": _sums}))
    f.calls = calls
    poses, ncc, state = fit.fit6(f, torch.tensor([[0.0, 0, 1, 0, 1, 0, 0, 0]] * 3), iters=2)
    assert [c for c in calls if c != "local6"] == ["own", "step", "own", "keep", "step", "own", "keep"]
    assert poses.shape == (3, 8) and ncc.shape == (3,) and state.shape == (3,)


@pytest.mark.parametrize("sub", [False, True])
def test_fit6_of_a_plain_field_is_one_call(sub, monkeypatch):
    import torch
    monkeypatch.setattr(fit.nat, "load", lambda: _lib([]))
    monkeypatch.setattr(engine, "stream_ptr", lambda: None)
    f = _field(type("Named", (fit.PoseField,), {"name": "mine"}) if sub else fit.PoseField)
    with pytest.raises(WholeFit):
        fit.fit6(f, torch.zeros((3, 8)))


@pytest.mark.parametrize("iters,turns", [(0, 0), (7, 7), (-3, 0), (True, 1)])
def test_fit6_takes_whole_numbers_of_turns(iters, turns, monkeypatch):
    import torch
    seen = []
    lib = _lib([])
    lib.zb_fit6 = lambda *a: seen.append(a[7]) or 0
    monkeypatch.setattr(fit.nat, "load", lambda: lib)
    monkeypatch.setattr(engine, "stream_ptr", lambda: None)
    fit.fit6(_field(fit.PoseField), torch.zeros((3, 8)), iters=iters)
    assert seen == [turns]
    with pytest.raises(TypeError):
        fit.fit6(_field(fit.PoseField), torch.zeros((3, 8)), iters=2.5)
