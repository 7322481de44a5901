"""A scan uploaded once gives the results of one page-locked and uploaded step by step, for every pixel type:
index (static background, calibration, several steps), cells out of order, a scan set after another."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import NI, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _scan(dtype, rows, cols, seed):
    rng = np.random.default_rng(seed)
    r, c = np.meshgrid(np.arange(48), np.arange(60), indexing="ij")
    x = 90 + 40 * np.exp(-((r - 20) ** 2 + (c - 33) ** 2) / 900.0) + 12 * np.cos(0.4 * r * rng.normal(size=(rows, cols, 1, 1)) + 0.3 * c)
    return np.clip(x + rng.normal(0, 5, x.shape), 0, 250).astype(dtype)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.float32])
def test_resident_scan_gives_the_page_locked_scans_results(dtype, monkeypatch):
    from zebsdsolve_amd import Solver, engine
    print(f"resident scan {np.dtype(dtype).name}", flush=True)
    out = []
    for resident in (True, False):
        if not resident:
            monkeypatch.setattr(engine.Engine, "_upload_scan", lambda self, a: None)
        with Solver() as s:
            s.configure(bandwidth=24, refine_iters=3, batch=64)
            s.set_geometry(pc=cases.PC, sample_tilt_deg=70.0, px_um=70.0, step_x_um=2.0, step_y_um=2.0)
            s.add_phase(NI)
            for seed in (1, 2):
                s.set_patterns(_scan(dtype, 17, 23, seed))
                s._step_cells = 100
                assert (s._e._resident is not None) == resident
                out.append((s.index(), s.index_cells([300, 5, 17]), s.chance(0)))
    for a, b in ((out[0], out[2]), (out[1], out[3])):
        for x, y in ((a[0], b[0]), (a[1], b[1])):
            assert all(np.array_equal(x[k], y[k], equal_nan=True) for k in x)
        assert a[2] == b[2]
