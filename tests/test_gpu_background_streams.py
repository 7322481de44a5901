"""The static background of a scan that was just set, met first by batches on streams of their own, is the
one a single stream subtracts; and a second stream that meets it later waits for it. (Some milliseconds of
idling stand between the gather of its patterns and their sum.)"""
import numpy as np
import pytest

from tests import cases
from tests.conftest import NI, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


def _scan(rows, cols, dtype):
    rng = np.random.default_rng(7)
    r, c = np.meshgrid(np.arange(40), np.arange(40), indexing="ij")
    x = 90 + 40 * np.exp(-((r - 17) ** 2 + (c - 23) ** 2) / 700.0) + 12 * np.cos(0.4 * r * rng.normal(size=(rows, cols, 1, 1)) + 0.3 * c)
    return np.clip(x + rng.normal(0, 5, x.shape), 0, 250).astype(dtype)


def _solver():
    from zebsdsolve_amd import Solver
    s = Solver()
    s.configure(bandwidth=16, refine_iters=2, static_background="average")
    s.set_geometry(pc=cases.PC, sample_tilt_deg=70.0)
    s.add_phase(NI)
    return s


@pytest.fixture
def slow_background(monkeypatch):
    import torch
    from zebsdsolve_amd import engine
    gather = engine._gather

    def slow(patterns, cells):
        out = gather(patterns, cells)
        torch.cuda._sleep(20_000_000)
        return out

    monkeypatch.setattr(engine, "_gather", slow)


@pytest.mark.parametrize("dtype", [np.uint8, np.uint16])
def test_a_new_scans_background_over_two_lanes(dtype, slow_background):
    print(f"background over two lanes {np.dtype(dtype).name}", flush=True)
    scan = _scan(64, 130, dtype)
    n = 64 * 130
    out = []
    for lanes in (1, 2):
        s = _solver()
        s.set_patterns(scan)
        s._e.index_lanes = lanes
        assert s._e._bg is None
        out.append(s._e.index_cells(np.arange(n)))
    assert len(s._e._lanes) >= 2
    assert np.array_equal(out[0][..., :7], out[1][..., :7])


def test_a_second_stream_waits_for_the_background(slow_background):
    import torch
    print("background met by a second stream", flush=True)
    scan = _scan(20, 30, np.uint8)
    s = _solver()
    s.set_patterns(scan)
    want = s._e.index_cells(np.arange(600))
    s.set_patterns(scan)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(a):
        s._e.static_background()
    with torch.cuda.stream(b):
        got = s._e.index_cells(np.arange(600))
    torch.cuda.synchronize()
    assert np.array_equal(want[..., :7], got[..., :7])


def test_the_scan_outlives_its_engine_for_a_stream_that_reads_it():
    import gc
    import torch
    print("scan read by a stream after its engine is closed", flush=True)
    scan = _scan(64, 130, np.uint8)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    s = _solver()
    s.set_patterns(scan)
    assert s._e._resident is not None
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        raw = s._e._raw_for(np.arange(64 * 130))
        torch.cuda._sleep(50_000_000)
        got = raw.clone()
    del raw
    s.close()
    del s
    gc.collect()
    # memory of the scan's size from the stream that uploaded it, written while the other one idles
    other = [torch.full(scan.shape, 255, dtype=torch.uint8, device="cuda") for _ in range(2)]
    torch.cuda.synchronize()
    assert np.array_equal(got.cpu().numpy().reshape(scan.shape), scan) and int(other[0].min()) == 255
