"""A refinement block's waves add their sums in turn. A record for which a wave gave up waiting for its turn
carries no stamp, and every stamped one is the record of an unlimited wait (the knob refine_polls lowered
to a single look: the waits end at once, the kernel as always)."""
import numpy as np
import pytest

from tests.conftest import gpu_available
from tests.test_gpu_refine_forms import _refine, _setup

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.fixture
def one_look():
    from zebsdsolve_amd import _native as nat
    lib = nat.load()

    def looks(n):
        assert lib.zb_knob_set(b"refine_polls", n) > 0

    yield looks
    lib.zb_knob_set(b"refine_polls", 1 << 22)


@pytest.mark.parametrize("h,w,waits", [(48, 48, True), (60, 60, True), (120, 120, True), (257, 256, False)])
def test_a_record_out_of_turn_has_no_stamp(h, w, waits, one_look):
    print(f"refine turns {h}x{w}", flush=True)
    n = 24
    c = _setup(h, w, n, 3)
    whole = _refine(c, n)
    assert np.all(whole[:, 7] == 9.0)
    one_look(1)
    cut = _refine(c, n)
    one_look(1 << 22)
    stamped = cut[:, 7] == 9.0
    assert np.all(stamped | np.isnan(cut[:, 7]))
    # 24 items of 9 passes whose second wave looks once, its own look-ups as long as the first's
    assert stamped.all() != waits
    assert np.array_equal(cut[stamped], whole[stamped])
    assert np.array_equal(_refine(c, n), whole)


@pytest.mark.parametrize("queue", [0, 1])
def test_the_host_refuses_records_out_of_turn(queue, one_look):
    from tests import cases
    from tests.conftest import NI
    from zebsdsolve_amd import Solver, _native as nat
    print(f"records out of turn, queue {queue}", flush=True)
    lib = nat.load()
    s = Solver()
    s.configure(bandwidth=16, refine_iters=3)
    s.set_geometry(pc=cases.PC, sample_tilt_deg=70.0)
    s.add_phase(NI)
    s.set_patterns(np.random.default_rng(3).integers(0, 250, (8, 32, 60, 60), dtype=np.uint8))
    lib.zb_knob_set(b"refine_queue", queue)
    try:
        want = s._e.index_cells(np.arange(256))
        nmi = s._e.nmi_at(0, np.arange(256), want[0, :, :4])
        one_look(1)
        with pytest.raises(RuntimeError, match="stamp"):
            s._e.index_cells(np.arange(256))
        with pytest.raises(RuntimeError, match="stamp"):
            s._e.nmi_at(0, np.arange(256), want[0, :, :4])
        one_look(1 << 22)
        assert np.array_equal(s._e.index_cells(np.arange(256))[..., :7], want[..., :7])
        assert np.array_equal(s._e.nmi_at(0, np.arange(256), want[0, :, :4]), nmi)
    finally:
        lib.zb_knob_set(b"refine_queue", 0)


@pytest.mark.parametrize("h,w", [(8, 8), (14, 14), (16, 16), (24, 24), (30, 30), (32, 32)])
def test_records_do_not_depend_on_the_waves_a_count_takes(h, w):
    """Small frames take one wave a block for many items and one or two for few: the same records."""
    print(f"refine waves {h}x{w}", flush=True)
    n = 1030
    c = _setup(h, w, n, 5)
    many = _refine(c, n, iters=4)
    assert np.all(many[:, 7] == 9.0)
    for few in (1, 7, 1024):
        assert np.array_equal(_refine(c, few, iters=4), many[:few]), few


@pytest.mark.parametrize("n", [40, 1100])
def test_the_persistent_grid_takes_one_wave_a_block_too(n):
    from tests import cases
    from tests.conftest import NI
    from zebsdsolve_amd import Solver, _native as nat
    print(f"refine queue of one wave, {n} cells", flush=True)
    lib = nat.load()
    s = Solver()
    s.configure(bandwidth=16, refine_iters=3, static_background="none", dynamic_background="none")
    s.set_geometry(pc=cases.PC, sample_tilt_deg=70.0)
    s.add_phase(NI)
    s.set_patterns(np.random.default_rng(3).integers(0, 250, (1, n, 16, 16), dtype=np.uint8))
    want = s._e.index_cells(np.arange(n))
    lib.zb_knob_set(b"refine_queue", 1)
    try:
        got = s._e.index_cells(np.arange(n))
    finally:
        lib.zb_knob_set(b"refine_queue", 0)
    assert np.array_equal(got[..., :7], want[..., :7])
