"""A few items' correlation (the GEMM's blocks along b, waves whose items are all padding) gives each
item the record it has in a batch that fills the chip, bit for bit: item counts about a wave's 32 and
a block's 128 items, the row counts of every transform length, FP32 and 16-bit products."""
import numpy as np
import pytest

from tests import cases
from tests.conftest import GAN, NI, gpu_available

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="needs a GPU")]


@pytest.mark.parametrize("master,L,precision", [("ni", 16, "fp32"), ("ni", 33, "fp32"), ("ni", 64, "fp32"), ("ni", 64, "fp16"), ("ni", 96, "fp32"), ("ni", 96, "bf16"),
                                                ("gan", 48, "fp32")])
def test_few_items_records_are_those_of_a_large_batch(master, L, precision):
    import torch
    from zebsdsolve_amd import engine
    from zebsdsolve_amd.geometry import Geometry
    print(f"vcorr split {master} L {L} {precision}", flush=True)
    e = engine.Engine()
    e.settings.apply(static_background="none", dynamic_background="none", bandwidth=L, refine_iters=1, correlation_precision=precision)
    e.geo = Geometry(pc=cases.PC, sample_tilt_deg=70.0)
    e.add_phase(NI if master == "ni" else GAN)
    n, h, w = 1600, 60, 60
    e.set_patterns(np.zeros((1, 1, h, w), np.float32))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(L)
    raw = torch.rand((n, h, w), generator=gen, device="cuda")
    t = e.positions(np.zeros(n, np.int64)).astype(np.float32)
    items = torch.from_numpy(np.concatenate([t, np.arange(n, dtype=np.float32)[:, None]], 1)).cuda()
    full = e.run_batch(raw, items)[0][..., :7].clone()
    for k in (1, 3, 32, 33, 128, 129, 400):
        few = e.run_batch(raw[:k].contiguous(), items[:k].contiguous())[0][..., :7]
        assert torch.equal(few, full[:, :k]), k
