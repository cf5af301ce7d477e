"""Stage times are read once their evaluation has run, beside later work on the plan's stream."""
import numpy as np
import pytest

from simplefmm_amd import api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("recorded", [False, True], ids=["last", "recorded"])
def test_stage_times_do_not_wait_for_later_work(recorded):
    import torch
    pos = np.random.default_rng(5).uniform(size=(5000, 3))
    part = api.OctreePartitioner(pos, api.Box(corner=[0.0, 0.0, 0.0], width=1.0)).refine(8, 40)
    fmm = api.FMM3D(part, 6, ncharge=1)
    q = torch.ones(len(pos), dtype=torch.float64, device="cuda")
    u = torch.zeros((len(pos), 4), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    stream = torch.cuda.ExternalStream(fmm.stream())
    read = (lambda: fmm.recorded_stage_ms(1)[0]) if recorded else fmm.stage_ms
    for _ in range(2):  # the first call makes what later ones use
        if recorded:
            fmm.record_stages(1)
        fmm.evaluate_device(api.POTGRAD, 1, q.data_ptr(), u.data_ptr())
        with torch.cuda.stream(stream):
            torch.cuda._sleep(50_000_000)  # 20 ms at the least
        got = read()
        waiting = not stream.query()
        fmm.synchronize()
        assert waiting and got == read()
        assert 0.0 < got["total"] < 20.0
