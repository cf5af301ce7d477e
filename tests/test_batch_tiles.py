"""A tuned batch of unlike sizes: the mixed M2L's tile shape, which a plan's size
decides, is timed apart for small and large trees."""
import numpy as np
import pytest

from simplefmm_amd import api, workloads as W

pytestmark = pytest.mark.gpu


def test_small_plans_keep_their_shape_beside_a_large_one():
    # 20k Plummer points at p = 12: 0.49 ms with 4 wavefronts, 0.67 with 8
    import torch
    dev = torch.device("cuda:0")
    probs = []
    for n in (20_000, 600_000, 15_000):
        pos, q = W.plummer(n, seed=n)
        part = api.OctreePartitioner(pos, api.Box(pos)).refine(20, 64)
        probs.append(dict(n=n, fmm=api.FMM3D(part, 12, ncharge=1, precision=api.MIXED), dq=torch.from_numpy(q).to(dev),
                          du=torch.zeros((n, 4), dtype=torch.float64, device=dev)))
    assert [pb["fmm"].tiles()["m2l_waves"] for pb in probs] == [4, 8, 4]
    batch = api.Batch([(pb["fmm"], api.POTGRAD, 1, pb["dq"].data_ptr(), pb["du"].data_ptr()) for pb in probs],
                      streams=0)
    shapes = [pb["fmm"].tiles() for pb in probs]
    print(f"tuned shapes {shapes}", flush=True)
    assert shapes[0]["m2l_waves"] == 4 and shapes[2] == shapes[0]
    for pb in probs:
        pb["du"].zero_()
    torch.cuda.synchronize()
    batch.launch()
    batch.synchronize()
    for pb in probs:  # one launch gives what the plan's own evaluation gives
        u = torch.zeros_like(pb["du"])
        pb["fmm"].evaluate_device(api.POTGRAD, 1, pb["dq"].data_ptr(), u.data_ptr())
        pb["fmm"].synchronize()
        assert np.array_equal(u.cpu().numpy(), pb["du"].cpu().numpy()), pb["n"]
