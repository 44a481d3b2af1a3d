"""The fused launch of several networks against one launch per batch, bit for bit, with more particles
than are resident at once (workgroups that go on to a second particle and to other networks)."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")


@pytest.mark.parametrize("sizes,mixed", [((2500, 600, 0), False), ((360, 360, 180), False), ((2500, 700, 600), False),
                                         ((2500, 600, 0), True)])
def test_fused_is_per_batch(sizes, mixed):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0, helm_table=TABLE)
    ctx.set_max_iterations(100)
    cfgs = [workloads.config(c, n=n, seed=61 + c) for c, n in zip((2, 3, 4), sizes) if n]
    print(f"fused: {sizes} mixed={mixed}", flush=True)

    def call(fused):
        ctx.set_fused_launch(fused)
        sts = [nm.device_state(torch, c["net"], c["rho"], c["temp"], c["Y"], c["dt"]) for c in cfgs]
        ctx.compute([ctx.make_batch(c["net"], st, eos=c["eos"], Z=c["Z"],
                                    precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)
                     for c, st in zip(cfgs, sts)], 1e-5)
        torch.cuda.synchronize()
        return [{k: v.cpu().numpy() for k, v in st.items()} for st in sts]

    for c, a, b in zip(cfgs, call(True), call(False)):
        for k in a:
            assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), (c["net"], k)
    ctx.close()
