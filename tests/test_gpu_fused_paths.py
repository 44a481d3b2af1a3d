"""The fused launch of three networks against one launch per batch, bit for bit, over the paths the
launch has: both EOS, both precisions, with and without cost hints and each form of drho/dt; more
particles than are resident at once."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")
SIZES = ((14, 2500), (86, 700), (87, 600))


@pytest.mark.parametrize("eos,mixed,hints,drhodt", [(0, False, False, 0), (0, False, True, 1), (0, False, False, 2),
                                                    (0, True, False, 0), (0, True, True, 2), (1, False, True, 0),
                                                    (1, False, False, 1), (1, False, True, 2), (1, True, False, 0),
                                                    (1, True, True, 2)])
def test_fused_is_per_batch(eos, mixed, hints, drhodt):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0, helm_table=TABLE)
    ctx.set_max_iterations(60)
    rng = np.random.default_rng(17)
    cfgs = []
    for (net, n), cid in zip(SIZES, (2, 3, 4)):
        c = workloads.config(cid, n=n, seed=71 + cid)
        c["rm1"] = np.where(rng.random(n) < 0.1, 0., c["rho"] * (1 + 0.02 * rng.standard_normal(n)))
        c["hint"] = np.where(rng.random(n) < 0.3, 0, rng.integers(0, 1 << 14, n)).astype(np.int32)
        assert c["net"] == net
        cfgs.append(c)
    print(f"fused paths: eos={eos} mixed={mixed} hints={hints} drhodt={drhodt}", flush=True)

    def call(fused):
        ctx.set_fused_launch(fused)
        sts = []
        for c in cfgs:
            st = nm.device_state(torch, c["net"], c["rho"], c["temp"], c["Y"], c["dt"])
            if hints:
                st["cost_hint"] = torch.from_numpy(c["hint"]).to("cuda:0")
            if drhodt:
                st["rho_m1"] = torch.from_numpy(c["rm1"].copy()).to("cuda:0")
            sts.append(st)
        ctx.compute([ctx.make_batch(c["net"], st, eos=eos, mu=10.0, Z=c["Z"] if eos else None,
                                    precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)
                     for c, st in zip(cfgs, sts)], 1e-5, previous_dt=1e-5, use_drhodt=drhodt)
        torch.cuda.synchronize()
        return [{k: v.cpu().numpy() for k, v in st.items()} for st in sts]

    a, b = call(True), call(False)
    for c, x, y in zip(cfgs, a, b):
        assert int(x["newton"].sum()) > c["rho"].size  # the particles burn
        for k in x:
            assert np.array_equal(x[k].view(np.uint8), y[k].view(np.uint8)), (c["net"], k)
    ctx.close()
