"""A call without a dispatch order (dense particles first, once the particles do not all start at
once) leaves what the same call with an order leaves, bit for bit, and runs every particle once."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")


@pytest.mark.parametrize("net,mixed", [(14, False), (14, True), (86, False), (87, False)])
@pytest.mark.parametrize("extra", [-1, 0, 1, 333])
def test_dense_first_is_any_order(net, mixed, extra):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0, helm_table=TABLE)
    ctx.set_max_iterations(3)
    prec = nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64
    n = ctx.resident_slots(net, nm.EOS_IDEAL, prec) + extra
    cfg = workloads.config({14: 1, 86: 3, 87: 4}[net], n=n, seed=12)
    rng = np.random.default_rng(3)
    rho = 10 ** rng.uniform(4.5, 9.5, n)  # thin (left out), below and above the line
    rho[rng.random(n) < 0.05] = 1e7
    rho[rng.random(n) < 0.02] = np.nan
    rm1 = rho * 0.98
    print(f"dense first: net{net} mixed={mixed} n={n}", flush=True)

    def call(hint):
        st = nm.device_state(torch, net, rho, cfg["temp"], cfg["Y"], cfg["dt"])
        st["rho_m1"] = torch.from_numpy(rm1.copy()).to("cuda:0")
        st["status"].fill_(77)
        if hint is not None:
            st["cost_hint"] = torch.from_numpy(hint).to("cuda:0")
        ctx.compute([ctx.make_batch(net, st, eos=nm.EOS_IDEAL, mu=10.0, precision=prec)], 1e-4, previous_dt=1e-4,
                    use_drhodt=nm.DRHODT_CPU)
        torch.cuda.synchronize()
        return {k: v.cpu().numpy() for k, v in st.items() if k != "cost_hint"}

    a = call(None)
    for hint in (np.ones(n, np.int32), np.zeros(n, np.int32), rng.integers(0, 1 << 20, n).astype(np.int32)):
        b = call(hint)
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=a[k].dtype == np.float64), k
    runs = (rho > 1e5) & (cfg["temp"] > 1e8)
    assert np.array_equal(a["status"] == 1, ~runs) and (a["newton"][runs] > 0).all()
    # rho_m1 became drho/dt once where the particle was integrated
    assert np.array_equal(a["rho_m1"][runs], ((rho - rm1) / 1e-4)[runs])
    ctx.close()
