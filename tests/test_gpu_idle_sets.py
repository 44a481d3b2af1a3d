"""Calls without an order on sets of which a part does not burn: the same results as with an order,
every particle looked at once, and positions taken once where most of them are idle."""
import os
import time

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")


def _set(net, n, idle, seed=5):
    cfg = workloads.config({14: 2, 86: 3, 87: 4}[net], n=n, seed=seed)
    rng = np.random.default_rng(seed)
    rho, temp = 10 ** rng.uniform(5.2, 9, n), 10 ** rng.uniform(8.2, 9.5, n)
    off = rng.random(n) < idle
    thin = off & (rng.random(n) < 0.5)  # half of the idle ones are thin, half cold (dense ones among them)
    rho[thin] = 10 ** rng.uniform(2, 4.9, thin.sum())
    temp[off & ~thin] = 10 ** rng.uniform(6, 7.9, (off & ~thin).sum())
    return cfg, rho, temp, off


def _call(torch, nm, ctx, cfg, rho, temp, mixed=False, hint=None):
    st = nm.device_state(torch, cfg["net"], rho, temp, cfg["Y"], cfg["dt"])
    st["status"].fill_(77)
    if hint is not None:
        st["cost_hint"] = torch.from_numpy(hint).to("cuda:0")
    b = ctx.make_batch(cfg["net"], st, eos=cfg["eos"], mu=10.0, Z=cfg["Z"],
                       precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)
    ctx.compute([b], 1e-5)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in st.items() if k != "cost_hint"}, b, st


@pytest.mark.parametrize("net,mixed", [(14, False), (86, False), (86, True), (87, False)])
@pytest.mark.parametrize("idle", [0., 0.2, 0.45, 0.55, 0.9, 1.])
def test_idle_share_changes_no_result(net, mixed, idle):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0, helm_table=TABLE)
    ctx.set_max_iterations(3)
    prec = nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64
    n = ctx.resident_slots(net, nm.EOS_HELMHOLTZ, prec) + 333
    cfg, rho, temp, off = _set(net, n, idle)
    print(f"idle sets: net{net} mixed={mixed} idle={idle} n={n}", flush=True)
    a, *_ = _call(torch, nm, ctx, cfg, rho, temp, mixed)
    b, *_ = _call(torch, nm, ctx, cfg, rho, temp, mixed, hint=np.ones(n, np.int32))
    for k in a:
        assert np.array_equal(a[k].view(np.uint8), b[k].view(np.uint8)), k
    assert np.array_equal(a["status"] == 1, off) and (a["newton"][~off] > 0).all()
    ctx.close()


@pytest.mark.parametrize("net", [14, 86])
def test_idle_set_takes_each_position_once(net):
    # an idle call's time is its positions taken (one atomic each): twice as many take twice as long.
    # The ordered call takes each once.
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    ctx = nm.Context(0, helm_table=TABLE)
    n = 200000
    cfg, rho, temp, _ = _set(net, n, 1.)
    print(f"idle set timing: net{net}", flush=True)
    best = []
    for hint in (None, np.ones(n, np.int32)):
        _, b, st = _call(torch, nm, ctx, cfg, rho, temp, hint=hint)
        t = []
        for _ in range(9):
            t0 = time.perf_counter()
            ctx.compute([b], 1e-5)
            t.append(time.perf_counter() - t0)
        best.append(min(t))
    print(f"idle set timing: net{net} without an order {best[0] * 1e3:.3f} ms, with {best[1] * 1e3:.3f} ms", flush=True)
    assert best[0] < 1.4 * best[1]
    ctx.close()
