"""Attempts that restart from an accepted state on the device: a call that runs many of them, keeping
the state's rates and Jacobian from one to the next, leaves the timesteps that calls ending after
each attempt leave (every call computes them anew), bit for bit."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")
K = 24  # Newton iterations of the long call


@pytest.mark.parametrize("cid,n,mixed,drhodt", [(1, 200, False, 0), (2, 400, False, 0), (2, 400, True, 2), (3, 4000, False, 0),
                                                (3, 1500, True, 0), (4, 1200, False, 0), (4, 1200, False, 2)])
def test_restarted_attempts_are_the_kept_ones(cid, n, mixed, drhodt):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    cfg = workloads.config(cid, n=n, seed=31)
    ctx = nm.Context(0, helm_table=TABLE)
    rm1 = cfg["rho"] * (1 + 0.02 * np.random.default_rng(5).standard_normal(n))

    def call(dt, cap):
        st = nm.device_state(torch, cfg["net"], cfg["rho"], cfg["temp"], cfg["Y"], dt)
        if drhodt:
            st["rho_m1"] = torch.from_numpy(rm1.copy()).to("cuda:0")
        ctx.set_max_iterations(cap)
        ctx.compute([ctx.make_batch(cfg["net"], st, eos=cfg["eos"], mu=10.0, Z=cfg["Z"],
                                    precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)],
                    cfg["hydro_dt"], previous_dt=cfg["hydro_dt"], use_drhodt=drhodt)
        torch.cuda.synchronize()
        return {k: st[k].cpu().numpy() for k in ("dt", "status", "substeps", "fp64_solves") if k in st}

    print(f"retries: set {cid} n={n} mixed={mixed} drhodt={drhodt}", flush=True)
    runs = [call(cfg["dt"], k) for k in range(1, K + 1)]
    dts = np.stack([cfg["dt"]] + [r["dt"] for r in runs])
    # every attempt rejected in its L-th iteration, no substep accepted: the restarted call starts
    # each attempt from the same state (a mixed call that leaves a particle to the FP64 solve repeats
    # all of its attempts there, calls of single attempts only the one that failed: left out)
    open_ = np.all([(r["status"] == 4) & (r["substeps"] == 0) for r in runs], axis=0)
    if mixed:
        open_ &= runs[-1]["fp64_solves"] == 0
    changed = dts[1:] != dts[:-1]
    found = 0
    for L in (1, 2, 3):
        ends = np.arange(1, K + 1) % L == 0
        sel = open_ & np.all(changed == ends[:, None], axis=0)
        found += int(sel.sum())
        dt = cfg["dt"]
        for j in range(K // L if sel.any() else 0):
            dt = call(dt, L)["dt"]
            assert np.array_equal(dt[sel], dts[(j + 1) * L][sel]), (L, j)
        print(f"retries: {int(sel.sum())} particles with attempts of {L}", flush=True)
    if cid == 2 and not mixed:  # the alpha network's set always holds such particles
        assert found >= 1
    ctx.close()
