"""Attempts after a rejection in a later iteration: their first iteration takes the accepted state's
arrays back from registers.  For every particle and every attempt before its first accepted substep,
a call that starts with the timestep the attempt before it left, and ends with the attempt's last
iteration, has to leave the timestep that the long call leaves, bit for bit; each configuration must
hold attempts after one-iteration attempts and after longer ones.

The mixed solve is here for net14 alone: on net86 and net87 it leaves a particle to the FP64 solve
before a second attempt (none of 100,000 particles of either network keeps one)."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")
K = 12  # Newton iterations of the long call


@pytest.mark.parametrize("cid,eos,n,mixed,drhodt", [(1, 0, 3000, False, 0), (2, 1, 2000, False, 0), (2, 1, 2000, False, 2),
                                                    (3, 1, 3000, False, 0), (3, 1, 3000, False, 2), (3, 0, 3000, False, 0),
                                                    (4, 1, 2000, False, 0), (4, 1, 2000, False, 2),
                                                    (1, 0, 40000, True, 0), (2, 1, 40000, True, 0),
                                                    (2, 1, 40000, True, 2)])
def test_attempts_after_later_rejections(cid, eos, n, mixed, drhodt):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    cfg = workloads.config(cid, n=n, seed=31)
    rng = np.random.default_rng(9)
    dt0 = 10 ** rng.uniform(-12, -3, n)  # from timesteps that are accepted to ones that fail often
    rm1 = cfg["rho"] * (1 + 0.02 * rng.standard_normal(n))
    ctx = nm.Context(0, helm_table=TABLE)

    def call(dt, cap):
        st = nm.device_state(torch, cfg["net"], cfg["rho"], cfg["temp"], cfg["Y"], dt)
        st["rho_m1"] = torch.from_numpy(rm1.copy()).to("cuda:0")
        ctx.set_max_iterations(cap)
        ctx.compute([ctx.make_batch(cfg["net"], st, eos=eos, mu=10.0, Z=cfg["Z"] if eos else None,
                                    precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)],
                    1e-2, previous_dt=1e-2, use_drhodt=drhodt)
        torch.cuda.synchronize()
        return {k: st[k].cpu().numpy() for k in ("dt", "status", "substeps", "fp64_solves")}

    print(f"restored: set {cid} eos={eos} n={n} mixed={mixed} drhodt={drhodt}", flush=True)
    runs = [call(dt0, k) for k in range(1, K + 1)]
    dts = np.stack([dt0] + [r["dt"] for r in runs])
    # still before the first accepted substep (and not left to the FP64 solve)
    alive = np.stack([(r["status"] == 4) & (r["substeps"] == 0) & (r["fp64_solves"] == 0 if mixed else True)
                      for r in runs])
    ended = (dts[1:] != dts[:-1]) & alive  # an attempt was rejected in this iteration
    last = np.zeros(n, int)  # iterations before the running attempt
    prev = np.zeros(n, int)  # length of the attempt before it (0: none)
    found = {"after one": 0, "after more": 0}
    for k in range(K):
        length = k + 1 - last
        for L in np.unique(length[ended[k]]):
            sel = ended[k] & (length == L) & (prev > 0)
            if sel.any():
                dt = dts[last, np.arange(n)]
                assert np.array_equal(call(dt, int(L))["dt"][sel], dts[k + 1][sel]), (k, L)
                found["after one"] += int((sel & (prev == 1)).sum())
                found["after more"] += int((sel & (prev > 1)).sum())
        prev = np.where(ended[k], length, prev)
        last = np.where(ended[k], k + 1, last)
    print(f"restored: attempts {found}", flush=True)
    assert min(found.values()) >= 5
    ctx.close()
