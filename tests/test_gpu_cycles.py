"""Exact cycles of rejected attempts on the device: the timestep a capped particle is left with
follows the particle's period, whichever cap stops it, and its counts and state are the cap's."""
import os

import numpy as np
import pytest

import workloads

pytestmark = pytest.mark.gpu

TABLE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sph-exa-nnet_amd", "data",
                     "helm_table.bin")
FIRST, SPAN, PERIOD = 400, 41, 20  # trajectory caps FIRST .. FIRST + SPAN - 1, longest period looked for


@pytest.mark.parametrize("cid,n,mixed", [(2, 400, False), (2, 400, True), (3, 6000, False), (4, 300, False)])
def test_capped_particles_follow_their_period(cid, n, mixed):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    import nnet_mi355x as nm
    cfg = workloads.config(cid, n=n, seed=77)
    ctx = nm.Context(0, helm_table=TABLE)

    def step(cap):
        st = nm.device_state(torch, cfg["net"], cfg["rho"], cfg["temp"], cfg["Y"], cfg["dt"])
        ctx.set_max_iterations(cap)
        ctx.compute([ctx.make_batch(cfg["net"], st, eos=cfg["eos"], Z=cfg["Z"],
                                    precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)], cfg["hydro_dt"])
        torch.cuda.synchronize()
        return {k: v.cpu().numpy() for k, v in st.items()}

    print(f"cycles: set {cid} n={n} mixed={mixed}", flush=True)
    runs = [step(FIRST + k) for k in range(SPAN)]
    dts = np.stack([r["dt"] for r in runs])
    far = step(3 * FIRST + 7), step(2003)
    capped = (runs[0]["status"] == 4) & (far[0]["status"] == 4) & (far[1]["status"] == 4)
    found = 0
    for p in np.nonzero(capped)[0]:
        L = next((q for q in range(1, PERIOD + 1) if np.array_equal(dts[q:, p], dts[:-q, p])), 0)
        if not L:
            continue
        if any(r["substeps"][p] != far[1]["substeps"][p] for r in runs):
            continue
        found += 1
        for r, cap in ((far[0], 3 * FIRST + 7), (far[1], 2003)):
            assert r["newton"][p] == cap and r["substeps"][p] == runs[0]["substeps"][p]
            assert r["dt"][p] == dts[(cap - FIRST) % L, p], (p, L, cap)
            assert r["temp"][p] == runs[0]["temp"][p] and np.array_equal(r["Y"][:, p], runs[0]["Y"][:, p])
    print(f"cycles: {found} periodic of {int(capped.sum())} capped", flush=True)
    assert found >= 1
    # a particle that ends under the lowest cap does not depend on the cap
    done = runs[0]["status"] != 4
    for k in ("Y", "temp", "dt", "status", "substeps", "newton"):
        assert np.array_equal(runs[0][k][..., done], far[1][k][..., done], equal_nan=True), k
    ctx.close()
