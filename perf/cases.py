"""The work a program has this framework do, as cases that can be timed and compared.

Two public calls carry a hydro step's nuclear physics, and both are here through the package's
binding as a program calls them:

  solve  Context.compute: the implicit network integration of a particle set over hydro steps
         (net14 / net86 / net87, ideal-gas or Helmholtz EOS, FP64 or mixed-precision solve, with
         and without the dispatch hints of an earlier step, with and without drho/dt, one network
         or several per call);
  eos    Context.helm_eos: the post-step Helmholtz refresh of u, cv, p, c and dP/dT.

The particle sets are the distributions of workloads.py (C1 - C5) and of the ideal-gas tests of
net86 / net87.  run() of a solve case first writes the particle state the hydro code hands over
(abundances, temperature, timestep), so that every pass integrates the same inputs.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "sph-exa-nnet_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import nnet_mi355x as nm  # noqa: E402
import workloads  # noqa: E402

TABLE = os.path.join(PKG, "data", "helm_table.bin")
DEV = "cuda:0"
NSP = {14: 14, 86: 86, 87: 87}

# hydro step (s) of each particle set: workloads.config's, and the ideal-gas tests' of net86 / net87
HYDRO_DT = {(14, 0): 1e-3, (14, 1): 1e-4, (86, 0): 1e-4, (86, 1): 1e-4, (87, 0): 1e-4, (87, 1): 1e-5}

# Newton iterations per particle and hydro step of each set (measured means, cap 10,000), for work()
NEWTON = {(14, 0): 13.0, (14, 1): 680.0, (86, 0): 20.0, (86, 1): 11.0, (87, 0): 20.0, (87, 1): 310.0}


def _solve(name, net, n, eos=1, mixed=False, steps=1, hints=False, drhodt=0, cap=10000):
    return {"name": name, "kind": "solve", "net": net, "n": n, "eos": eos, "mixed": mixed, "steps": steps,
            "hints": hints, "drhodt": drhodt, "cap": cap}


def _eos(name, net, n):
    return {"name": name, "kind": "eos", "net": net, "n": n}


def listed():
    return [
        # EOS refresh of a handful of zones: a one-zone burn or a debugging run; latency only
        _eos("eos net14 n=100", 14, 100),
        # EOS refresh of a small, odd share of particles after an alpha-network step
        _eos("eos net14 n=50021", 14, 50021),
        # EOS refresh of a full GPU's particles (the size the benchmark quotes)
        _eos("eos net86 n=2097152", 86, 2097152),
        # the reference driver's own size: 1,000 ideal-gas zones on net14
        _solve("net14 ideal n=1000", 14, 1000, eos=0),
        # a few zones of a parameter study, the guard on Newton iterations lowered
        _solve("net14 n=37 cap=2000", 14, 37, cap=2000),
        # an alpha-network supernova run's share of particles, first step (no hints yet)
        _solve("net14 n=50021", 14, 50021),
        # small ideal-gas net86 set with the density derivative integrated
        _solve("net86 ideal drhodt n=517", 86, 517, eos=0, drhodt=2),
        # net86, first hydro step of a large particle set (the benchmark's workload)
        _solve("net86 n=524288", 86, 524288),
        # net86, two hydro steps, the second dispatched by the first one's Newton counts
        _solve("net86 hints 2 steps n=60013", 86, 60013, steps=2, hints=True, cap=2000),
        # net86 with the mixed-precision solve, two steps with both hints
        _solve("net86 mixed 2 steps n=20011", 86, 20011, mixed=True, steps=2, hints=True, cap=2000),
        # net87 (electron captures) at the iteration cap the multi-step tests use
        _solve("net87 n=4099 cap=2000", 87, 4099, cap=2000),
        # net14 + net86 + net87 particles (2:2:1) in one call
        {"name": "fused n=5005 cap=2000", "kind": "fused", "n": 5005, "steps": 1, "hints": False, "cap": 2000},
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["eos", "solve", "solve", "solve", "solve", "fused"])
    if kind == "eos":
        c = _eos("", rng.choice([14, 86, 87]), _logint(rng, 1, 2000000))
    elif kind == "fused":
        c = {"name": "", "kind": "fused", "n": _logint(rng, 15, 6000), "steps": 1, "hints": rng.random() < 0.5,
             "cap": 2000}
    else:
        net, eos = rng.choice([14, 14, 86, 86, 87]), 0 if rng.random() < 0.25 else 1
        steps = rng.choice([1, 1, 2])
        cap = rng.choice([2000, 2000, 10000]) if steps == 1 else 2000
        hi = {14: 30000, 86: 200000, 87: 4000}[net] // steps
        if net == 87 and cap == 10000:
            hi = 2000
        c = _solve("", net, _logint(rng, 16, hi), eos=eos, mixed=rng.random() < 0.25, steps=steps,
                   hints=steps > 1 and rng.random() < 0.7, drhodt=rng.choice([0, 0, 0, 1, 2]), cap=cap)
    c.pop("name")
    return c


_contexts = {}


def _context():
    """One context per process, as a hydro program keeps it (tables uploaded once)."""
    if "ctx" not in _contexts:
        _contexts["ctx"] = nm.Context(0, helm_table=TABLE)
    return _contexts["ctx"]


def _particles(net, eos, n, seed):
    """rho, temp and the occupied abundance rows {species: values} of n particles."""
    if eos == 1:
        if net != 86:
            c = workloads.config(2 if net == 14 else 4, n=n, seed=seed)
            return c["rho"], c["temp"], {s: c["Y"][s] for s in np.nonzero(c["Y"].any(axis=1))[0]}
        # workloads.config(3)'s distribution without its dense 86 x n host array
        rng = np.random.default_rng(seed)
        hot = rng.random(n) < 0.3
        u, v = rng.random(n), rng.random(n)
        rho = 10 ** np.where(hot, 7 + u * (math.log10(5e9) - 7), 4 + 3 * u)
        temp = 10 ** np.where(hot, math.log10(3e9) + v * math.log10(8 / 3), 8 + v)
        o = workloads.net14_species_order()
        return rho, temp, {int(o[1]): np.full(n, 0.3 / 12), int(o[2]): np.full(n, 0.6 / 16),
                           int(o[3]): np.full(n, 0.1 / 20)}
    rng = np.random.default_rng(seed)
    o = workloads.net14_species_order() if net != 14 else np.arange(14)
    rho = 10 ** rng.uniform(6, 9, n)
    temp = 10 ** rng.uniform(9, math.log10(6e9) if net == 14 else 9.7, n)
    rows = {int(o[1]): np.full(n, 0.5 / 12), int(o[2]): np.full(n, 0.5 / 16)}
    if net == 87:
        rows[86] = np.full(n, 0.5)
    return rho, temp, rows


def _up(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _group(net, eos, n, seed, mixed, hints, drhodt):
    rho, temp, rows = _particles(net, eos, n, seed)
    Y0 = torch.zeros((NSP[net], n), dtype=torch.float64, device=DEV)
    for s, v in rows.items():
        Y0[s].copy_(_up(v))
    first = {"Y": Y0, "temp": _up(temp), "dt": torch.full((n,), workloads.INITIAL_DT, dtype=torch.float64, device=DEV)}
    st = {k: v.clone() for k, v in first.items()}
    st["rho"] = _up(rho)
    if drhodt:
        # the previous hydro step's density, a few percent away (0: no previous density)
        rng = np.random.default_rng(seed + 1)
        rm1 = rho * (1 + 0.02 * rng.standard_normal(n))
        rm1[rng.random(n) < 0.1] = 0
        first["rho_m1"] = _up(rm1)
        st["rho_m1"] = first["rho_m1"].clone()
    st["status"] = torch.zeros(n, dtype=torch.uint8, device=DEV)
    for k in ("substeps", "newton", "fp64_solves"):
        st[k] = torch.zeros(n, dtype=torch.int32, device=DEV)
    if hints:
        st["cost_hint"] = st["newton"]
        if mixed:
            st["fp64_hint"] = st["fp64_solves"]
    Z = workloads.helmholtz_Z(net) if eos == 1 else None
    batch = _context().make_batch(net, st, eos=eos, mu=10.0, Z=Z,
                                  precision=nm.PRECISION_MIXED if mixed else nm.PRECISION_FP64)
    return {"first": first, "st": st, "batch": batch, "mixed": mixed, "hints": hints, "drhodt": drhodt}


def _eos_inputs(net, n, seed):
    """Burnt compositions (every species present), rho and temp over the sets' ranges."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s: torch.rand(s, generator=g, device=DEV, dtype=torch.float64)  # noqa: E731
    A = torch.tensor(workloads.mass_numbers(net), dtype=torch.float64, device=DEV)
    d = NSP[net]
    nuclei = min(d, 86)
    Y = torch.zeros((d, n), dtype=torch.float64, device=DEV)
    Y[:nuclei] = r(nuclei, n).square_()
    Y[:nuclei] /= Y[:nuclei].sum(0)
    Y[:nuclei] /= A[:nuclei, None]
    if net == 87:
        Y[86] = 0.45 + 0.05 * r(n)
    lo, hi, tlo, thi = {14: (1e5, 5e9, 5e8, 7e9), 86: (1e4, 5e9, 1e8, 8e9), 87: (1e7, 1e10, 2e9, 9e9)}[net]
    rho = 10 ** (math.log10(lo) + r(n) * math.log10(hi / lo))
    temp = 10 ** (math.log10(tlo) + r(n) * math.log10(thi / tlo))
    # net87's refresh runs over the 86 nuclei's charges and the electron's, as its solve does; the
    # charges of nuclei and electrons cancel there, so the refresh is given the nuclei alone
    Z = workloads.helmholtz_Z(net)[:nuclei]
    return Y[:nuclei], rho, temp, Z


def prepare(case, seed):
    ctx = _context()
    if case["kind"] == "eos":
        Y, rho, temp, Z = _eos_inputs(case["net"], case["n"], seed)
        out = {k: torch.zeros(case["n"], dtype=torch.float64, device=DEV) for k in ("u", "cv", "p", "c", "dpdT")}
        return {"kind": "eos", "ctx": ctx, "Z": Z, "Y": Y, "rho": rho, "temp": temp, "out": out}
    if case["kind"] == "fused":
        n87 = case["n"] // 5
        n14 = (case["n"] - n87) // 2
        groups = [_group(net, 1, n, seed + 7 * net, False, case["hints"], 0)
                  for net, n in ((14, n14), (86, case["n"] - n87 - n14), (87, n87)) if n > 0]
        hydro_dt, drhodt = 1e-5, 0
    else:
        groups = [_group(case["net"], case["eos"], case["n"], seed, case["mixed"], case["hints"], case["drhodt"])]
        hydro_dt, drhodt = HYDRO_DT[(case["net"], case["eos"])], case["drhodt"]
    return {"kind": "solve", "ctx": ctx, "groups": groups, "batches": [g["batch"] for g in groups],
            "hydro_dt": hydro_dt, "drhodt": drhodt, "steps": case["steps"], "cap": case["cap"]}


def run(state):
    stream = torch.cuda.current_stream().cuda_stream
    ctx = state["ctx"]
    if state["kind"] == "eos":
        ctx.helm_eos(state["Z"], state["temp"], state["rho"], state["Y"], state["out"], stream=stream, sync=False)
        return state["out"]
    for g in state["groups"]:
        for k, v in g["first"].items():
            g["st"][k].copy_(v)
        if g["hints"]:  # the first step has none
            g["st"]["newton"].zero_()
            if g["mixed"]:
                g["st"]["fp64_solves"].zero_()
    ctx.set_max_iterations(state["cap"])
    for _ in range(state["steps"]):
        ctx.compute(state["batches"], state["hydro_dt"], previous_dt=state["hydro_dt"], use_drhodt=state["drhodt"],
                    stream=stream, sync=False)
    keys = ["Y", "temp", "dt", "status", "substeps", "newton"]
    return [{k: g["st"][k] for k in keys + (["fp64_solves"] if g["mixed"] else []) +
             (["rho_m1"] if g["drhodt"] else [])} for g in state["groups"]]


def _newton_flops(net):
    """One Newton iteration: dense unpivoted LU and solve of n = d + 1 unknowns, and the assembly."""
    d = NSP[net]
    n = d + 1
    return 2 * n ** 3 / 3 + 1.5 * n ** 2 - 7 * n / 6 + 3 * d ** 2


def work(case):
    if case["kind"] == "eos":
        d = min(NSP[case["net"]], 86)
        return {"bytes": 8.0 * (d + 7) * case["n"], "flops": 900.0 * case["n"]}
    n87 = case["n"] // 5
    n14 = (case["n"] - n87) // 2
    parts = ([(14, 1, n14), (86, 1, case["n"] - n87 - n14), (87, 1, n87)] if case["kind"] == "fused"
             else [(case["net"], case["eos"], case["n"])])
    b = f = 0.0
    for net, eos, n in parts:
        b += case["steps"] * n * (8.0 * (2 * NSP[net] + 5) + 9)
        f += case["steps"] * n * NEWTON[(net, eos)] * min(1.0, case["cap"] / 10000) ** 0.7 * _newton_flops(net)
    return {"bytes": b, "flops": f}


# ---- what the EOS refresh returns, in plain torch at 64 bits -----------------------------------
# Helmholtz EOS of Timmes & Swesty (ApJS 126, 501, 2000): radiation, ideal ions, the
# electron-positron Helmholtz free energy by biquintic Hermite interpolation of the table, its
# dP/drho by bicubic interpolation, and the uniform-background Coulomb corrections of Yakovlev &
# Shalybkov (1989).


def _hermite(z, order):
    """Quintic Hermite basis (value, first and second derivative at the left node) and its
    `order`-th derivative at z, as columns (p0, p1, p2)."""
    if order == 0:
        return (1 + z ** 3 * (-10 + z * (15 - 6 * z)), z * (1 + z ** 2 * (-6 + z * (8 - 3 * z))),
                0.5 * z ** 2 * (1 + z * (-3 + z * (3 - z))))
    if order == 1:
        return (z ** 2 * (-30 + z * (60 - 30 * z)), 1 + z ** 2 * (-18 + z * (32 - 15 * z)),
                0.5 * z * (2 + z * (-9 + z * (12 - 5 * z))))
    return (z * (-60 + z * (180 - 120 * z)), z * (-36 + z * (96 - 60 * z)), 0.5 * (2 + z * (-18 + z * (36 - 20 * z))))


def _basis(x, h, order):
    """Weights [node][derivative] of a cell of width h at x in [0, 1], differentiated `order` times."""
    l, r = _hermite(x, order), _hermite(1 - x, order)
    s = (-1.0) ** order
    return ([l[k] * h ** (k - order) for k in range(3)],
            [s * (-1.0) ** k * r[k] * h ** (k - order) for k in range(3)])


def exact(case, seed):
    if case["kind"] != "eos":
        return None  # a hydro step is thousands of dependent implicit solves: minutes in plain torch
    Y, rho, T, Z = _eos_inputs(case["net"], case["n"], seed)
    f64 = dict(dtype=torch.float64, device=DEV)
    tab = torch.from_numpy(np.fromfile(TABLE, dtype=np.float64).reshape(21, 541, 201)).to(DEV)
    ytot = Y.sum(0)
    zsum = (Y * torch.tensor(Z, **f64)[:, None]).sum(0)
    del Y
    zbar, ye = zsum / ytot, zsum.clamp_min(1e-16)
    din = ye * rho
    dl, tl = 27.0 / 540, 10.0 / 200
    j = ((torch.log10(T) - 3) / tl).long().clamp(1, 199)
    i = ((torch.log10(din) + 12) / dl).long().clamp(1, 539)
    tg, dg = 10 ** (3 + tl * torch.arange(201, **f64)), 10 ** (-12 + dl * torch.arange(541, **f64))
    ht, hd = tg[j + 1] - tg[j], dg[i + 1] - dg[i]
    xt, xd = ((T - tg[j]) / ht).clamp_min(0), ((din - dg[i]) / hd).clamp_min(0)
    bt, bd = [_basis(xt, ht, k) for k in range(3)], [_basis(xd, hd, k) for k in range(2)]
    index = {(0, 0): 0, (1, 0): 1, (0, 1): 2, (2, 0): 3, (0, 2): 4, (1, 1): 5, (2, 1): 6, (1, 2): 7, (2, 2): 8}
    F = {k: torch.zeros_like(T) for k in ((0, 0), (1, 0), (0, 1), (0, 2), (1, 1))}
    for (kd, kt), q in index.items():
        for a in (0, 1):
            for b in (0, 1):
                v = tab[q, i + a, j + b]
                for (od, ot), acc in F.items():
                    acc += v * bd[od][a][kd] * bt[ot][b][kt]
    c3 = lambda z: (z ** 2 * (2 * z - 3) + 1, z * (z * (z - 2) + 1))  # noqa: E731
    ct = [[c3(xt)[0], c3(xt)[1] * ht], [c3(1 - xt)[0], -c3(1 - xt)[1] * ht]]
    cd = [[c3(xd)[0], c3(xd)[1] * hd], [c3(1 - xd)[0], -c3(1 - xd)[1] * hd]]
    dpdd_e = torch.zeros_like(T)
    for (kd, kt), q in {(0, 0): 9, (1, 0): 10, (0, 1): 11, (1, 1): 12}.items():
        for a in (0, 1):
            for b in (0, 1):
                dpdd_e += tab[q, i + a, j + b] * cd[a][kd] * ct[b][kt]
    dpdd_e = (ye * dpdd_e).clamp_min(1e-30)
    avo, clight, kerg, ssol, qe = 6.0221417930e23, 2.99792458e10, 1.380650424e-16, 5.6704e-5, 4.8032042712e-10
    asol, kt = 4 * ssol / clight, kerg * T
    prad = asol * T ** 4 / 3
    dprad, erad = 4 * prad / T, 3 * prad / rho
    derad = 3 * dprad / rho
    xni = avo * ytot * rho
    pion, dpion_d, dpion_t = xni * kt, avo * ytot * kt, xni * kerg
    eion, deion_t = 1.5 * pion / rho, 1.5 * dpion_t / rho
    pele, dpele_t = din ** 2 * F[(1, 0)], din ** 2 * F[(1, 1)]
    eele, deele_t = ye * F[(0, 0)] - T * ye * F[(0, 1)], -T * ye * F[(0, 2)]
    s = math.pi * 4 / 3 * xni
    lam = s ** (-1 / 3)
    gam = zbar ** 2 * qe ** 2 / kt / lam
    gam_d, gam_t = gam / rho / 3, -gam / T
    a1, b1, c1, d1, a2, b2, c2 = -0.898004, 0.96786, 0.220703, -0.86097, 0.29561, 1.9885, 0.288675
    x = gam ** 0.25
    e_s = avo * ytot * kerg * T * (a1 * gam + b1 * x + c1 / x + d1)
    y = avo * ytot * kt * (a1 + 0.25 / gam * (b1 * x - c1 / x))
    de_d, de_t = y * gam_d, y * gam_t + e_s / T
    p_s, dp_d_s, dp_t_s = rho * e_s / 3, e_s + rho / 3 * de_d / 3, rho / 3 * de_t
    x, y = gam * gam.sqrt(), gam ** b2
    w = c2 * x - a2 * y / 3
    p_w = -pion * w
    e_w = 3 * p_w / rho
    dw = 1.5 * c2 * x / gam - a2 * b2 * y / gam / 3
    dp_d_w, dp_t_w = -dpion_d * w - pion * dw * gam_d, -dpion_t * w - pion * dw * gam_t
    strong = gam >= 1
    pick = lambda u, v: torch.where(strong, u, v)  # noqa: E731
    pc, ec, dpc_d, dpc_t, dec_t = (pick(p_s, p_w), pick(e_s, e_w), pick(dp_d_s, dp_d_w), pick(dp_t_s, dp_t_w),
                                   pick(de_t, 3 / rho * dp_t_w))
    bad = (prad + pion + pele + pc <= 0) | (erad + eion + eele + ec <= 0)
    pc, ec, dpc_d, dpc_t, dec_t = (torch.where(bad, torch.zeros_like(v), v) for v in (pc, ec, dpc_d, dpc_t, dec_t))
    pres, ener = prad + pion + pele + pc, erad + eion + eele + ec
    dpdT, cv = dprad + dpion_t + dpele_t + dpc_t, derad + deion_t + deele_t + dec_t
    dpdd = dpion_d + dpdd_e + dpc_d
    chit, chid = T / pres * dpdT, dpdd * rho / pres
    gam1 = chit * (pres / rho * chit / (T * cv)) + chid
    c = clight * torch.sqrt(gam1 / (1 + (ener + clight ** 2) * rho / pres))
    return {"u": ener, "cv": cv, "p": pres, "c": c, "dpdT": dpdT}
