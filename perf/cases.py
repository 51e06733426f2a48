"""The calls whose speed is measured, over the range that callers use.

One time step of a reacting-flow solver on this library integrates the
chemistry of every cell (plain, or by the guided solve with the tuned options),
evaluates the transport properties of the ghosted block and forms the
molar-diffusion correction; a caller with an integrator of its own asks for
right-hand sides and production rates of many states; the network of the
surrogate is trained on mini-batches and evaluated over whole blocks.  Blocks
run from a single small patch to 128^3, with odd extents, ghost layers, wall
rows and all four mechanisms.

``listed()`` holds the fixed cases, ``draw(rng)`` one more of the same ranges;
``prepare`` makes the fields on the GPU from a seed (the distributions of
tiger_nga_amd/inputs.py), ``run`` makes one call.  The chemistry step advances
its fields in place and the transport-source update adds to its array, so
``run`` first copies the fields that the transport step would have produced
into the working arrays.  ``exact`` is the same quantity in plain torch in 64
bits from the mechanism's generated tables.
"""
import functools
import json
import math
import os
import re

import numpy as np
import torch

from tiger_nga_amd import autotune, flops, inputs, metric, mlp
from tiger_nga_amd.finitechem import FiniteChem, Grid
from tiger_nga_amd.mech import meta

R_CST = 8314.34  # finitechem.f90:15
R_F4 = float(np.float32(8314.34))  # the mechanism files' binary32 literal
MECHS = ("h2", "gri30", "dme39", "ethyred")
WORKLOAD = {"h2": "h2", "gri30": "gri30_uneven", "dme39": "dme39", "ethyred": "ethyred"}
FUEL = {"gri30": ("CH4", 1, 4, 2.0, 0), "dme39": ("CH3OCH3", 2, 6, 3.0, 1), "ethyred": ("C2H4", 2, 4, 3.0, 0)}

# Mean operation counts of one cell over one step of the states below, from the
# solver's own counters (tiger_nga_amd.flops.step_flops / guided_flops).
STEP_FLOPS = {"h2": 0.505e6, "gri30": 9.1e6, "dme39": 19.9e6, "ethyred": 10.6e6}
GUIDED_FLOPS = {"h2": 0.507e6, "gri30": 5.5e6, "dme39": 13.1e6, "ethyred": 4.34e6}


def listed():
    return [
        # a handful of cells, as in a patch that holds little chemistry: latency of one cell's serial integration
        {"name": "step_h2_64cells", "kind": "step", "mech": "h2", "nx": 4, "ny": 4, "nz": 4, "nover": 0, "wall": False,
         "host": False, "guided": False},
        # the drop-in call of a Fortran host: host arrays with ghost layers and a wall row, odd extents
        {"name": "step_gri30_host", "kind": "step", "mech": "gri30", "nx": 21, "ny": 18, "nz": 17, "nover": 2,
         "wall": True, "host": True, "guided": False},
        # the mechanism that the reference links by default, fields resident on the GPU
        {"name": "step_ethyred", "kind": "step", "mech": "ethyred", "nx": 40, "ny": 33, "nz": 29, "nover": 1,
         "wall": False, "host": False, "guided": False},
        # the main path: the guided step on a large block of unevenly stiff GRI-3.0 cells
        {"name": "guided_gri30", "kind": "step", "mech": "gri30", "nx": 96, "ny": 80, "nz": 64, "nover": 0,
         "wall": False, "host": False, "guided": True},
        # the same on a smaller odd block at 10 atm, where some cells fall back to the plain step
        {"name": "guided_dme39", "kind": "step", "mech": "dme39", "nx": 31, "ny": 29, "nz": 37, "nover": 1,
         "wall": True, "host": False, "guided": True},
        # right-hand sides of a block's states for a caller's own integrator
        {"name": "rhs_gri30_64cubed", "kind": "rhs", "mech": "gri30", "n": 262144},
        # production rates of an odd number of states
        {"name": "prodrates_ethyred", "kind": "prodrates", "mech": "ethyred", "n": 100003},
        # density, viscosity and diffusivities of the whole ghosted block, every flow step
        {"name": "properties_gri30_128cubed", "kind": "properties", "mech": "gri30", "nx": 128, "ny": 128, "nz": 128,
         "nover": 1, "wall": False, "lewis": False},
        # the molar-diffusion correction of the same block, the default second-order stencil
        {"name": "diffusion_gri30_128cubed", "kind": "diffusion", "mech": "gri30", "nx": 128, "ny": 128, "nz": 128,
         "nover": 1, "order": 2, "molar": True, "gasrad": False, "cv": False, "wall": False, "src": False},
        # fourth order on an odd block with walls, gas radiation and the transport-source update
        {"name": "diffusion_dme39_order4", "kind": "diffusion", "mech": "dme39", "nx": 61, "ny": 47, "nz": 35,
         "nover": 3, "order": 4, "molar": True, "gasrad": True, "cv": True, "wall": True, "src": True},
        # training of the network: Adam steps on mini-batches, the parameters read back at the end
        {"name": "train_gri30_4096", "kind": "train", "mech": "gri30", "rows": 4096, "hidden": 256, "layers": 4,
         "steps": 8},
        # the network over a whole 64^3 block
        {"name": "infer_gri30_64cubed", "kind": "infer", "mech": "gri30", "rows": 262144, "hidden": 256, "layers": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extents(rng, lo, hi):
    """Three extents, odd ones among them, whose product is log-uniform in [lo, hi]."""
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    a, b = rng.uniform(0.7, 1.4), rng.uniform(0.7, 1.4)
    e = n ** (1.0 / 3.0)
    ext = [max(2, int(round(e * f))) for f in (a, b, 1.0 / (a * b))]
    while ext[0] * ext[1] * ext[2] > hi:
        ext[ext.index(max(ext))] -= 1
    return dict(zip(("nx", "ny", "nz"), ext))


def draw(rng):
    kind = rng.choice(("step", "step", "guided", "rhs", "prodrates", "properties", "diffusion", "diffusion", "train",
                       "infer"))
    mech = rng.choice(MECHS)
    if kind in ("step", "guided"):
        ext = _extents(rng, 8, 20000) if kind == "step" else _extents(rng, 4000, 65536)
        return {"kind": "step", "mech": mech, **ext, "nover": rng.choice((0, 1, 2)), "wall": rng.random() < 0.4,
                "host": kind == "step" and rng.random() < 0.3, "guided": kind == "guided"}
    if kind in ("rhs", "prodrates"):
        return {"kind": kind, "mech": mech, "n": _log_int(rng, 1, 262144)}
    if kind == "properties":
        return {"kind": kind, "mech": mech, **_extents(rng, 512, 1500000), "nover": rng.choice((1, 2, 3)),
                "wall": rng.random() < 0.4, "lewis": rng.random() < 0.5}
    if kind == "diffusion":
        order = rng.choice((2, 2, 4))
        return {"kind": kind, "mech": mech, **_extents(rng, 512, 1500000 if order == 2 else 150000),
                "nover": {2: rng.choice((1, 2)), 4: 3}[order], "order": order, "molar": rng.random() < 0.8,
                "gasrad": rng.random() < 0.4, "cv": rng.random() < 0.4, "wall": rng.random() < 0.4,
                "src": rng.random() < 0.4}
    net = {"mech": mech, "hidden": rng.choice((128, 256, 256)), "layers": rng.choice((2, 3, 4, 4))}
    if kind == "train":
        return {"kind": kind, **net, "rows": 64 * _log_int(rng, 2, 128), "steps": rng.choice((4, 6, 8))}
    return {"kind": kind, **net, "rows": 64 * _log_int(rng, 1, 4096)}


# ---- inputs --------------------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _random(gen, n):
    """Independent uniform numbers per cell."""
    return lambda lo, hi: lo + (hi - lo) * torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)


def _smooth(gen, sh):
    """Smooth fields in [lo, hi] over a block of extents sh (flattened, i fastest): three long waves."""
    ax = [torch.arange(s, device="cuda", dtype=torch.float64) / max(8, s) for s in sh]

    def field(lo, hi):
        p = torch.rand(12, generator=gen, device="cuda", dtype=torch.float64).tolist()
        f = torch.zeros(sh[2], sh[1], sh[0], device="cuda", dtype=torch.float64)
        for w in range(3):
            ph = [2 * math.pi * (0.5 + p[4 * w + d]) * ax[d] for d in range(3)]
            f += torch.sin(ph[0][None, None, :] + ph[1][None, :, None] + ph[2][:, None, None] + 6.2 * p[4 * w + 3])
        return (lo + (hi - lo) * (0.5 + f / 6.0)).reshape(-1)
    return field


def _states(mech, n, u):
    """(Y[nsp, n], T[n], rho[n], P): the states of tiger_nga_amd/inputs.py, u(lo, hi) giving n numbers of that range."""
    _, _, P, _ = inputs.WORKLOADS[WORKLOAD[mech]]
    sp = meta.species(mech)
    W = torch.tensor(meta.molar_mass(mech), device="cuda", dtype=torch.float64)
    at = sp.index
    Y = torch.zeros(len(sp), n, device="cuda", dtype=torch.float64)
    fuel, nC, nH, o2, oF = FUEL.get(mech, ("H2", 0, 2, 0.5, 0))
    Z = u(0.0, 1.0 if mech == "h2" else 0.15)
    Y[at(fuel)] = Z
    Y[at("O2")] = 0.233 * (1 - Z)
    Y[at("N2")] = 0.767 * (1 - Z)
    if mech == "gri30":  # 70 % near equilibrium, 20 % at an ignition front, 10 % cold
        v = u(0.0, 1.0)
        c = torch.where(v < 0.7, u(0.9, 1.0), torch.where(v < 0.9, u(0.05, 0.2), u(0.0, 0.05)))
        T = torch.where(v < 0.7, u(1800.0, 2300.0), torch.where(v < 0.9, u(1000.0, 1300.0), u(300.0, 600.0)))
    else:
        c = u(0.0, 1.0)
        T = u(*{"h2": (900.0, 2200.0), "dme39": (600.0, 2200.0), "ethyred": (800.0, 2400.0)}[mech])
    xi = c * torch.minimum(Y[at(fuel)] / W[at(fuel)], Y[at("O2")] / W[at("O2")] / o2)
    burnt = {"H2O": 0.5 * nH * xi}
    if nC:
        burnt = {"CO2": 0.9 * nC * xi, "CO": 0.1 * nC * xi, "H2O": 0.475 * nH * xi, "H2": 0.025 * nH * xi}
    used = 0.5 * (2 * burnt.get("CO2", 0.0) + burnt.get("CO", 0.0) + burnt["H2O"] - oF * xi)
    Y[at(fuel)] -= xi * W[at(fuel)]
    Y[at("O2")] -= used * W[at("O2")]
    for s, mol in burnt.items():
        if s in sp:
            Y[at(s)] += mol * W[at(s)]
    for k, s in enumerate(sp):
        if s not in ("N2", "O2", "H2", "H2O", "CO", "CO2", fuel):
            Y[k] = 10.0 ** (u(-6.0, -3.0) if mech == "h2" else u(-8.0, -3.0))
    Y = Y.clamp_min(0.0)
    Y /= Y.sum(dim=0)
    return Y, T, P / (R_CST * T * (Y / W[:, None]).sum(dim=0)), P


def _fortran(planes, sh):
    """planes[..., cells (i fastest)] as a Fortran-ordered tensor sh (+ planes)."""
    t = planes.reshape(planes.shape[:-1] + (sh[2], sh[1], sh[0]))
    return t.permute(2, 1, 0) if planes.dim() == 1 else t.permute(3, 2, 1, 0)


def _zeros(sh, nplane=None):
    return _fortran(torch.zeros((() if nplane is None else (nplane,)) + (sh[0] * sh[1] * sh[2],), device="cuda",
                                dtype=torch.float64), sh)


def _wall(g):
    """mask of the block's array with a wall row along i (1 = wall)."""
    ny = g.jmax_ - g.jmin_ + 1
    m = torch.zeros(g.mask_shape[1], g.mask_shape[0], dtype=torch.int32, device="cuda")
    m[g.jmin_ - g.jmino_ + ny // 2, :] = 1
    return m.t()


def _block(case, seed, smooth):
    """(grid, RHO_, SC_, mask, P, dt) of a block; species first, then T, then one passive scalar."""
    nsp = len(meta.species(case["mech"]))
    g = Grid.block(case["nx"], case["ny"], case["nz"], nsp + 2, 1, nsp + 1, nover=case["nover"])
    sh = g.shape
    gen = _gen(seed)
    n = sh[0] * sh[1] * sh[2]
    Y, T, rho, P = _states(case["mech"], n, _smooth(gen, sh) if smooth else _random(gen, n))
    SC_ = _fortran(torch.cat([Y, T[None], torch.full_like(T, 0.3)[None]]), sh)
    dt = inputs.WORKLOADS[WORKLOAD[case["mech"]]][3]
    return g, _fortran(rho, sh), SC_, _wall(g) if case["wall"] else None, P, dt


def _diffusion_inputs(case, seed):
    g, rho, SC_, mask, P, dt = _block(case, seed, True)
    rng = np.random.default_rng(seed)
    faces = [1e-4 * np.cumsum(np.concatenate([[0.0], 1.0 + 0.3 * rng.random(s)])) for s in g.shape[:2]]
    m = metric.cartesian(g, faces[0], faces[1], 1.1e-4, case["order"])
    # rho D of each species and lambda / cp: 2e-5 (T / 300)^0.7 over a Lewis number per scalar
    lew = torch.tensor(rng.uniform(0.3, 1.8, g.nscalar), device="cuda")
    T = SC_[..., g.isc_T - 1]
    D = _zeros(g.shape, g.nscalar)
    for s in range(g.nscalar):
        D[..., s] = 2e-5 * (T / 300.0) ** 0.7 / lew[s]
    return g, m, rho, SC_, D, mask, dt


def _net_inputs(case, seed):
    """Parameters, standardised inputs (bfloat16, padded columns 0) and targets."""
    nsp = len(meta.species(case["mech"]))
    nin, nout = nsp + 2, nsp + 1
    gen = _gen(seed)
    x = torch.zeros(case["rows"], (nin + 63) // 64 * 64, device="cuda", dtype=torch.bfloat16)
    x[:, :nin] = torch.randn(case["rows"], nin, generator=gen, device="cuda").to(torch.bfloat16)
    P = torch.randn(nin, nout, generator=gen, device="cuda") / math.sqrt(nin)
    tgt = torch.tanh(x[:, :nin].float() @ P).contiguous()
    return nin, nout, mlp.init_params(nin, nout, case["hidden"], case["layers"], seed=seed), x, tgt


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("train", "infer"):
        nin, nout, flat, x, tgt = _net_inputs(case, seed)
        net = mlp.MLP(nin, nout, case["hidden"], case["layers"])
        net.set_params(flat)
        return {"case": case, "net": net, "x": x, "tgt": tgt}
    fc = FiniteChem(case["mech"])
    if kind in ("rhs", "prodrates"):
        Y, T, rho, P = _states(case["mech"], case["n"], _random(_gen(seed), case["n"]))
        if kind == "rhs":
            return {"case": case, "fc": fc, "sol": torch.cat([rho * Y, (rho * T)[None]]).contiguous(), "P": P}
        C = rho * Y / torch.tensor(fc.molar_mass, device="cuda")[:, None]
        return {"case": case, "fc": fc, "C": C.contiguous(), "T": T, "P": torch.full_like(T, P)}
    if kind == "diffusion":
        g, m, rho, SC_, D, mask, dt = _diffusion_inputs(case, seed)
        md = {k: v if k in ("st1", "st2") else torch.from_numpy(v.ravel(order="F").copy()).cuda() for k, v in m.items()}
        st = {"case": case, "fc": fc, "g": g, "m": md, "rho": rho, "sc": SC_, "D": D, "mask": mask, "dt": dt,
              "corr": _zeros(g.shape, fc.nsp + 1), "gp": _zeros(g.shape, 3), "src": None}
        if case["src"]:
            st["src0"] = _zeros(g.shape, g.nscalar) + 1e-7
            st["src"] = st["src0"].clone()
        return st
    g, rho, SC_, mask, P, dt = _block(case, seed, False)
    st = {"case": case, "fc": fc, "g": g, "rho": rho, "sc": SC_, "mask": mask, "P": P, "dt": dt}
    if kind == "properties":
        st["lewis"] = 0.5 + torch.rand(fc.nsp, generator=_gen(seed + 1), device="cuda",
                                       dtype=torch.float64) if case["lewis"] else None
        st["out"] = {"RHO_": _zeros(g.shape), "VISC_": _zeros(g.shape), "DIFF_": _zeros(g.shape, g.nscalar)}
        return st
    if case["guided"]:
        autotune.apply(fc, case["nx"] * case["ny"] * case["nz"])
        fc.load_surrogate(os.path.join(os.path.dirname(meta.__file__), "..", "models", case["mech"] + ".bin"))
    st.update({"sc0": SC_, "sc": SC_.clone(), "hr": _zeros(g.shape), "src": _zeros(g.shape, 3)})
    if case["host"]:
        for k in ("rho", "sc0", "sc", "hr", "src", "mask"):
            if st[k] is not None:
                st[k] = np.asfortranarray(st[k].cpu().numpy())
    return st


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "train":
        net, k = state["net"], case["steps"]
        for it in range(k):
            loss = net.train_step(state["x"], state["tgt"], 1e-3, want_loss=it == k - 1)
        return {"loss": loss, "params": net.get_params()}
    if kind == "infer":
        return state["net"].forward(state["x"])
    fc = state["fc"]
    if kind == "rhs":
        return fc.compute_rhs(state["sol"], state["P"])
    if kind == "prodrates":
        return fc.prodrates(state["C"], state["T"], state["P"])
    g = state["g"]
    if kind == "properties":
        fc.properties(state["sc"], g, state["P"], mask=state["mask"], Lewis=state["lewis"], **state["out"])
        return state["out"]
    if kind == "diffusion":
        if case["src"]:
            state["src"].copy_(state["src0"])
        fc.diffusion(state["dt"], g, state["m"], state["rho"], state["sc"], state["D"], mask=state["mask"],
                     diff_corr=state["corr"], diff_gp=state["gp"], src=state["src"], molar=case["molar"],
                     gasrad=case["gasrad"], cv=case["cv"])
        return {"corr": state["corr"], "gp": state["gp"], "src": state["src"]}
    if case["host"]:
        np.copyto(state["sc"], state["sc0"])
    else:
        state["sc"].copy_(state["sc0"])
    step = fc.source_chemistry_surrogate if case["guided"] else fc.source_chemistry
    step(state["rho"], state["sc"], g, state["dt"], state["P"], mask=state["mask"], HR_gp=state["hr"],
         chemsrc_gp=state["src"], sync=False)
    return {"sc": state["sc"], "hr": state["hr"], "src": state["src"]}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _info(mech):
    """Table sizes of a mechanism as tiger_nga_amd.flops takes them."""
    d = _data(mech)
    rx = d["rx"]
    fo, rev = [r for r in rx if r["kind"] == 2], [r for r in rx if r["rev"]]
    return {"nsp": len(d["species"]), "nrxn": len(rx), "n_reversible": len(rev), "n_falloff": len(fo),
            "n_rev_falloff": sum(r["rev"] for r in fo), "n_fc_terms": sum(len(r["fc"]) for r in fo),
            "n_third_body_rxn": sum(r["kind"] == 1 for r in rx), "n_nu": sum(len(r["nu"]) for r in rx),
            "n_conc_factors": sum(len(r["reac"]) for r in rx) + sum(len(r["prod"]) for r in rev),
            "n_eff_corr": sum(e != 1.0 for row in d["eff"] for e in row)}


def work(case):
    kind, mech = case["kind"], case["mech"]
    if kind in ("train", "infer"):
        nsp = len(meta.species(mech))
        nw = (nsp + 2) * case["hidden"] + (case["layers"] - 1) * case["hidden"] ** 2 + case["hidden"] * (nsp + 1)
        rows = case["rows"]
        if kind == "infer":
            return {"bytes": rows * (2 * (nsp + 2) + 4 * (nsp + 1)) + 2 * nw, "flops": 2.0 * rows * nw}
        per = rows * (2 * (nsp + 2) + 4 * (nsp + 1)) + 26 * nw  # Adam: read p, m, v, write them and the bf16 copy
        return {"bytes": case["steps"] * per, "flops": 6.0 * case["steps"] * rows * nw}
    nsp = len(meta.species(mech))
    if kind in ("rhs", "prodrates"):
        f = flops.rhs_flops(_info(mech))
        if kind == "prodrates":
            f -= nsp * 24 + 2
        return {"bytes": 8 * case["n"] * (2 * nsp + 2), "flops": f * case["n"]}
    no = 2 * case["nover"]
    cells = case["nx"] * case["ny"] * case["nz"]
    if kind == "properties":
        cells = (case["nx"] + no) * (case["ny"] + no) * (case["nz"] + no)
        return {"bytes": 8 * cells * (nsp + 1 + nsp + 3), "flops": cells * flops.properties_flops(nsp)}
    if kind == "diffusion":
        return {"bytes": flops.diffusion_bytes(nsp, cells) + (16 * cells * (nsp + 1) if case["src"] else 0),
                "flops": cells * nsp * 80.0}
    if case["wall"]:
        cells -= case["nx"] * case["nz"]
    return {"bytes": flops.step_bytes({"nsp": nsp}, cells),
            "flops": cells * (GUIDED_FLOPS if case["guided"] else STEP_FLOPS)[mech]}


def tolerance(case):
    kind = case["kind"]
    # the networks: hidden units in another order (sums over K in another order) moved the outputs by 2.2e-4 (largest
    # 0.021) and the trained parameters by 1.6e-4 (0.017): a bf16 activation that rounds the other way
    if kind == "train":
        return {"rel": 7e-4, "max": 0.08}
    if kind == "infer":
        return {"rel": 1e-3, "max": 0.1}
    # inputs off by one unit in the last place change step sequences: sources, differences over dt, moved by 9.6e-7
    # (largest 1.4e-4) in the guided step, by 4.2e-7 (5.6e-6) in the plain one
    if kind == "step":
        return {"rel": 4e-6, "max": 6e-4} if case["guided"] else {"rel": 2e-6, "max": 3e-5}
    # against exact(): 1.4e-14 (3.9e-13) for the divergence of fluxes, 4.5e-16 (2.5e-15) for the properties, 3.6e-15
    # (2.6e-14) for the rates
    if kind == "diffusion":
        return {"rel": 6e-14, "max": 2e-12}
    return {"rel": 2e-15, "max": 1e-14} if kind == "properties" else {"rel": 1.5e-14, "max": 1e-13}


# ---- the same quantities in plain torch, 64 bits ----------------------------------------------------------------------

@functools.lru_cache(maxsize=None)
def _data(mech):
    """The mechanism's numbers, from its generated tables (layout: tiger_nga_amd/csrc/mech_tables.h)."""
    with open(os.path.join(os.path.dirname(meta.__file__), "..", "csrc", "mech_%s.h" % mech)) as f:
        text = f.read()

    def table(name):
        body = re.search(r"%s_%s(?:\[\d+\])+ = (\{.*?\});" % (mech, name), text, re.S).group(1)
        body = re.sub(r"-?0x[0-9a-f.]+p[+-]\d+", lambda m: repr(float.fromhex(m.group())), body)
        return json.loads(body.replace("{", "[").replace("}", "]"))
    th, nu = table("thermo"), table("nu")
    nsp = len(th) // 2
    rx = []
    for (kind, rev, m, nr, npr, nfc, reac, prod, nu0, nnu, _, _, _, f, b, f0, b0, fc, fk, fd) in table("rxn"):
        rx.append({"kind": kind, "rev": bool(rev), "m": m, "reac": reac[:nr], "prod": prod[:npr], "f": f, "b": b,
                   "f0": f0, "b0": b0, "nu": nu[nu0:nu0 + nnu], "fc": list(zip(fc, fk, fd))[:nfc]})
    tmid = float.fromhex(re.search(r"%s_tables = \{[^}]*?(0x[0-9a-f.]+p[+-]\d+)" % mech, text).group(1))
    return {"species": meta.species(mech), "W": table("W"), "mu": table("mucoeff"), "koe": table("koveps"),
            "eff": table("eff"), "rx": rx, "thermo": {"hi": th[:nsp], "lo": th[nsp:]}, "tmid": tmid}


def _t(a, dtype=torch.float64):
    return torch.tensor(a, device="cuda", dtype=dtype)


@functools.lru_cache(maxsize=None)
def _tables(mech):
    d = _data(mech)
    rx = d["rx"]
    nsp = len(d["species"])

    def slots(key):
        return _t([(([] if key == "prod" and not r["rev"] else r[key]) + [nsp] * 3)[:3] for r in rx]).long()
    nu = torch.zeros(nsp, len(rx), device="cuda", dtype=torch.float64)
    for i, r in enumerate(rx):
        for k, v in r["nu"]:
            nu[k, i] += v
    th = {r: [_t(d["thermo"][r])[:, c, None] for c in (slice(0, 7), slice(7, 13))] for r in ("hi", "lo")}
    return {"W": _t(d["W"])[:, None], "eff": _t(d["eff"]), "nu": nu, "reac": slots("reac"), "prod": slots("prod"),
            **{q: [_t([r[q][c] for r in rx])[:, None] for c in range(3)] for q in ("f", "b", "f0", "b0")},
            "rev": _t([float(r["rev"]) for r in rx])[:, None],
            "mw": _t([r["m"] if r["kind"] == 1 else len(d["eff"]) for r in rx]).long(),
            "rx": rx, "tmid": d["tmid"], "th": th, "mu": _t(d["mu"])[:, None], "koe": _t(d["koe"])[:, None],
            "species": d["species"]}


def _thermo(t, T):
    """h[nsp, n], cp[nsp, n] (COMPTHERMODATA, HYDROGENF.f90:514-673)."""
    out = []
    for q in range(2):
        c = torch.where(T[None, None, :] > t["tmid"], t["th"]["hi"][q], t["th"]["lo"][q])
        p = c[:, 1] + T * (c[:, 2] + T * (c[:, 3] + T * (c[:, 4] + T * c[:, 5])))
        out.append(c[:, 0] * (T * p + c[:, 6]) if q == 0 else c[:, 0] * p)
    return out


def _prodrates(mech, C, T, P):
    """CDOT[nsp, n] (PRODRATES / GETLINDRATECOEFF, HYDROGENF.f90:4-316)."""
    t = _tables(mech)
    lt, rt = T.log(), R_F4 * T
    one = torch.ones_like(T)[None]
    M = torch.cat([t["eff"] @ C, one])
    k = {q: t[q][0] * torch.exp(t[q][1] * lt + t[q][2] / rt) for q in ("f", "b", "f0", "b0")}
    c32 = lambda v: float(np.float32(v))
    for i, r in enumerate(t["rx"]):
        if r["kind"] != 2:
            continue
        conc = M[r["m"]] if r["m"] >= 0 else torch.zeros_like(T)
        conc = torch.where(conc > 0, conc, P / rt)
        fc = sum(c * torch.exp(-(d / T) if q == 1 else -(T / d)) for c, q, d in r["fc"])
        lf = fc.log10()
        for q in ("f", "b") if r["rev"] else ("f",):
            kinf = k[q][i]
            pr = k[q + "0"][i] * conc / kinf.clamp_min(1e-60)
            lg = pr.log10() - c32(0.4) - c32(0.67) * lf
            x = lg / (0.75 - c32(1.27) * lf - c32(0.14) * lg)
            k[q][i] = kinf * fc ** (1 / (x * x + 1)) * pr / (1 + pr)
    c1 = torch.cat([C, one])
    q = k["f"] * c1[t["reac"][:, 0]] * c1[t["reac"][:, 1]] * c1[t["reac"][:, 2]]
    q -= t["rev"] * k["b"] * c1[t["prod"][:, 0]] * c1[t["prod"][:, 1]] * c1[t["prod"][:, 2]]
    q *= M[t["mw"]]
    return t["nu"] @ q


def _rhs(mech, sol, P):
    """finitechem_compute_rhs (finitechem.f90:93-175) of sol[neq, n]."""
    t = _tables(mech)
    rho = sol[:-1].sum(dim=0)
    T = sol[-1] / rho
    h, cp = _thermo(t, T)
    r = _prodrates(mech, sol[:-1] / t["W"], T, P) * t["W"]
    return torch.cat([r, (-(h * r).sum(dim=0) / (sol[:-1] / rho * cp).sum(dim=0))[None]])


def _integrate(mech, sol, P, dt, nstep=300):
    """sol[neq, n] after dt: Radau IIA of order 5 on steps that grow geometrically from 1e-7 dt, Newton to rounding."""
    s6 = math.sqrt(6.0)
    A = _t([[(88 - 7 * s6) / 360, (296 - 169 * s6) / 1800, (-2 + 3 * s6) / 225],
            [(296 + 169 * s6) / 1800, (88 + 7 * s6) / 360, (-2 - 3 * s6) / 225],
            [(16 - s6) / 36, (16 + s6) / 36, 1 / 9]])
    neq, n = sol.shape
    ends = dt * np.concatenate([[0.0], np.geomspace(1e-7, 1.0, nstep)])
    eye = torch.eye(3 * neq, device="cuda", dtype=torch.float64)
    y = sol.clone()
    for a, b in zip(ends[:-1], ends[1:]):
        h = b - a
        f0 = _rhs(mech, y, P)
        inc = 1e-8 * y.abs().clamp_min(1e-9 * y[:-1].sum(dim=0).max())
        yp = (y[:, None, :] + torch.diag_embed(inc.t()).permute(2, 1, 0)).reshape(neq, -1)
        J = (_rhs(mech, yp, P).reshape(neq, neq, n) - f0[:, None, :]) / inc[None]
        lu = torch.linalg.lu_factor(eye - h * torch.einsum("ij,abn->niajb", A, J).reshape(n, 3 * neq, 3 * neq))
        Z = torch.zeros(3, neq, n, device="cuda", dtype=torch.float64)
        for _ in range(12):
            F = _rhs(mech, (y[None] + Z).permute(1, 0, 2).reshape(neq, -1), P).reshape(neq, 3, n).permute(1, 0, 2)
            res = h * torch.tensordot(A, F, 1) - Z
            d = torch.linalg.lu_solve(*lu, res.permute(2, 0, 1).reshape(n, -1, 1)).reshape(n, 3, neq).permute(1, 2, 0)
            Z = Z + d
            if float((d.abs() / (y.abs() + 1e-12)).max()) < 1e-13:
                break
        y = y + Z[2]
    return y


def _exact_step(case, seed):
    g, rho, SC_, mask, P, dt = _block(case, seed, False)
    t = _tables(case["mech"])
    nsp = len(t["species"])
    S = SC_.permute(3, 2, 1, 0).reshape(g.nscalar, -1)
    r = rho.permute(2, 1, 0).reshape(-1)
    sol = torch.cat([(r * S[:nsp]).clamp_min(0.0), (r * S[nsp])[None]])
    out = _integrate(case["mech"], sol, P, dt)
    new = S.clone()
    new[:nsp + 1] = out / r
    # HR_gp = -c_p of the new state times d(rho T) / dt has rounding of its own in a step this short: left out
    src = torch.stack([(out[t["species"].index(s)] - sol[t["species"].index(s)]) / dt if s in t["species"]
                       else torch.zeros_like(r) for s in ("H2O", "CO", "CO2")])
    return {"sc": _fortran(new, g.shape), "hr": None, "src": _fortran(src, g.shape)}


def _exact_properties(case, seed):
    g, _, SC_, mask, P, _ = _block(case, seed, False)
    t = _tables(case["mech"])
    nsp = len(t["species"])
    lew = 0.5 + torch.rand(nsp, generator=_gen(seed + 1), device="cuda",
                           dtype=torch.float64) if case["lewis"] else torch.ones(nsp, device="cuda")
    S = SC_.permute(3, 2, 1, 0).reshape(g.nscalar, -1)
    n = S.shape[1]
    rho, visc, diff = (torch.zeros(*s, n, device="cuda", dtype=torch.float64) for s in ((), (), (g.nscalar,)))
    live = torch.ones(g.shape, device="cuda", dtype=torch.bool)
    if mask is not None:
        live &= mask[:, :, None] != 1
    live = live.permute(2, 1, 0).reshape(-1)
    W = t["W"]
    for a in range(0, n, 1 << 18):
        c = slice(a, min(n, a + (1 << 18)))
        Y, T = S[:nsp, c], S[nsp, c]
        yt = Y.clamp(0.0, 1.0)
        Wm = yt.sum(dim=0) / (yt / W).sum(dim=0)
        rho[c] = P * Wm / (R_CST * T)
        T = T.clamp(50.0, 5000.0)
        x = T * t["koe"]
        om = (3.3530622607 + x * (2.53272006 + x * (2.9024238575 + x * 0.11186138893))) / (
            0.8662326188 + x * (1.3913958626 + x * (3.158490576 + x * (0.18973411754 + x * 0.00018682962894))))
        eta = t["mu"] * T.sqrt() / om
        v = torch.zeros_like(T)
        for k in range(nsp):
            phi = (1 + (eta[k] / eta).sqrt() * (W / W[k]) ** 0.25) ** 2 / (8.0 * (1 + W[k] / W)).sqrt()
            phi[k] = 1.0
            v += torch.where(Y[k] > 0, Y[k] * Wm * eta[k] / (W[k] * (Y * Wm * phi / W).sum(dim=0)), 0.0)
        visc[c] = v
        cp = _thermo(t, T)[1]
        cond = eta * (cp + 1.25 * R_CST / W)
        lam = 0.5 * ((Y * cond * Wm / W).sum(dim=0) + 1 / (Y * Wm / (cond * W)).sum(dim=0))
        D = lam / (Y * cp).sum(dim=0)
        diff[:nsp, c] = D / lew[:, None]
        diff[nsp, c] = D
    return {"RHO_": _fortran(rho * live, g.shape), "VISC_": _fortran(visc * live, g.shape),
            "DIFF_": _fortran(diff * live, g.shape)}


def _exact_diffusion(case, seed):
    """finitechem_diffusion (finitechem.f90:538-923), fields as [k, j, i]."""
    g, m, rho, SC_, D, mask, dt = _diffusion_inputs(case, seed)
    t = _tables(case["mech"])
    nsp, st1, st2 = len(t["species"]), m["st1"], m["st2"]
    stp = st1 + st2
    lo = [x - o for x, o in ((g.kmin_, g.kmino_), (g.jmin_, g.jmino_), (g.imin_, g.imino_))]  # first interior cell
    ni = [g.kmax_ - g.kmin_ + 1, g.jmax_ - g.jmin_ + 1, g.imax_ - g.imin_ + 1]
    S, Dk = SC_.permute(3, 2, 1, 0), D.permute(3, 2, 1, 0)
    wall = torch.zeros(S.shape[1:], device="cuda", dtype=torch.bool)
    if mask is not None:
        wall |= mask.t()[None] == 1
    op = {k: torch.from_numpy(np.ascontiguousarray(v.transpose(2, 1, 0))).cuda() for k, v in m.items()
          if k not in ("st1", "st2")}

    def part(f, d, s, face):  # f on the interior (or the face range) of the block, shifted by s along d
        a = [x - (st1 if face else 0) for x in lo]
        n = [x + (stp if face else 0) for x in ni]
        a[d] += s
        return f[tuple(slice(a[q], a[q] + n[q]) for q in range(3))]

    dims = {2: ("interp_sc_x", "grad_x", "div_u", "interp_u_xm", "grad_xm"),
            1: ("interp_sc_y", "grad_y", "div_v", "interp_v_ym", "grad_ym"),
            0: ("interp_sc_z", "grad_z", "div_w", "interp_w_zm", "grad_zm")}

    def face_op(d, which):  # operator on the face range, cut from the extents that it has
        o = op[dims[d][which]]
        nj, nf = ni[1] + stp, ni[2] + stp
        if which == 0 and d == 2:
            o = o[:, lo[1] - st1:lo[1] - st1 + nj]
        elif which == 0:
            o = o[:, :, lo[2] - st1:lo[2] - st1 + nf]
        return o

    def at_faces(f, d, which):
        return sum(face_op(d, which)[s + st2] * part(f, d, s, True) for s in range(-st2, st1 + 1))

    def at_cells(f, d, which):  # f on the face range
        def cut(s):
            a = [st1, st1, st1]
            a[d] += s
            return f[tuple(slice(a[q], a[q] + ni[q]) for q in range(3))]
        return sum(op[dims[d][which]][s + st1] * cut(s) for s in range(-st1, st2 + 1))

    def grad_m(f, d):
        return sum(op[dims[d][4]][s + stp] * part(f, d, s, False) for s in range(-stp, stp + 1))

    T = S[nsp]
    cp = _thermo(t, T.reshape(-1))[1].reshape((nsp,) + tuple(T.shape))
    Wg = torch.ones_like(T)
    y = S[:nsp].clamp(0.0, 1.0)
    w = y.sum(dim=0) / (y / t["W"][:, :, None, None]).sum(dim=0)
    Wg = torch.where(wall, Wg, w)
    cpm = (S[:nsp] * cp).sum(dim=0)
    cpm = torch.where(wall, 0.0, cpm - R_CST / w if case["cv"] else cpm)
    fwall = part(wall, 0, 0, True)
    live = ~part(wall, 0, 0, False)
    fick = lambda k, d: torch.where(fwall, 0.0, at_faces(Dk[k], d, 0) * at_faces(S[k], d, 1))
    gw = [at_faces(Wg, d, 1) for d in range(3)]
    mol = lambda k, d: at_faces(Dk[k], d, 0) * at_faces(S[k] / Wg, d, 0) * gw[d] if case["molar"] else 0.0
    vel = [sum(fick(k, d) + torch.where(fwall, 0.0, torch.as_tensor(mol(k, d), device="cuda")) for k in range(nsp))
           for d in range(3)]
    gT, gc = [grad_m(T, d) for d in range(3)], [grad_m(cpm, d) for d in range(3)]
    inner = tuple(slice(lo[q], lo[q] + ni[q]) for q in range(3))
    corr = torch.zeros((nsp + 1,) + tuple(T.shape), device="cuda", dtype=torch.float64)
    gp = torch.zeros((3,) + tuple(T.shape), device="cuda", dtype=torch.float64)
    eT = torch.zeros(ni, device="cuda", dtype=torch.float64)
    for k in range(nsp):
        dc = df = 0.0
        for d in range(3):
            fc = torch.where(fwall, 0.0, mol(k, d) - vel[d] * at_faces(S[k], d, 0))
            ff = fick(k, d)
            dc = dc + at_cells(fc, d, 2)
            df = df + at_cells(ff, d, 2)
            eT += cp[k][inner] * at_cells(fc + ff, d, 3) * gT[d]
        corr[k][inner] = torch.where(live, dc * dt, 0.0)
        if t["species"][k] in ("H2O", "CO", "CO2"):
            gp[("H2O", "CO", "CO2").index(t["species"][k])][inner] = torch.where(live, df + dc, 0.0)
    Ti = T[inner]
    if case["gasrad"]:
        u = 1000.0 / Ti
        a = {"H2O": -0.23093 + u * (-1.12390 + u * (9.41530 + u * (-2.99880 + u * (0.51382 + u * -1.86840e-05)))),
             "CO2": 18.741 + u * (-121.310 + u * (273.500 + u * (-194.050 + u * (56.310 + u * -5.8169)))),
             "CH4": 6.6334 - 0.0035686 * Ti + 1.6682e-08 * Ti ** 2 + 2.5611e-10 * Ti ** 3 - 2.6558e-14 * Ti ** 4,
             "CO": torch.where(Ti <= 750.0, 4.7869 + Ti * (-0.06953 + Ti * (2.95775e-4 + Ti * (-4.25732e-7 + Ti
                                                                                               * 2.02894e-10))),
                               10.09 + Ti * (-0.01183 + Ti * (4.7753e-6 + Ti * (-5.87209e-10 + Ti * -2.5334e-14))))}
        at = t["species"].index
        x = sum(a[s] * S[at(s)][inner] / t["W"][at(s)] for s in a if s in t["species"])
        r = rho.permute(2, 1, 0)[inner]
        eT += -4.0 * 5.67051e-8 * 8314.34 / 101320.0 * r * Ti * (Ti ** 4 - 298.0 ** 4) * x
    for d in range(3):
        eT += Dk[nsp][inner] * gc[d] * gT[d]
    corr[nsp][inner] = torch.where(live, eT / cpm[inner] * dt, 0.0)
    src = None
    if case["src"]:
        src = torch.full_like(S, 1e-7)
        src[:nsp + 1] += corr
        src = src.permute(3, 2, 1, 0)
    return {"corr": corr.permute(3, 2, 1, 0), "gp": gp.permute(3, 2, 1, 0), "src": src}


def _layers(flat, case, nin, nout):
    out, off = [], 0
    for fo, fi, _, _ in mlp.layer_shapes(nin, nout, case["hidden"], case["layers"]):
        out.append((flat[off:off + fo * fi].reshape(fo, fi), flat[off + fo * fi:off + fo * fi + fo]))
        off += fo * fi + fo
    return out


def _net(case, flat, x, nin, nout):
    for l, (Wl, bl) in enumerate(_layers(flat, case, nin, nout)):
        x = x @ Wl.t() + bl
        if l < case["layers"]:
            x = torch.nn.functional.gelu(x)
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":  # cell by cell integration of the larger blocks takes minutes
        few = case["nx"] * case["ny"] * case["nz"] <= 256 and case["mech"] == "h2" and not case["guided"]
        return _exact_step(case, seed) if few and not case["wall"] and case["nover"] == 0 and not case["host"] else None
    if kind == "properties":
        return _exact_properties(case, seed)
    if kind == "diffusion":
        return _exact_diffusion(case, seed)
    if kind in ("rhs", "prodrates"):
        Y, T, rho, P = _states(case["mech"], case["n"], _random(_gen(seed), case["n"]))
        parts = []
        for a in range(0, case["n"], 65536):
            c = slice(a, min(case["n"], a + 65536))
            if kind == "rhs":
                parts.append(_rhs(case["mech"], torch.cat([rho * Y, (rho * T)[None]])[:, c], P))
            else:
                C = rho * Y / _tables(case["mech"])["W"]
                parts.append(_prodrates(case["mech"], C[:, c], T[c], torch.full_like(T[c], P)))
        return torch.cat(parts, dim=1)
    nin, nout, flat, x, tgt = _net_inputs(case, seed)
    p = torch.from_numpy(flat).cuda().double()
    x, tgt = x.double(), tgt.double()
    if kind == "infer":
        return _net(case, p, x, nin, nout)
    m, v = torch.zeros_like(p), torch.zeros_like(p)
    for it in range(1, case["steps"] + 1):
        q = p.clone().requires_grad_(True)
        loss = ((_net(case, q, x, nin, nout)[:, :nout] - tgt) ** 2).mean()
        gr, = torch.autograd.grad(loss, q)
        m, v = 0.9 * m + 0.1 * gr, 0.999 * v + 0.001 * gr * gr
        p = p - 1e-3 * (m / (1 - 0.9 ** it)) / ((v / (1 - 0.999 ** it)).sqrt() + 1e-8)
    return {"loss": float(loss.detach()), "params": p}
