"""What a user of this framework has it do, as cases that can be measured.

A flow solver hands the chemistry its boxes (or flat arrays) of cells and gets
the reacted state back; a 0-D or analysis code calls the mechanism functions;
an optimisation calls the adjoint.  The cases below are those calls through
``pelephysics_amd.reactor``, at the sizes, tolerances and states of this
repository's benchmark, throughput tool and tests.  A box or 1-D call updates
its arrays in place, so a pass first writes the solver's new state into them
(one device copy), as the solver's transport step does between two calls.

``exact`` restates the chemistry (NASA7 thermodynamics, modified Arrhenius,
third-body, Lindemann and Troe falloff, equilibrium from Gibbs energies) in
torch float64 from the mechanism data files and integrates it by other means
than the framework does.
"""
import json
import math
import os

import torch

from pelephysics_amd.reactor import ReactorBase

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
RU = 8.31446261815324e7  # erg/(mol K)
PATM = 1.01325e6  # dyn/cm^2

FUEL = {"LiDryer": ("H2", 0.5), "drm19": ("CH4", 2.0), "dodecane_lu": ("NC12H26", 18.5),
        "heptane_lu_88sk": ("NC7H16", 11.0), "LuEthylene_qss": ("C2H4", 3.0)}

# right-hand sides, Newton-matrix factorisations and Jacobians per cell of one
# call, typical of the case's state (they vary by cell and by seed)
TYPICAL = {
    "mixed drm19 field": (111, 12, 1), "mixed dodecane_lu uneven": (81, 10, 1),
    "mixed heptane_lu_88sk ignition": (68, 10, 1), "mixed LuEthylene_qss ignition": (59, 10, 1),
    "cvode drm19 fresh": (6, 2, 1), "bdf LiDryer fresh": (3, 1, 1), "bdf drm19 fresh": (3, 1, 1),
    "rk64 drm19 fresh": (60, 0, 0),
}


def listed():
    return [
        # the headline: a 64^3 grid of a methane flame in one call, 300-2200 K
        box("flame_box_64", "mixed", "drm19", 64, 64, 64, "field"),
        # the same flame in a ragged AMReX box of a refined level
        box("flame_box_small", "mixed", "drm19", 23, 14, 9, "field"),
        # the reference's default fixed-step integrator: hydrogen, flat arrays ...
        flat("h2_fixed_step", "bdf", "LiDryer", 32768, "fresh", dt=1e-6),
        # ... and methane boxes of an explicit-diffusion solver's short steps
        box("ch4_fixed_step_box", "bdf", "drm19", 32, 32, 32, "fresh", dt=1e-6),
        # the smallest calls: one 8^3 box, where launches and latency count
        box("h2_fixed_step_box_8", "bdf", "LiDryer", 8, 8, 8, "fresh", dt=1e-6),
        # explicit low-storage RK of a compressible solver (internal energy form)
        box("ch4_rk64_box", "rk64", "drm19", 32, 32, 32, "fresh", dt=1e-6, energy=1),
        # ReactorCvode's options and defaults
        box("ch4_cvode_box", "cvode", "drm19", 15, 16, 14, "fresh", rtol=1e-6, atol=1e-10),
        # very uneven stiffness: 70% cold, 25% near ignition at 1-40 atm, 5% burnt
        flat("dodecane_uneven", "mixed", "dodecane_lu", 10000, "uneven"),
        # the largest mechanism near ignition, 10-50 atm
        flat("heptane_ignition", "mixed", "heptane_lu_88sk", 2048, "ignition", dt=1e-6, rtol=1e-8, atol=1e-14),
        # a mechanism with quasi-steady-state species
        flat("ethylene_qss", "mixed", "LuEthylene_qss", 4096, "ignition"),
        # sensitivities of T, Y_CO, Y_OH to every pre-exponential over 10 steps
        {"name": "adjoint_ch4", "kind": "adjoint", "mech": "drm19", "cells": 4096, "calls": 10, "dt": 1e-5},
        # mechanism functions over a field: species source terms and Jacobians
        {"name": "source_terms", "kind": "rates", "mech": "drm19", "cells": 262144},
    ]


def box(name, integ, mech, nx, ny, nz, state, dt=1e-5, rtol=1e-10, atol=1e-16, energy=2):
    c = {"kind": "box", "integ": integ, "mech": mech, "nx": nx, "ny": ny, "nz": nz, "state": state, "dt": dt,
         "rtol": rtol, "atol": atol, "energy": energy}
    return dict(c, name=name) if name else c


def flat(name, integ, mech, cells, state, dt=1e-5, rtol=1e-10, atol=1e-16, energy=2):
    c = {"kind": "flat", "integ": integ, "mech": mech, "cells": cells, "state": state, "dt": dt, "rtol": rtol,
         "atol": atol, "energy": energy}
    return dict(c, name=name) if name else c


def draw(rng):
    def size(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def sides(lo, hi):
        return size(lo, hi), size(lo, hi), size(lo, hi)

    what = rng.randrange(9)
    if what == 0:
        return box(None, "mixed", "drm19", *sides(5, 64), "field", energy=rng.choice((1, 2)))
    if what == 1:
        return flat(None, "bdf", "LiDryer", size(300, 300000), "fresh", dt=1e-6, energy=rng.choice((1, 2)))
    if what == 2:
        return box(None, "bdf", "drm19", *sides(5, 40), "fresh", dt=1e-6, energy=rng.choice((1, 2)))
    if what == 3:
        return box(None, "rk64", "drm19", *sides(5, 40), "fresh", dt=1e-6, energy=rng.choice((1, 2)))
    if what == 4:
        return box(None, "cvode", "drm19", *sides(5, 40), "fresh", rtol=1e-6, atol=1e-10)
    if what == 5:
        return flat(None, "mixed", "dodecane_lu", size(500, 10000), "uneven")
    if what == 6:
        return flat(None, "mixed", "LuEthylene_qss", size(300, 8192), "ignition")
    if what == 7:
        return {"kind": "adjoint", "mech": "drm19", "cells": size(200, 6000), "calls": rng.randrange(2, 11), "dt": 1e-5}
    return {"kind": rng.choice(("rates", "jacobian")), "mech": rng.choice(("LiDryer", "drm19", "dodecane_lu")),
            "cells": size(500, 50000)}


# ------------------------------------------------------ mechanism data ----
_MECH = {}


class Mech:
    """A mechanism's data on one device; species-major arrays (species, cells)."""

    def __init__(self, name, dev):
        with open(os.path.join(ROOT, "pelephysics_amd", "mechanisms", name + ".json")) as f:
            d = json.load(f)
        self.names = [s["name"].upper() for s in d["species"]]
        self.NS, self.NR = len(d["species"]), len(d["reactions"])
        self.qss = bool(d.get("qss_species"))
        t = lambda v: torch.tensor(v, dtype=torch.float64, device=dev)  # noqa: E731
        self.dev, self.species = dev, d["species"]
        self.mw, self.imw = t([s["mw"] for s in d["species"]]), t([s["imw"] for s in d["species"]])
        self.tmid = t([s["tmid"] for s in d["species"]])
        self.lo, self.hi = t([s["low"] for s in d["species"]]).T, t([s["high"] for s in d["species"]]).T
        if self.qss:
            return
        rx = d["reactions"]
        nu = torch.zeros(self.NS, self.NR, dtype=torch.float64)
        eff = torch.zeros(self.NR, self.NS, dtype=torch.float64)
        slots = {"reactants": [], "products": []}
        for j, r in enumerate(rx):
            for side, sign in (("reactants", -1.0), ("products", 1.0)):
                row = []
                for k, v in r[side].items():
                    nu[int(k), j] += sign * v
                    row += [int(k)] * int(v)
                slots[side].append((row + [self.NS] * 3)[:3])
            if r["kind"] != "elementary":
                for k, v in r["efficiencies"].items():
                    eff[j, int(k)] += v - r["default_eff"]
        self.nu, self.eff = nu.to(dev), eff.to(dev)
        self.deff = t([[r["default_eff"]] for r in rx])
        self.rs, self.ps = ([torch.tensor([row[i] for row in slots[s]], device=dev) for i in range(3)]
                            for s in ("reactants", "products"))
        self.dorder = t([[-sum(r["products"].values()) + sum(r["reactants"].values())] for r in rx])
        self.rev = t([[float(r["reversible"])] for r in rx])
        self.arr = [t([[r["rate"][k]] for r in rx]) for k in ("A", "b", "EaR")]
        self.tb = torch.tensor([j for j, r in enumerate(rx) if r["kind"] == "three-body"], device=dev, dtype=torch.long)
        fo = [j for j, r in enumerate(rx) if r["kind"] == "falloff"]
        self.fo = torch.tensor(fo, device=dev, dtype=torch.long)
        self.low = [t([[rx[j]["low"][k]] for j in fo]).reshape(-1, 1) for k in ("A", "b", "EaR")]
        troe = [rx[j]["troe"] for j in fo]
        self.troe_on = t([[float(bool(p))] for p in troe]).reshape(-1, 1)
        p4 = [(list(p) + [1e30])[:4] if p else [0.0, 1.0, 1.0, 1e30] for p in troe]
        self.troe = [t([[p[i]] for p in p4]).reshape(-1, 1) for i in range(4)]

    def thermo(self, T):
        """cp/R, h/RT and g/RT (NS, cells)."""
        a = torch.where(T[None, None, :] < self.tmid[None, :, None], self.lo[:, :, None], self.hi[:, :, None])
        cp = a[0] + T * (a[1] + T * (a[2] + T * (a[3] + T * a[4])))
        h = a[0] + T * (a[1] / 2 + T * (a[2] / 3 + T * (a[3] / 4 + T * a[4] / 5))) + a[5] / T
        s = a[0] * torch.log(T) + T * (a[1] + T * (a[2] / 2 + T * (a[3] / 3 + T * a[4] / 4))) + a[6]
        return cp, h, h - s

    def wdot(self, c, T, g, mixture=None):
        """Molar production rates (mol/m^3/s) from concentrations (mol/m^3);
        mixture: the total concentration where it is taken as a constant."""
        invT, logT = 1.0 / T, torch.log(T)
        A, b, E = self.arr
        kf = A * torch.exp(b * logT - E * invT)
        mixture = c.sum(0, keepdim=True) if mixture is None else mixture
        corr = torch.ones_like(kf)
        alpha = self.deff * mixture + self.eff @ c
        if len(self.tb):
            corr = corr.index_copy(0, self.tb, alpha[self.tb])
        if len(self.fo):
            A0, b0, E0 = self.low
            pr = A0 * torch.exp(b0 * logT - E0 * invT) * alpha[self.fo] / kf[self.fo]
            a, t3, t1, t2 = self.troe
            fc = (1 - a) * torch.exp(-T / t3) + a * torch.exp(-T / t1) + torch.exp(-t2 / T)
            lfc = torch.log10(torch.where(self.troe_on > 0, fc, torch.ones_like(fc)))
            cc, nn = -0.4 - 0.67 * lfc, 0.75 - 1.27 * lfc
            x = cc + torch.log10(pr)
            x = x / (nn - 0.14 * x)
            corr = corr.index_copy(0, self.fo, pr / (1 + pr) * torch.exp(math.log(10.0) * lfc / (1 + x * x)))
        cx = torch.cat([c, torch.ones_like(c[:1])])
        pf = cx[self.rs[0]] * cx[self.rs[1]] * cx[self.rs[2]]
        pb = cx[self.ps[0]] * cx[self.ps[1]] * cx[self.ps[2]]
        refc = 101325.0 / 8.31446 * invT
        # K_c^-1 = exp(sum nu g) refC^(reactant order - product order)
        kcinv = self.rev * torch.exp(self.rev * (self.nu.T @ g)) * refc ** self.dorder
        return self.nu @ (kf * corr * (pf - kcinv * pb))

    def rhs(self, y, src, rxsrc, energy):
        """d(rhoY, T)/dt in CGS units, y (NS + 1, cells)."""
        ry, T = y[:-1], y[-1]
        cp, h, g = self.thermo(T)
        w = self.wdot(ry * self.imw[:, None] * 1e6, T, g) * 1e-6 * self.mw[:, None] + src
        e, c = (h, cp) if energy == 2 else (h - 1, cp - 1)
        heat = (ry * self.imw[:, None] * c).sum(0) * RU
        return torch.cat([w, ((rxsrc - (w * e * self.imw[:, None]).sum(0) * (RU * T)) / heat)[None]])

    def mass_energy(self, Y, T, energy):
        _, h, _ = self.thermo(T)
        return ((h if energy == 2 else h - 1) * Y * self.imw[:, None]).sum(0) * (RU * T)

    def T_of_energy(self, e, Y, T, energy):
        for _ in range(60):
            cp, _, _ = self.thermo(T)
            c = ((cp if energy == 2 else cp - 1) * Y * self.imw[:, None]).sum(0) * RU
            T = T + ((e - self.mass_energy(Y, T, energy)) / c).clamp(-100.0, 100.0)
        return T


def mech(name, dev="cuda"):
    if name not in _MECH:
        _MECH[name] = Mech(name, torch.device(dev))
    return _MECH[name]


# ------------------------------------------------------------- states ----
def gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2654435761 % (1 << 62))
    return g


def uniform(g, n, lo, hi):
    return lo + (hi - lo) * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)


def mass(m, X):
    n = next(iter(X.values())).shape[0]
    Y = torch.zeros(m.NS, n, device="cuda", dtype=torch.float64)
    for k, x in X.items():
        Y[m.names.index(k)] += x * m.mw[m.names.index(k)]
    return Y / Y.sum(0)


def fuel_air(m, name, phi):
    fuel, s = FUEL[name]
    one = torch.ones_like(phi)
    return mass(m, {fuel: phi, "O2": s * one, "N2": 3.76 * s * one})


def products(m, name, phi):
    fuel, s = FUEL[name]
    comp = m.species[m.names.index(fuel)]["composition"]
    burnt = phi.clamp(max=1.0)
    X = {fuel: phi - burnt, "O2": s * (1 - burnt), "N2": 3.76 * s * torch.ones_like(phi),
         "H2O": 0.5 * comp.get("H", 0.0) * burnt}
    if comp.get("C", 0.0):
        X["CO2"] = comp["C"] * burnt
    return mass(m, X)


def state_of(case, g):
    """Mass fractions (NS, cells), T, p of the case's cells, cell index i fastest."""
    name = case["mech"]
    m = mech(name)
    kind = case.get("state", "field")
    n = case["nx"] * case["ny"] * case["nz"] if case.get("kind") == "box" else case["cells"]
    p = torch.full((n,), PATM, device="cuda", dtype=torch.float64)
    if kind == "field":
        # mixture fraction: Gaussian random field, an eighth of the box long
        shape = (case["nz"], case["ny"], case["nx"]) if case.get("kind") == "box" else (1, 1, n)
        w = torch.randn(shape, generator=g, device="cuda", dtype=torch.float64)
        k2 = sum(f ** 2 for f in torch.meshgrid(*[torch.fft.fftfreq(s, device="cuda", dtype=torch.float64) * s
                                                  for s in shape], indexing="ij"))
        f = torch.fft.ifftn(torch.fft.fftn(w) * torch.exp(-0.5 * (2 * math.pi / 8.0) ** 2 * k2)).real.reshape(-1)
        Z = torch.special.ndtr((f - f.mean()) / f.std())
        c = uniform(g, n, 0.0, 1.0)
        mw = lambda s: m.mw[m.names.index(s)]  # noqa: E731
        burnt = torch.minimum(Z / mw("CH4"), 0.233 * (1 - Z) / mw("O2") / 2.0)
        Y = torch.zeros(m.NS, n, device="cuda", dtype=torch.float64)
        for s, v in (("CH4", Z - c * burnt * mw("CH4")), ("O2", 0.233 * (1 - Z) - 2 * c * burnt * mw("O2")),
                     ("N2", 0.767 * (1 - Z)), ("CO2", c * burnt * mw("CO2")), ("H2O", 2 * c * burnt * mw("H2O"))):
            Y[m.names.index(s)] = v.clamp(min=0.0)
        T = 300.0 + 1900.0 * c
    elif kind == "fresh":
        T = uniform(g, n, 1000.0, 1400.0) if name == "LiDryer" else uniform(g, n, 1100.0, 1500.0)
        Y = fuel_air(m, name, uniform(g, n, 0.5, 1.5))
        if name == "LiDryer":
            for s in ("H", "O", "OH", "HO2", "H2O2"):
                Y[m.names.index(s)] = 1e-8
    elif kind == "uneven":
        nf, ni = int(0.70 * n), int(0.25 * n)
        nb = n - nf - ni
        T = torch.cat([uniform(g, nf, 300.0, 700.0), uniform(g, ni, 900.0, 1200.0),
                       torch.full((nb,), 2300.0, device="cuda", dtype=torch.float64)])
        phi = torch.cat([torch.ones(nf, device="cuda", dtype=torch.float64), uniform(g, ni, 0.7, 1.3)])
        p[nf:nf + ni] *= uniform(g, ni, 1.0, 40.0)
        Y = torch.cat([fuel_air(m, name, phi), products(m, name, torch.ones(nb, device="cuda", dtype=torch.float64))],
                      dim=1)
        order = torch.randperm(n, generator=g, device="cuda")
        Y, T, p = Y[:, order], T[order], p[order]
    else:
        hot = name == "heptane_lu_88sk"
        T = uniform(g, n, 800.0, 1300.0) if hot else uniform(g, n, 900.0, 1200.0)
        phi = uniform(g, n, 0.5, 2.0) if hot else uniform(g, n, 0.7, 1.3)
        p = p * (uniform(g, n, 10.0, 50.0) if hot else uniform(g, n, 1.0, 40.0))
        Y = fuel_air(m, name, phi)
    return Y / Y.sum(0), T, p


def inputs(case, seed):
    """rhoY (NS, cells), T, rho e or rho h, and their external sources."""
    g = gen(seed)
    m = mech(case["mech"])
    Y, T, p = state_of(case, g)
    rho = p / ((Y * m.imw[:, None]).sum(0) * RU * T)
    ry, rx = rho * Y, rho * m.mass_energy(Y, T, case["energy"])
    # transport terms of the flow solver: up to 20 /s of each quantity
    src = ry * uniform(g, ry.shape[1], -20.0, 20.0)
    rxsrc = rho * 1e9 * uniform(g, ry.shape[1], -20.0, 20.0)
    return ry, T, rx, src, rxsrc


INTEGRATOR = {"mixed": "ReactorBDFAdaptiveMixed", "bdf": "ReactorBDF", "rk64": "ReactorRK64", "cvode": "ReactorCvode"}


def prepare(case, seed):
    m = mech(case["mech"])
    if case["kind"] in ("rates", "jacobian"):
        sc, T = concentrations(case, seed)
        R = ReactorBase.create("ReactorBDF")
        R.init(2, case["cells"], mechanism=case["mech"])
        return {"kind": case["kind"], "R": R, "sc": sc.T.contiguous(), "T": T.contiguous()}
    if case["kind"] == "adjoint":
        ry, T, rx = adjoint_inputs(case, seed)
        R = ReactorBase.create("ReactorBDF")
        R.init(2, case["cells"], mechanism="drm19_table")
        start = torch.cat([ry, T[None]]).T.contiguous()
        return {"kind": "adjoint", "R": R, "start": start, "y": start.clone(), "rX": rx, "calls": case["calls"],
                "dt": case["dt"]}
    ry, T, rx, src, rxsrc = inputs(case, seed)
    R = ReactorBase.create(INTEGRATOR[case["integ"]])
    ode = {"mixed": dict(tuned="box" if case["kind"] == "box" else "1d", rtol=case["rtol"], atol=case["atol"]),
           "cvode": dict(rtol=case["rtol"], atol=case["atol"])}.get(case["integ"], {})
    R.init(case["energy"], T.shape[0], mechanism=case["mech"], **ode)
    s = {"kind": case["kind"], "R": R, "dt": case["dt"]}
    if case["kind"] == "box":
        shape = (case["nz"], case["ny"], case["nx"])
        s["start"] = torch.cat([ry, T[None], rx[None]]).reshape(m.NS + 2, *shape).contiguous()
        s["now"] = s["start"].clone()
        s["src"] = torch.cat([src, rxsrc[None]]).reshape(m.NS + 1, *shape).contiguous()
        s["fc"] = torch.zeros((1, *shape), device="cuda", dtype=torch.float64)
    else:
        y = torch.cat([ry, T[None]]).T.reshape(-1)
        s["start"] = torch.cat([y, rx])
        s["now"] = s["start"].clone()
        s["src"], s["rxsrc"], s["ny"] = src.T.reshape(-1).contiguous(), rxsrc.contiguous(), y.shape[0]
    return s


def run(s):
    R, kind = s["R"], s["kind"]
    if kind == "rates":
        return R.production_rate(s["sc"], s["T"])
    if kind == "jacobian":
        return R.ajacobian(s["sc"], s["T"], 1)
    if kind == "adjoint":
        s["y"].copy_(s["start"])
        out, grad = R.adjoint_1d(s["y"], s["rX"], s["calls"], s["dt"])
        return {"y": s["y"], "out": out, "grad": grad}
    s["now"].copy_(s["start"])
    if kind == "box":
        ns = R.nspec
        rY, T, rE = s["now"][:ns], s["now"][ns:ns + 1], s["now"][ns + 1:]
        R.react(rY, s["src"][:ns], T, rE, s["src"][ns:], s["fc"], s["dt"])
        return {"rY": rY, "T": T, "rE": rE, "FC": s["fc"].to(torch.int32)}
    y, rX = s["now"][:s["ny"]], s["now"][s["ny"]:]
    R.react_1d(y, s["src"], rX, s["rxsrc"], s["dt"])
    y = y.view(rX.shape[0], -1)
    return {"rY": y[:, :-1], "T": y[:, -1], "rX": rX}


def concentrations(case, seed):
    """Concentrations (mol/m^3) and temperatures of a partly burnt field."""
    g = gen(seed)
    m = mech(case["mech"])
    n = case["cells"]
    T, phi, c = uniform(g, n, 500.0, 2500.0), uniform(g, n, 0.5, 1.5), uniform(g, n, 0.0, 1.0)
    Y = (1 - c) * fuel_air(m, case["mech"], phi) + c * products(m, case["mech"], phi)
    Y = Y + 10.0 ** uniform(g, m.NS * n, -9.0, -3.0).reshape(m.NS, n)  # radicals and intermediates
    Y = Y / Y.sum(0)
    rho = PATM * uniform(g, n, 1.0, 10.0) / ((Y * m.imw[:, None]).sum(0) * RU * T)
    return rho * Y * m.imw[:, None] * 1e6, T


def adjoint_inputs(case, seed):
    g = gen(seed)
    m = mech(case["mech"])
    T, phi = uniform(g, case["cells"], 1100.0, 1500.0), uniform(g, case["cells"], 0.6, 1.4)
    Y = fuel_air(m, case["mech"], phi)
    rho = PATM / ((Y * m.imw[:, None]).sum(0) * RU * T)
    return rho * Y, T, rho * m.mass_energy(Y, T, 2)


# ------------------------------------------------------ work, tolerance ----
def work(case):
    with open(os.path.join(ROOT, "pelephysics_amd", "mechanisms", case["mech"] + ".json")) as f:
        d = json.load(f)
    ns, nr = len(d["species"]), len(d["reactions"])
    n = ns + 1
    rhs, jac = 45.0 * nr + 90.0 * ns, 110.0 * nr + 90.0 * ns  # FP64 operations, a transcendental as one
    if case["kind"] == "rates":
        return {"bytes": 8.0 * case["cells"] * (2 * ns + 1), "flops": rhs * case["cells"]}
    if case["kind"] == "jacobian":
        return {"bytes": 8.0 * case["cells"] * (n + n * n), "flops": jac * case["cells"]}
    if case["kind"] == "adjoint":
        # per step forward and back: two right-hand sides, Jacobian, factors,
        # and the Jacobian's derivative along the n equations
        per = case["calls"] * (2 * rhs + jac * (2 + n) + 4.0 / 3.0 * n ** 3)
        return {"bytes": 8.0 * case["cells"] * (2 * n + 4 + 3 * nr), "flops": per * case["cells"]}
    cells = case["nx"] * case["ny"] * case["nz"] if case["kind"] == "box" else case["cells"]
    nrhs, nlu, njac = TYPICAL["%s %s %s" % (case["integ"], case["mech"], case["state"])]
    per = nrhs * (rhs + 2.0 * n * n) + nlu * 2.0 / 3.0 * n ** 3 + njac * jac
    return {"bytes": 8.0 * cells * (3 * n + 2 + (1 if case["kind"] == "box" else 0)), "flops": per * cells}


def tolerance(case):
    kind = case["kind"]
    if kind in ("rates", "jacobian"):
        return {"rel": 1e-11}
    if kind == "adjoint":
        return {"rel": 1e-7}
    if case["integ"] == "mixed":
        # where a Newton iteration or a step is decided by rounding the results
        # differ by the step error, a few times rtol; step counts by one
        return {"rel": 20 * case["rtol"], "differ": 0.05}
    if case["integ"] == "cvode":
        return {"rel": 1e-6, "differ": 0.05}
    if case["integ"] == "bdf":  # GMRES stops at a residual of 1e-10 (CGS units), not at rounding
        return {"rel": 4e-7 if case["mech"] == "LiDryer" else 1e-8, "differ": 0.001}
    return {"rel": 1e-10, "differ": 0.001}


# --------------------------------------------------------------- exact ----
def exact(case, seed):
    m = mech(case["mech"])
    if case["kind"] in ("rates", "jacobian"):
        sc, T = concentrations(case, seed)
        if case["kind"] == "rates":
            return m.wdot(sc, T, m.thermo(T)[2]).T.contiguous()
        return exact_jacobian(m, sc, T) if m.NS * m.NR * case["cells"] < 2e8 else None
    if case["kind"] == "adjoint" or m.qss or m.NS > 30:
        return None
    ry, T, rx, src, rxsrc = inputs(case, seed)
    cells, dt = T.shape[0], case["dt"]
    if case["kind"] == "box":  # the box form takes T from the energy
        T = m.T_of_energy(rx / ry.sum(0), ry / ry.sum(0), T, case["energy"])
    y = torch.cat([ry, T[None]])
    if case["integ"] == "bdf":
        y = exact_fixed_step(m, y, src, rxsrc, dt, case["energy"])
    elif case["integ"] == "rk64":
        y = exact_rk64(m, y, src, rxsrc, dt, case["energy"])
    else:
        if cells > 4000:
            return None
        y = exact_solution(m, y, src, rxsrc, dt, case["energy"])
    rx = rx + dt * rxsrc
    if case["kind"] == "box":
        rho = y[:-1].sum(0)
        T = m.T_of_energy(rx / rho, y[:-1] / rho, y[-1], case["energy"])
        shape = (case["nz"], case["ny"], case["nx"])
        return {"rY": y[:-1].reshape(-1, *shape), "T": T.reshape(1, *shape), "rE": rx.reshape(1, *shape), "FC": None}
    return {"rY": y[:-1].T.contiguous(), "T": y[-1].contiguous(), "rX": rx}


def exact_solution(m, y, src, rxsrc, dt, energy, steps=240):
    """The solution itself: three-stage Radau IIA of order 5, every cell on the
    same geometric steps (from 1e-9 dt), each step's stages by Newton
    iterations with the Jacobian at its start."""
    r6 = math.sqrt(6.0)
    A = torch.tensor([[(88 - 7 * r6) / 360, (296 - 169 * r6) / 1800, (-2 + 3 * r6) / 225],
                      [(296 + 169 * r6) / 1800, (88 + 7 * r6) / 360, (-2 - 3 * r6) / 225],
                      [(16 - r6) / 36, (16 + r6) / 36, 1 / 9]], dtype=torch.float64, device=y.device)
    n, cells = y.shape
    eye = torch.eye(3 * n, dtype=torch.float64, device=y.device)
    basis = torch.eye(n, dtype=torch.float64, device=y.device)[:, :, None].expand(n, n, cells)
    wide = [v[..., None].expand(*v.shape, 3).reshape(*v.shape[:-1], -1) for v in (src, rxsrc)]
    t = 0.0
    for i in range(1, steps + 1):
        t_new = dt * 1e-9 ** (1.0 - i / steps)
        h, t = t_new - t, t_new
        J = torch.func.vmap(lambda v: torch.func.jvp(lambda u: m.rhs(u, src, rxsrc, energy), (y,), (v,))[1])(basis)
        J = J.permute(2, 1, 0)  # (cells, row, column)
        N = eye - (h * A[None, :, None, :, None] * J[:, None, :, None, :]).reshape(cells, 3 * n, 3 * n)
        lu = torch.linalg.lu_factor(N)
        z = torch.zeros(n, cells, 3, dtype=torch.float64, device=y.device)
        for _ in range(6):
            f = m.rhs((y[:, :, None] + z).reshape(n, -1), *wide, energy).reshape(n, cells, 3)
            res = h * (f @ A.T) - z
            d = torch.linalg.lu_solve(*lu, res.permute(1, 2, 0).reshape(cells, 3 * n, 1))
            z = z + d.reshape(cells, 3, n).permute(2, 0, 1)
        y = y + z[:, :, 2]
    return y


def exact_rk64(m, y, src, rxsrc, dt, energy):
    """The 6-stage low-storage RK with its step controller, each cell its own step."""
    al = (0.218150805229859, 0.256702469801519, 0.527402592007520, 0.0484864267224467, 1.24517071533530, 0.412366034843237)
    be = (-0.113554138044166, -0.215118587818400, -0.0510152146250577, -1.07992686223881, -0.248664241213447, 0.0)
    er = (-0.0554699315064507, 0.158481845574980, -0.0905918835751907, -0.219084567203338, 0.164022338959433,
          0.0426421977505659)
    atol, guess, most, least = 1e-10, 10, 500, 5
    t = torch.zeros_like(y[-1])
    h = torch.full_like(t, dt / guess)
    carry = y.clone()
    for _ in range(4 * most):
        on = t < dt
        if not bool(on.any()):
            break
        err = torch.zeros_like(y)
        h = torch.where(on, h, torch.zeros_like(h))
        for s in range(6):
            f = m.rhs(y, src, rxsrc, energy)
            err = err + er[s] * h * f
            y1 = carry + al[s] * h * f
            carry = torch.where(on, y1 + be[s] * h * f, carry)
            y = torch.where(on, y1, y)
        t = t + h
        e = err.abs().amax(0).clamp(min=1e-50)
        h = torch.where(e < atol, (h * (atol / e) ** 0.25).clamp(max=dt / least), (h * (atol / e) ** 0.2).clamp(min=dt / most))
        h = torch.minimum(h, dt - t)
    return y


def derivatives(m, c, T, energy):
    """d wdot / d c, d wdot / d T and the same of dT/dt = -T sum(e wdot) / sum(c cv),
    laid out (cells, column, row); in the enthalpy form third-body
    concentrations take the mixture sum as constant."""
    n = c.shape[1]
    out = torch.zeros(n, m.NS + 1, m.NS + 1, dtype=torch.float64, device=c.device)
    mix = c.sum(0, keepdim=True) if energy == 2 else None

    def f(c, T):
        cp, h, g = m.thermo(T)
        w = m.wdot(c, T, g, mix)
        e, cc = (h, cp) if energy == 2 else (h - 1, cp - 1)
        return torch.cat([w, (-T * (e * w).sum(0) / (cc * c).sum(0))[None]])

    for k in range(m.NS + 1):
        vc, vT = torch.zeros_like(c), torch.zeros_like(T)
        if k < m.NS:
            vc[k] = 1.0
        else:
            vT[:] = 1.0
        _, d = torch.func.jvp(f, (c, T), (vc, vT))
        out[:, k, :] = d.T
    return out


def exact_jacobian(m, sc, T):
    return derivatives(m, sc, T, 2)


def exact_fixed_step(m, y, src, rxsrc, dt, energy):
    """One linearised trapezoidal step, (1/dt - J/2) d = f, by dense solves."""
    f = m.rhs(y, src, rxsrc, energy)
    J = derivatives(m, y[:-1] * m.imw[:, None] * 1e6, y[-1], energy).transpose(1, 2)  # (cells, row, column), SI
    one = torch.ones_like(m.mw[:1])
    J = J * torch.cat([m.mw * 1e-6, one])[:, None] * torch.cat([m.imw * 1e6, one])[None, :]
    A = torch.eye(m.NS + 1, dtype=torch.float64, device=y.device) / dt - 0.5 * J
    return y + torch.linalg.solve(A, f.T[:, :, None])[:, :, 0].T
