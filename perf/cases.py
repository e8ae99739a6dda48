"""Performance cases of the SU(3) gauge-link path: what a lattice program does with it.

A program makes a configuration (``gauge_configuration``), puts links on it, and then runs one of
the library's long-lived jobs: quenched HMC (plain or stout-smeared action, three integrators, three
precision forms), checkerboard heatbath + overrelaxation, Wilson flow with its observables, field
strength measurements, or the forward/backward pair an AD rule of the stout map calls.  What it
keeps at the end comes back to the host: the configuration, and the numbers the job reports.  In the
forms that compute in single precision (f32, f32force) it keeps single-precision copies.

Links are the ones quenched lattices at beta = 6 have in the mean (plaquette near 0.6): independent
SU(3) matrices scattered about the unit matrix, made on the GPU from the seed.  Momenta are drawn
on the device at the start of every trajectory, as HMC does.

A case: {"kind", "nx", "ny", "nz", "nt", "form" (f64, f32, f32force), ...}; see listed().
"""
import importlib
import math

import numpy as np
import torch

import __graft_entry__

__graft_entry__.load_package()
api = importlib.import_module("gaugefields_jl_amd.api")

BETA = 6.0
DEV = "cuda" if torch.cuda.is_available() else "cpu"
SPREAD = 0.2  # scatter of the links about the unit matrix: plaquette 0.6


def listed():
    return [
        # plain quenched HMC on the smallest lattice used in earnest (tests, tuning, teaching): 10
        # leapfrog steps a trajectory; every launch and every wait counts
        hmc("hmc_4", (4, 4, 4, 4), "QPQ", 10, 5),
        # the same on extents without a power of two, one of them odd, in single precision
        hmc("hmc_f32_odd", (10, 6, 14, 9), "2MN", 10, 5, form="f32"),
        # an ordinary development lattice, Omelyan integrator
        hmc("hmc_16", (16, 16, 16, 16), "2MN", 15, 5),
        # production plain HMC: half steps merged (fused)
        hmc("hmc_32", (32, 32, 32, 32), "2MN", 10, 8, fused=True),
        # stout-smeared HMC, three levels, double precision: one trajectory of 10 Omelyan steps
        hmc("stout_24", (24, 24, 24, 24), "2MN", 10, 1, levels=3, rho=0.1),
        # its memory-saving mode on a small lattice, forces in single precision over a double state
        hmc("stout_f32force_12", (12, 12, 12, 24), "2MN", 10, 2, levels=2, rho=0.1, mode="recompute",
            form="f32force"),
        # production stout HMC in single precision: 16 merged Omelyan steps
        hmc("stout_f32_32", (32, 32, 32, 32), "2MN", 16, 1, levels=3, rho=0.12, form="f32", fused=True),
        # Wilson flow of a production lattice to t = 1, E(t) every tenth step
        flow("flow_32", (32, 32, 32, 32), 100, 10),
        # Wilson flow with plaquette, clover and improved observables of a finite-temperature lattice
        flow("flow_measure_20", (20, 20, 20, 10), 40, 4, observables=True),
        # quenched ensemble generation: heatbath sweeps with four overrelaxation sweeps each
        heatbath("heatbath_24", (24, 24, 24, 48), 5, 4),
        # one configuration's field strengths: density of the improved charge, clover energy
        measure("charge_24", (24, 24, 24, 48), "improved"),
        # the stout map under automatic differentiation: smeared links out, cotangent in, gradient out
        backprop("stout_ad_12", (12, 12, 12, 12), 2, 0.1),
    ]


def _case(kind, name, dims, form, **more):
    c = {"kind": kind, "nx": dims[0], "ny": dims[1], "nz": dims[2], "nt": dims[3], "form": form, **more}
    if name:
        c["name"] = name
    return c


def hmc(name, dims, integrator, steps, trajectories, *, form="f64", levels=0, rho=0.0, mode="auto", fused=False):
    return _case("hmc", name, dims, form, integrator=integrator, steps=steps, trajectories=trajectories,
                 levels=levels, rho=rho, mode=mode, fused=fused)


def flow(name, dims, steps, every, *, form="f64", observables=False):
    return _case("flow", name, dims, form, steps=steps, every=every, observables=observables)


def heatbath(name, dims, sweeps, overrelax, *, form="f64"):
    return _case("heatbath", name, dims, form, sweeps=sweeps, overrelax=overrelax)


def measure(name, dims, method, *, form="f64"):
    return _case("measure", name, dims, form, method=method)


def backprop(name, dims, levels, rho, *, form="f64"):
    return _case("backprop", name, dims, form, levels=levels, rho=rho)


def _dims(case):
    return case["nx"], case["ny"], case["nz"], case["nt"]


def _volume(case):
    return case["nx"] * case["ny"] * case["nz"] * case["nt"]


def _extents(rng, most, even):
    """four extents of a volume spread evenly over the logarithm of 256 .. most"""
    v = math.exp(rng.uniform(math.log(256), math.log(most)))
    side = v ** 0.25
    while True:
        d = []
        for _ in range(4):
            n = max(2, round(side * math.exp(rng.uniform(-0.35, 0.35))))
            if rng.random() < 0.4:
                n = max(4, 4 * round(n / 4))  # round extents are the usual choice
            d.append(n + n % 2 if even else n)
        if 200 <= math.prod(d) <= most:
            return tuple(d)


def draw(rng):
    kind = rng.choice(["hmc", "hmc", "hmc", "stout", "stout", "flow", "flow", "heatbath", "measure", "backprop"])
    form = rng.choice(["f64", "f64", "f32"])
    if kind in ("hmc", "stout"):
        form = rng.choice([form, form, form, "f32force"])
        dims = _extents(rng, 600_000 if kind == "hmc" else 250_000, False)
        integrator = rng.choice(["QPQ", "PQP", "2MN"])
        steps, fused = rng.randint(6, 16), rng.random() < 0.4
        if kind == "hmc":
            return hmc(None, dims, integrator, steps, rng.randint(1, 4), form=form, fused=fused)
        return hmc(None, dims, integrator, steps, 1, form=form, levels=rng.randint(1, 3), rho=rng.choice([0.08, 0.1, 0.12]),
                   mode=rng.choice(["auto", "auto", "recompute"]), fused=fused)
    if kind == "flow":
        every = rng.randint(2, 10)
        return flow(None, _extents(rng, 500_000, False), every * rng.randint(2, 6), every, form=form,
                    observables=rng.random() < 0.4)
    if kind == "heatbath":
        return heatbath(None, _extents(rng, 600_000, True), rng.randint(1, 6), rng.randint(0, 5))
    if kind == "measure":
        return measure(None, _extents(rng, 600_000, False), rng.choice(["plaquette", "clover", "improved"]), form=form)
    return backprop(None, _extents(rng, 60_000, False), rng.randint(1, 3), rng.choice([0.08, 0.1, 0.12]), form=form)


# ------------------------------------------------------------------------- inputs


def _links(dims, seed):
    """independent SU(3) links about the unit matrix, (4, V, 3, 3) complex128 on the GPU"""
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    v = math.prod(dims)
    r = torch.randn(4, v, 2, 3, 2, generator=g, device=DEV, dtype=torch.float64)
    m = torch.view_as_complex(r) * SPREAD
    a = m[..., 0, :] + torch.tensor([1.0, 0, 0], device=DEV)
    b = m[..., 1, :] + torch.tensor([0, 1.0, 0], device=DEV)
    a = a / a.abs().square().sum(-1, keepdim=True).sqrt()
    b = b - (b * a.conj()).sum(-1, keepdim=True) * a
    b = b / b.abs().square().sum(-1, keepdim=True).sqrt()
    return torch.stack([a, b, torch.linalg.cross(a, b).conj()], -2)


def _reference_layout(m):
    """(4, V, 3, 3) [..., i, j] -> the host layout (4, V, 9), element (i, j) at i + 3 j"""
    return m.transpose(-1, -2).reshape(4, -1, 9).resolve_conj().cpu().numpy()


def _cotangent(dims, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 1_000_003)
    return torch.view_as_complex(torch.randn(4, math.prod(dims), 3, 3, 2, generator=g, device=DEV, dtype=torch.float64))


def prepare(case, seed):
    form = case["form"]
    U = api.gauge_configuration(_dims(case), backend=api.HIPBackend(), seed=seed,
                                eltype=np.complex64 if form == "f32" else np.complex128,
                                force_eltype=np.complex64 if form == "f32force" else None)
    U.from_host(_reference_layout(_links(_dims(case), seed)))
    s = {"case": case, "U": U, "seed": int(seed), "single": form != "f64"}
    if case["kind"] == "hmc":
        loops = api.make_loops_fromname("plaquette")
        action = api.GaugeAction(U).push(BETA / 2, loops + api.dagger(loops))
        if case["levels"]:
            action = api.SmearedGaugeAction(action, api.stout_smearing(U, rho=case["rho"], levels=case["levels"],
                                                                      mode=case["mode"]))
        integrator = {"QPQ": api.QPQ, "PQP": api.PQP, "2MN": api.OmelyanPQP}[case["integrator"]]()
        s["P"] = api.gauge_momenta(U)
        s["driver"] = api.md_driver(U, action, steps=case["steps"], trajectory_length=_tau(case), integrator=integrator)
        s["metropolis"] = np.random.default_rng(int(seed))
        s["sweep"] = 0
    elif case["kind"] == "flow":
        s["flow"] = api.gradient_flow(U, steps=case["steps"], step_size=0.01)
    elif case["kind"] == "heatbath":
        s["heatbath"] = api.Heatbath(U, BETA, seed=int(seed))
    elif case["kind"] == "backprop":
        s["smearing"] = api.stout_smearing(U, rho=case["rho"], levels=case["levels"])
        s["cotangent"] = _reference_layout(_cotangent(_dims(case), seed))
    return s


def _tau(case):
    """trajectory length: as many steps of a size at which most trajectories are accepted, from
    links that are not in equilibrium yet (the energy error then grows with the volume)"""
    step = (0.04 if case["integrator"] != "2MN" else 0.08) * (0.5 if case["levels"] else 1.0)
    return round(case["steps"] * step * (_volume(case) / 256) ** (-1 / 3), 4)


def _kept(x, s):
    """what a program keeps: as given in double precision, or its single-precision copy"""
    t = torch.from_numpy(np.asarray(x))
    return t.to({torch.complex128: torch.complex64, torch.float64: torch.float32}[t.dtype]) if s["single"] else t


# ------------------------------------------------------------------------- one pass


def run(s):
    return {"hmc": _run_hmc, "flow": _run_flow, "heatbath": _run_heatbath, "measure": _run_measure,
            "backprop": _run_backprop}[s["case"]["kind"]](s)


def _run_hmc(s):
    """trajectories with momentum refresh, Metropolis test and plaquette; the configuration"""
    U, P, driver = s["U"], s["P"], s["driver"]
    energies, accepted, plaquettes = [], [], []
    for _ in range(s["case"]["trajectories"]):
        api.gaussian_momenta_(P, seed=s["seed"], sweep=s["sweep"])
        s["sweep"] += 1
        U.copy_to_backup()
        d = api.md_trajectory(U, P, driver, fused=s["case"]["fused"])
        ok = s["metropolis"].random() < math.exp(min(0.0, -d["delta_hamiltonian"]))
        if not ok:
            U.restore_from_backup()
        energies.append((d["initial_hamiltonian"], d["final_hamiltonian"]))
        accepted.append(int(ok))
        plaquettes.append(api.measure_plaquette(U))
    return {"hamiltonians": _kept(energies, s), "accepted": torch.tensor(accepted), "plaquettes": _kept(plaquettes, s),
            "links": _kept(U.to_host(), s)}


def _run_flow(s):
    """the flow's observables along the way and the flowed configuration"""
    c = s["case"]
    if c["observables"]:
        rows = s["U"].lattice.flow_measure(s["flow"].eps, s["flow"].Nflow, c["every"])
        return {"rows": _kept(rows, s), "links": _kept(s["U"].to_host(), s)}
    E = api.flow(s["U"], s["flow"], measure_every=c["every"])
    return {"energy": _kept(E, s), "links": _kept(s["U"].to_host(), s)}


def _run_heatbath(s):
    plaquettes = []
    for _ in range(s["case"]["sweeps"]):
        api.heatbath(s["U"], s["heatbath"])
        for _ in range(s["case"]["overrelax"]):
            api.overrelaxation(s["U"], s["heatbath"])
        plaquettes.append(api.measure_plaquette(s["U"]))
    return {"plaquettes": _kept(plaquettes, s), "failures": s["heatbath"].failures, "links": _kept(s["U"].to_host(), s)}


def _run_measure(s):
    U = s["U"]
    return {"density": _kept(np.ascontiguousarray(api.topological_charge_density(U, method=s["case"]["method"]).T), s),
            "energy": _kept(api.calculate_energy_density(U), s), "plaquette": _kept(api.measure_plaquette(U), s)}


def _run_backprop(s):
    return {"smeared": _kept(api.smear(s["U"], s["smearing"]), s),
            "gradient": _kept(api.back_prop(s["cotangent"], s["smearing"], s["U"]), s)}


# ------------------------------------------------------------------------- work


def work(case):
    """Compulsory bytes and operations of a pass.  A link is 12 reals, a momentum 8, a general 3x3
    matrix 18; every MD update, flow stage, smearing level and checkerboard sweep reads and writes
    its fields once (a lattice does not stay in cache between them); the links come back as 18
    doubles.  Operations per site: 7.1e3 for the staple force of all four links, 4.4e3 for the four
    exponentials and link products, 28e3 for the backward pass of one smearing level, 0.6e3 for a
    plane's loop set of one leaf or rectangle pair."""
    v, c = _volume(case), case
    real = 4 if c["form"] == "f32" else 8
    U, P, M, force, expo, back = 48, 32, 72, 7.1e3, 4.4e3, 28e3
    out = 72 * 8
    if c["kind"] == "hmc":
        per_step = {"QPQ": 1, "PQP": 1, "2MN": 2}[c["integrator"]]
        n = c["trajectories"] * (c["steps"] * per_step + (c["integrator"] != "QPQ"))
        reals = n * (2 * U + 2 * P + c["levels"] * (4 * U + 4 * M + 2 * P)) + c["trajectories"] * (6 * U + 3 * P)
        flops = n * (force + expo + c["levels"] * (force + expo + back)) + c["trajectories"] * (3 * 3.5e3 + 2 * c["levels"] * (force + expo))
    elif c["kind"] == "flow":
        n = 3 * c["steps"]
        rows = c["steps"] // c["every"]
        reals, flops = n * 2 * (U + P) + rows * U, n * (force + expo) + rows * (90e3 if c["observables"] else 3.5e3)
    elif c["kind"] == "heatbath":
        n = c["sweeps"] * (1 + c["overrelax"])
        reals, flops = n * 2 * U + c["sweeps"] * U, n * (force + expo) + c["sweeps"] * 3.5e3
    elif c["kind"] == "measure":
        out = 8
        reals, flops = 3 * U, {"plaquette": 3.5e3, "clover": 14e3, "improved": 70e3}[c["method"]] + 14e3
    else:
        out = 3 * 72 * 8
        reals = 2 * c["levels"] * (2 * U + M) + c["levels"] * (U + 2 * M)
        flops = c["levels"] * (2 * (force + expo) + back)
    return {"bytes": float(v * (reals * real + out)), "flops": float(v * flops)}


# ------------------------------------------------------------------------- the same in plain torch, 64 bits


def exact(case, seed):
    """what run() returns for a new state, in complex128 torch; None where there is no closed value
    (the sampled heatbath) or it would take long"""
    if case["kind"] == "heatbath":
        return None
    v = _volume(case)
    if case["kind"] == "hmc" and v * case["trajectories"] * case["steps"] * (1 + 8 * case["levels"]) > 4e7:
        return None
    if case["kind"] == "flow" and v * case["steps"] > 3e7:
        return None
    L = _Torch(_dims(case))
    with torch.no_grad():
        U = _links(_dims(case), seed).reshape(L.shape)
        if case["kind"] == "hmc":
            return _exact_hmc(case, seed, L, U)
        if case["kind"] == "flow":
            return _exact_flow(case, L, U)
        if case["kind"] == "measure":
            density, energy = L.field_strengths(U)
            return {"density": density[case["method"]].cpu().numpy(), "energy": np.float64(energy.item()),
                    "plaquette": np.float64(L.plaquette_sum(U).item() / (18 * v))}
    D = _cotangent(_dims(case), seed).reshape(L.shape)
    U = U.clone().requires_grad_(True)
    S = L.smear(U, case["levels"], case["rho"])
    # D is dS/dU of the smeared links: dS = Re tr(D dU)
    (D.transpose(-1, -2) * S).real.sum().backward()
    return {"smeared": _reference_layout(S.detach()), "gradient": _reference_layout(U.grad.mH)}


def _exact_hmc(case, seed, L, U):
    levels, rho, steps = case["levels"], case["rho"], case["steps"]
    e, lam = _tau(case) / steps, 0.1931833275037836
    step = {"QPQ": [("U", 0.5), ("P", 1.0), ("U", 0.5)], "PQP": [("P", 0.5), ("U", 1.0), ("P", 0.5)],
            "2MN": [("P", lam), ("U", 0.5), ("P", 1 - 2 * lam), ("U", 0.5), ("P", lam)]}[case["integrator"]]

    def hamiltonian(U, p):
        return (-(BETA / 3) * L.plaquette_sum(L.smear(U, levels, rho)) + 0.5 * p.square().sum()).item()

    rng = np.random.default_rng(int(seed))
    energies, accepted, plaquettes = [], [], []
    for k in range(case["trajectories"]):
        p = _momenta(_dims(case), seed, k).reshape(L.shape[:-2] + (8,))
        old, F, h0 = U, None, hamiltonian(U, p)
        for _ in range(steps):
            for what, x in step:
                if what == "U":
                    U, F = L.mul(L.exponential(x * e * p), U), None
                else:
                    F = L.force(U, levels, rho) if F is None else F
                    p = p + x * e * F
        h1 = hamiltonian(U, p)
        ok = rng.random() < math.exp(min(0.0, h0 - h1))
        U = U if ok else old
        energies.append((h0, h1))
        accepted.append(int(ok))
        plaquettes.append(L.plaquette_sum(U).item() / (18 * _volume(case)))
    return {"hamiltonians": np.array(energies), "accepted": np.array(accepted), "plaquettes": np.array(plaquettes),
            "links": _reference_layout(U)}


def _exact_flow(case, L, U):
    eps, a, rows = 0.01, 0.0, []
    for n in range(1, case["steps"] + 1):
        for alpha, beta in ((-eps / 4, 0.0), (-8 * eps / 9, -17 / 9), (-3 * eps / 4, -1.0)):
            a = alpha * L.algebra(L.mul(U, L.staples(U))) + beta * a
            U = L.mul(L.exponential(a), U)
        if n % case["every"] == 0:
            p = L.plaquette_sum(U).item() / _volume(case)
            row = [2 * (18 - p)]
            if case["observables"]:
                q, energy = L.field_strengths(U)
                row = [eps * n, p / 18, 2 * (18 - p), energy.item()] + [q[m].sum().item() for m in ("plaquette", "clover", "improved")]
            rows.append(row)
    rows = np.array(rows)
    if case["observables"]:
        return {"rows": rows, "links": _reference_layout(U)}
    return {"energy": rows[:, 0], "links": _reference_layout(U)}


def _momenta(dims, seed, sweep):
    """Gaussian momenta of stream (seed, sweep): Philox4x32-10 (Salmon et al., SC'11) at counter
    (site, 1 << 24 | direction << 16 | block, sweep), Box-Muller pairs from two 53-bit uniforms"""
    v = math.prod(dims)
    site = np.arange(v, dtype=np.uint64)
    out = np.empty((4, v, 8))
    low = np.uint64(0xFFFFFFFF)
    for mu in range(4):
        for b in range(4):
            c = [site, np.full(v, (1 << 24) | (mu << 16) | b, np.uint64), np.full(v, sweep & 0xFFFFFFFF, np.uint64),
                 np.full(v, sweep >> 32, np.uint64)]
            k = [seed & 0xFFFFFFFF, (seed >> 32) & 0xFFFFFFFF]
            for _ in range(10):
                x, y = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
                c = [(y >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), y & low, (x >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), x & low]
                k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
            u = [((c[i] >> np.uint64(5)).astype(np.float64) * 2.0 ** 26 + (c[i + 1] >> np.uint64(6)).astype(np.float64) + 0.5) * 2.0 ** -53
                 for i in (0, 2)]
            r = np.sqrt(-2 * np.log(u[0]))
            out[mu, :, 2 * b], out[mu, :, 2 * b + 1] = r * np.cos(2 * np.pi * u[1]), r * np.sin(2 * np.pi * u[1])
    return torch.from_numpy(out).to(DEV)


class _Torch:
    """SU(3) lattice formulas on whole fields (4, NT, NZ, NY, NX, 3, 3)"""

    def __init__(self, dims):
        nx, ny, nz, nt = dims
        self.shape = (4, nt, nz, ny, nx, 3, 3)

    @staticmethod
    def mul(a, b):
        return sum(a[..., :, k:k + 1] * b[..., k:k + 1, :] for k in range(3))

    @staticmethod
    def at(f, mu, n=1):
        """f(x + n mu) of a field (NT, NZ, NY, NX, ...)"""
        return torch.roll(f, -n, 3 - mu)

    def plaquette_sum(self, U):
        s = 0.0
        for m in range(4):
            for n in range(m + 1, 4):
                s = s + (self.mul(U[m], self.at(U[n], m)) * self.mul(U[n], self.at(U[m], n)).conj()).real.sum()
        return s

    def staples(self, U):
        """Sigma_mu with sum_plaquettes tr(U_mu Sigma_mu)"""
        out = []
        for m in range(4):
            s = 0
            for n in range(4):
                if n != m:
                    up = self.mul(self.mul(self.at(U[n], m), self.at(U[m], n).mH), U[n].mH)
                    low = self.at(self.mul(self.mul(U[m], self.at(U[n], m)).mH, U[n]), n, -1)
                    s = s + up + low
            out.append(s)
        return torch.stack(out)

    @staticmethod
    def algebra(m):
        """Im tr(lambda_a m)"""
        e = lambda i, j: m[..., i, j]  # noqa: E731
        return torch.stack([(e(0, 1) + e(1, 0)).imag, (e(0, 1) - e(1, 0)).real, (e(0, 0) - e(1, 1)).imag,
                            (e(0, 2) + e(2, 0)).imag, (e(0, 2) - e(2, 0)).real, (e(1, 2) + e(2, 1)).imag,
                            (e(1, 2) - e(2, 1)).real, (e(0, 0) + e(1, 1) - 2 * e(2, 2)).imag / math.sqrt(3)], -1)

    def exponential(self, c):
        """exp(i sum_a c_a lambda_a / 2), Taylor series"""
        h = [0.5 * c[..., a] for a in range(8)]
        d = h[7] / math.sqrt(3)
        z = torch.zeros_like(d)
        rows = [torch.complex(z, h[2] + d), torch.complex(h[1], h[0]), torch.complex(h[4], h[3]),
                torch.complex(-h[1], h[0]), torch.complex(z, d - h[2]), torch.complex(h[6], h[5]),
                torch.complex(-h[4], h[3]), torch.complex(-h[6], h[5]), torch.complex(z, -2 * d)]
        x = torch.stack(rows, -1).reshape(c.shape[:-1] + (3, 3))
        one = torch.eye(3, device=x.device, dtype=x.dtype)
        terms = 24 if c.abs().max() > 0.5 else 15
        y = one + x / terms
        for n in range(terms - 1, 0, -1):
            y = one + self.mul(x, y) / n
        return y

    def smear(self, U, levels, rho):
        for _ in range(levels):
            U = self.mul(self.exponential(-rho * self.algebra(self.mul(U, self.staples(U)))), U)
        return U

    def force(self, U, levels, rho):
        """-dV/dU of V = -(beta / 3) sum Re tr P(smeared U) along the generators i lambda_a / 2"""
        if not levels:
            return -(BETA / 6) * self.algebra(self.mul(U, self.staples(U)))
        with torch.enable_grad():
            W = U.detach().requires_grad_(True)
            V = -(BETA / 3) * self.plaquette_sum(self.smear(W, levels, rho))
            G, = torch.autograd.grad(V, W)
        return 0.5 * self.algebra(self.mul(U, G.mH))

    def _loop(self, U, steps):
        """product of the links along a closed walk of (direction, signed length) from every x"""
        at, out = [0] * 4, None

        def moved(f):
            return torch.roll(f, [-n for n in at], [3 - d for d in range(4)])

        for d, n in steps:
            for _ in range(abs(n)):
                if n < 0:
                    at[d] -= 1
                link = moved(U[d])
                link = link.mH if n < 0 else link
                out = link if out is None else self.mul(out, link)
                if n > 0:
                    at[d] += 1
        return out

    def field_strengths(self, U):
        """charge densities by method and the clover energy density"""
        def corners(m, n, a, b):
            return [[(m, a), (n, b), (m, -a), (n, -b)], [(n, b), (m, -a), (n, -b), (m, a)],
                    [(n, -b), (m, a), (n, b), (m, -a)], [(m, -a), (n, -b), (m, a), (n, b)]]

        sets = {"plaquette": {}, "clover": {}, "rectangle": {}}
        for m in range(4):
            for n in range(m + 1, 4):
                leaves = [self._loop(U, w) for w in corners(m, n, 1, 1)]
                sets["plaquette"][m, n] = self.algebra(leaves[0])
                sets["clover"][m, n] = self.algebra(sum(leaves))
                sets["rectangle"][m, n] = self.algebra(sum(self._loop(U, w) for w in corners(m, n, 2, 1) + corners(m, n, 1, 2)))

        def charge(c, loops, norm):
            dot = (c[0, 1] * c[2, 3] - c[0, 2] * c[1, 3] + c[0, 3] * c[1, 2]).sum(-1)
            return norm * dot / (8 * math.pi ** 2 * loops ** 2)

        q = {"plaquette": charge(sets["plaquette"], 1, 1.0), "clover": charge(sets["clover"], 4, 1.0)}
        q["improved"] = 5 / 3 * q["clover"] - charge(sets["rectangle"], 8, 2.0) / 12
        energy = sum(c.square().sum() for c in sets["clover"].values()) / 32 / math.prod(self.shape[1:5])
        return q, energy

