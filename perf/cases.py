"""The work that a user of this framework has it do, as measured cases.

A pass takes a particle system through a frame of its run, by the public entry points: `steps` whole steps of a driver, then the download of the frame.
A program that runs one of the reference's drivers does that between two outputs.  The mixed form computes its pairs in FP32, and programs that use it keep
their frames so: its fields are handed on as float32, those of the FP64 form as float64.

`exact` repeats the same steps in plain torch, in 64 bits.  The Wendland kernel's casts to float are part of its definition (src/SPH_kernel.h:52-77), so they
are in there too.
"""
import math

import numpy as np
import torch

import tinysph_old_amd as T

PRECISION = {"fp64": T.PREC_FP64, "mixed": T.PREC_MIXED}
PRESET = {"still": T.CASE_STILL_WATER_DBC, "dam": T.CASE_DAM_BREAK_MDBC, "bt": T.CASE_DAM_BREAK_BT, "ale": T.CASE_ALE_DAM_BREAK,
          "rale": T.CASE_ALE_DAM_BREAK, "inflow": T.CASE_INFLOW_CHANNEL, "driver": T.CASE_DAM_BREAK_MDBC_REF}
# fluid area of the presets (m^2): about area / dx^2 particles
AREA = {"still": 0.5, "dam": 0.72, "bt": 0.18, "ale": 0.72, "rale": 0.72, "inflow": 0.99, "driver": 0.18}
FIELDS = ("r", "v", "rho", "p")
# the reference's water-level gauges (x, y0, inverse) and wall sensors (x, y) of the 1.61 x 1.0 m tank
GAUGES = [(0.3, 0.0, False), (0.3, 0.45, True), (0.865, 0.0, False), (0.865, 0.45, True)]
SENSORS = [(1.61, 0.003), (1.61, 0.015), (0.3, 0.03), (0.3, 0.08)]


def listed():
    return [
        # still water with dynamic walls, the size that also runs on a CPU: launches and latency count
        {"name": "still_fp64_6k", "kind": "still", "prec": "fp64", "dx": 0.01, "steps": 50},
        # the reference's own dam break at its own spacing, its driver calling stage by stage, with gauges and wall sensors after the steps
        {"name": "driver_fp64_8k", "kind": "driver", "prec": "fp64", "dx": 0.005, "steps": 10},
        # the reference's other wall treatment, in a small study: an odd spacing
        {"name": "bt_mixed_21k", "kind": "bt", "prec": "mixed", "dx": 0.0031, "steps": 50},
        # a dam break of ordinary size, both forms
        {"name": "dam_mixed_50k", "kind": "dam", "prec": "mixed", "dx": 0.004, "steps": 50},
        {"name": "dam_fp64_90k", "kind": "dam", "prec": "fp64", "dx": 0.0029, "steps": 40},
        # the benchmark's dam break, both forms
        {"name": "dam_mixed_740k", "kind": "dam", "prec": "mixed", "dx": 0.001, "steps": 100},
        {"name": "dam_fp64_740k", "kind": "dam", "prec": "fp64", "dx": 0.001, "steps": 60},
        # ALE-SPH with limited MUSCL reconstruction, both forms
        {"name": "ale_mixed_183k", "kind": "ale", "prec": "mixed", "dx": 0.002, "steps": 20},
        {"name": "ale_fp64_183k", "kind": "ale", "prec": "fp64", "dx": 0.002, "steps": 20},
        # first-order Riemann-ALE, as the reference's ALE driver runs
        {"name": "rale_fp64_47k", "kind": "rale", "prec": "fp64", "dx": 0.004, "steps": 30},
        # many tanks advanced together, 2,000 to 100,000 particles each
        {"name": "ensemble_mixed_16", "kind": "ensemble", "prec": "mixed", "tanks": 16, "geometry": 20241202, "nmin": 2000, "nmax": 100000, "steps": 50},
        # channel flow with inlet and outlet zones, mixed with compensated integration
        {"name": "inflow_mixed_1m", "kind": "inflow", "prec": "mixed", "dx": 0.001, "steps": 40},
    ]


# particles and steps that a drawn case may have, and how much a particle's step weighs (FP64 pairs cost about twice the mixed ones)
RANGE = {"still": (2000, 60000, 20, 80), "driver": (3000, 30000, 4, 20), "bt": (3000, 200000, 20, 80), "dam": (4000, 740000, 20, 100),
         "ale": (8000, 183000, 5, 20), "rale": (8000, 183000, 10, 40), "inflow": (30000, 1000000, 10, 40)}
MOST = 740000 * 60 * 2  # particles x steps x weight of the largest listed case


def _between(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["still", "driver", "bt", "dam", "dam", "dam", "ale", "ale", "rale", "ensemble", "inflow"])
    prec = "mixed" if kind == "inflow" else rng.choice(["fp64", "mixed"])
    if kind == "ensemble":
        return {"kind": kind, "prec": prec, "tanks": rng.randrange(3, 17), "geometry": rng.randrange(1 << 30), "nmin": 2000,
                "nmax": int(_between(rng, 5000, 100000)), "steps": rng.randrange(10, 41)}
    lo, hi, s0, s1 = RANGE[kind]
    n = _between(rng, lo, hi)
    weight = {"fp64": 2, "mixed": 1}[prec]
    steps = min(rng.randrange(s0, s1 + 1), int(MOST / (n * weight)))
    return {"kind": kind, "prec": prec, "dx": round(math.sqrt(AREA[kind] / n), 7), "steps": max(steps, 1)}


# ---- inputs ----------------------------------------------------------------------------------------------------------------------------
def _flow(arrays, seed, q=0):
    """A smooth flow of about 0.1 m/s, divergence-free, on top of the preset's own: its phases and wave lengths come from the seed."""
    g = np.random.RandomState((seed * 7919 + q * 104729 + 1) % (1 << 31))
    r, fluid = arrays["r"], arrays["type"] == T.FLUID
    v = arrays["v"].copy()
    for _ in range(3):
        kx, ky, ph = g.uniform(2.0, 12.0), g.uniform(2.0, 12.0), g.uniform(0, 2 * math.pi)
        c = 0.05 * np.cos(kx * r[:, 0] + ky * r[:, 1] + ph) / math.hypot(kx, ky)
        v[:, 0] += np.where(fluid, c * ky, 0.0)
        v[:, 1] -= np.where(fluid, c * kx, 0.0)
    arrays["v"] = v


def _inputs(case, seed):
    if case["kind"] == "ensemble":
        cs = T.build_ensemble(case["tanks"], case["geometry"], case["nmin"], case["nmax"])
    else:
        cs = [T.build_case(PRESET[case["kind"]], dx=case["dx"], jitter=0.02, seed=seed)]
    for q, c in enumerate(cs):
        _flow(c.arrays, seed, q)
    return cs


def prepare(case, seed):
    cs = _inputs(case, seed)
    kind, prec = case["kind"], PRECISION[case["prec"]]
    if kind == "ensemble":
        ps = T.batch_for_cases(cs, prec)
        ps.particle_to_cell()
        ps.density_to_pressure()
        ps.compute_forces(T.FORCES_WCSPH)
        ps.synchronize()
        return {"case": case, "ps": ps, "wall": T.WALL_MDBC, "step": 1}
    c = cs[0]
    ps = T.system_for_case(c, precision=prec)
    if kind in ("ale", "rale"):
        ps.ale_enable()
        ps.particle_to_cell()
    else:
        if kind == "inflow":
            ps.set_compensated(True)
        ps.particle_to_cell()
        ps.density_to_pressure()
        ps.compute_forces(T.forces_variant(c.wall))
    ps.synchronize()
    return {"case": case, "ps": ps, "wall": c.wall, "dt": c.dt, "step": 1}


# ---- one pass --------------------------------------------------------------------------------------------------------------------------
def _driver(ps, wall, dt, steps):
    """The reference's symplectic driver as it calls its stages (cases/damBreakLong_mDBC/SPH_simulationSymplectic.h:59-116)."""
    variant = T.forces_variant(wall)
    for _ in range(steps):
        ps.mdbc_density()
        ps.density_to_pressure()
        ps.predictor(dt)
        ps.clear_cells()
        ps.particle_to_cell()
        ps.density_to_pressure()
        ps.compute_forces(variant)
        ps.corrector(dt)
        ps.remove_out_of_domain()
        ps.clear_cells()
        ps.particle_to_cell()
        ps.density_to_pressure()
        ps.compute_forces(variant)


def run(state):
    case, ps, steps, wall = state["case"], state["ps"], state["case"]["steps"], state["wall"]
    kind, first = case["kind"], state["step"]
    state["step"] = first + steps
    kept = np.float32 if case["prec"] == "mixed" else np.float64
    if kind == "ensemble":
        ps.step(wall, steps)
        frames = [ps.download_case(q, FIELDS) for q in range(ps.ncases)]
        return {k: np.concatenate([f[k] for f in frames]).astype(kept, copy=False) for k in FIELDS}
    dt, out = state["dt"], {}
    if kind == "driver":
        _driver(ps, wall, dt, steps)
        out["gauges"] = [ps.water_elevation(x, y0, inverse) for x, y0, inverse in GAUGES]
        out["sensors"] = np.stack([ps.interpolate_point(x, y) for x, y in SENSORS])
    elif kind == "ale":
        ps.step_ale(dt, first, steps, T.MUSCL_MINMOD)
    elif kind == "rale":
        ps.step_rale(dt, first, steps)
    elif kind == "inflow":
        ps.step_inflow(wall, dt, steps)
    else:
        ps.step(wall, dt, steps)
    out.update({k: v.astype(kept, copy=False) for k, v in ps.download(FIELDS).items()})
    return out


def work(case):
    """The state read once and the frame written once; per step, every pair inside the support is computed once a pair pass
    (pi (2h)^2 / dx^2 neighbours: h = 1.5 dx for still water, sqrt(2) dx otherwise)."""
    kind, steps = case["kind"], case["steps"]
    if kind == "ensemble":
        n = sum(c.np for c in T.build_ensemble(case["tanks"], case["geometry"], case["nmin"], case["nmax"]))
    else:
        n = AREA[kind] / case["dx"] ** 2
    pairs = n * math.pi * 4 * (2.25 if kind == "still" else 2.0)
    # state: r, v, rho, p, a, drho, type; the ALE forms also omega, omega rho, omega v and their rates; frame: r, v, rho, p
    state = 73 + (64 if kind in ("ale", "rale") else 0)
    passes, flops = {"ale": (3, 130), "rale": (1, 110)}.get(kind, (2, 60))
    return {"bytes": float(n * (state + (48 if case["prec"] == "fp64" else 24))), "flops": float(pairs * passes * flops * steps)}


# ---- the same steps in plain torch, 64 bits ------------------------------------------------------------------------------------------------
ROWS = 120000  # particles whose neighbours are gathered together


def _neighbours(pts, query, radius, same):
    """Indices into pts of the points within `radius` of each query point, as rows padded with -1 (`same`: a point is not its own neighbour)."""
    lo = torch.minimum(pts.amin(0), query.amin(0)) - radius
    ny = int(((torch.maximum(pts.amax(0), query.amax(0)) - lo)[1] / radius).item()) + 4
    cell = lambda x: ((x - lo) / radius).long() + 1  # noqa: E731
    pc, qc = cell(pts), cell(query)
    key, order = torch.sort(pc[:, 0] * ny + pc[:, 1])
    rows, most = [], 0
    for a in range(0, len(query), ROWS):
        c, x = qc[a:a + ROWS], query[a:a + ROWS]
        base = torch.stack([(c[:, 0] + d) * ny + c[:, 1] for d in (-1, 0, 1)], 1).reshape(-1)
        start, end = torch.searchsorted(key, base - 1), torch.searchsorted(key, base + 2)
        count = end - start
        i = torch.repeat_interleave(torch.arange(len(base), device=pts.device), count)
        j = order[torch.arange(len(i), device=pts.device) - (torch.cumsum(count, 0) - count)[i] + start[i]]
        i = i // 3
        d = x[i] - pts[j]
        keep = (d * d).sum(1) <= radius * radius
        if same:
            keep &= j != i + a
        i, j = i[keep], j[keep]
        n = torch.bincount(i, minlength=len(x))
        rows.append((i, j, torch.arange(len(i), device=pts.device) - (torch.cumsum(n, 0) - n)[i], len(x)))
        most = max(most, int(n.max()) if len(i) else 0)
    out = torch.full((len(query), max(most, 1)), -1, dtype=torch.long, device=pts.device)
    a = 0
    for i, j, slot, m in rows:
        out[i + a, slot] = j
        a += m
    return out


class Exact:
    def __init__(self, c):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        p, A = c.params, c.arrays
        put = lambda x: torch.as_tensor(np.ascontiguousarray(x)).to(dev)  # noqa: E731
        self.h, self.cs, self.rho0, self.dp, self.dt = p["h"], p["cs"], p["rho0"], p["dp"], c.dt
        self.alpha, self.delta, self.wall, self.zones = p["avisc"], p["delta"], c.wall, c.zones
        self.m, self.g = p["rho0"] / (1 / p["dp"] * 1 / p["dp"]), 9.81
        self.awen = float(np.float32(0.557 / (p["h"] * p["h"])))
        self.bwen = float(np.float32(-2.7852 / (p["h"] * p["h"] * p["h"])))
        self.r, self.v, self.rho, self.p = (put(A[k]) for k in FIELDS)
        self.type = put(A["type"])
        self.gnr = put(A["gnr"]) if "gnr" in A else None
        self.n = put(A["n"]) if "n" in A else torch.zeros_like(self.r)
        self.a, self.drho = torch.zeros_like(self.r), torch.zeros_like(self.rho)
        self.at, self.list = None, None

    # pairs: lists with a skin, rebuilt once the particles could have crossed it
    def pairs(self):
        skin = 0.3 * self.h
        if self.at is None or len(self.at) != len(self.r) or float((self.r - self.at).square().sum(1).max()) > (skin / 2) ** 2:
            self.at, self.list = self.r.clone(), _neighbours(self.r, self.r, 2 * self.h + skin, True)
        for a in range(0, len(self.r), ROWS):
            i = torch.arange(a, min(a + ROWS, len(self.r)), device=self.r.device)
            j = self.list[a:a + ROWS]
            yield i, j.clamp(min=0), j >= 0

    def kernel(self, drs):
        q = drs / self.h
        w1 = (1.0 - 0.5 * q).float()
        w2 = (w1 * w1).double()
        return (self.awen * (q + q + 1.0).float().double() * w2 * w2, self.bwen * q * w2 * w1.double() / drs)

    def geometry(self, i, j, ok):
        dr = self.r[i][:, None] - self.r[j]
        drs = dr.square().sum(2).sqrt()
        ok = ok & (drs / self.h <= 2.0)
        drs = torch.where(ok, drs, self.h)
        w, f = self.kernel(drs)
        return dr, drs, torch.where(ok, w, 0.0), torch.where(ok, f, 0.0), ok

    def eos(self):
        self.p = self.cs ** 2 * self.rho0 / 7.0 * ((self.rho / self.rho0) ** 7 - 1)

    def forces(self):
        wall = self.type == T.WALL
        for i, j, ok in self.pairs():
            wi, wj = wall[i][:, None], wall[j]
            if self.wall == T.WALL_DBC:
                ok = ok & ~(wi & wj)
            dr, drs, w, f, ok = self.geometry(i, j, ok)
            dv, rho, nrho = self.v[i][:, None] - self.v[j], self.rho[i][:, None], self.rho[j]
            drdv = (dr * dv).sum(2)
            pt = (self.p[i][:, None] + self.p[j]) / (rho * nrho)
            d = drs * drs + 0.01 * self.h * self.h
            mu = self.h * drdv / d
            pt = pt + torch.where(drdv < 0, -drdv.clamp(min=self.alpha) * self.cs * mu / (0.5 * (rho + nrho)), 0.0)
            dW = dr * f[..., None]
            drhoH = self.rho0 * torch.expm1(torch.log1p(dr[..., 1] * self.rho0 * self.g / (self.cs ** 2 * self.rho0 / 7.0)) / 7)
            psi = 2 * self.cs * self.h * self.delta * ((nrho - rho) - drhoH) / d
            fl = ~wj if self.wall == T.WALL_BT else torch.ones_like(wj)
            acc = -(dW * (torch.where(fl, pt, 0.0) * self.m)[..., None]).sum(1)
            con = ((dv * dW).sum(2) * fl).sum(1) * self.m
            dif = -(psi * (dr * dW).sum(2) * self.m / nrho * fl).sum(1)
            if self.wall == T.WALL_BT:
                nb, ww = self.n[j], torch.where(wj, w, 0.0)
                acc = acc + (nb * (ww * pt * self.dp * nrho)[..., None]).sum(1)
                con = con - ((dv * nb).sum(2) * ww * nrho * self.dp).sum(1)
                gamma = (torch.where(wj, 0.0, w) * self.m / nrho).sum(1)
                some = gamma > 0.01
                gamma = torch.where(some, gamma, 1.0)
                acc, con, dif = (torch.where(some if x.dim() == 1 else some[:, None], x / (gamma if x.dim() == 1 else gamma[:, None]), 0.0) for x in (acc, con, dif))
            acc[:, 1] -= self.g
            if self.wall == T.WALL_DBC:
                acc[wall[i]] = 0.0
                act = torch.ones_like(i, dtype=torch.bool)
            else:
                act = self.type[i] == T.FLUID
            self.a[i[act]], self.drho[i[act]] = acc[act], (con + dif)[act]

    def walls(self):
        at = torch.nonzero(self.type == T.WALL)[:, 0]
        if self.wall == T.WALL_DBC or not len(at):
            return
        q = self.gnr[at] if self.wall == T.WALL_MDBC else self.r[at]
        j = _neighbours(self.r, q, 2 * self.h * 1.000001, False)
        ok = (j >= 0) & (self.type[j.clamp(min=0)] == T.FLUID)
        j = j.clamp(min=0)
        dr = q[:, None] - self.r[j]
        drs = dr.square().sum(2).sqrt()
        ok = ok & (drs / self.h <= 2.0)
        drs = torch.where(ok, drs, self.h)
        w, f = self.kernel(drs)
        w, f, mr = torch.where(ok, w, 0.0), torch.where(ok, f, 0.0), self.m / self.rho[j]
        if self.wall == T.WALL_BT:
            s = (w * mr).sum(1)
            rho = torch.where(s > 0, (self.m * w).sum(1) / torch.where(s > 0, s, 1.0), 1000.0)
        else:
            x, y = dr[..., 0], dr[..., 1]
            M = torch.stack([(t * mr).sum(1) for t in (w, x * w, y * w, x * f, x * x * f, x * y * f, y * f, y * x * f, y * y * f)], 1).reshape(-1, 3, 3)
            b = torch.stack([(t * self.m).sum(1) for t in (w, x * f, y * f)], 1)
            det = torch.linalg.det(M)
            good = det > 0.001
            s = torch.linalg.solve(torch.where(good[:, None, None], M, torch.eye(3, dtype=M.dtype, device=M.device)), b[..., None])[..., 0]
            d = self.r[at] - q
            full = s[:, 0] - s[:, 1] * d[:, 0] - s[:, 2] * d[:, 1]
            shep = torch.where(M[:, 0, 0] > 0, b[:, 0] / torch.where(M[:, 0, 0] > 0, M[:, 0, 0], 1.0), 1000.0)
            rho = torch.where(good, full, shep)
        self.rho[at] = rho.clamp(min=1000.0)

    def inlet(self, z):
        at = torch.nonzero((self.type == z["btype"]) & (self.r[:, 0] > z["x0"]))[:, 0]
        if not len(at):
            return
        new = self.r[at].clone()
        new[:, 0] -= abs(z["xm"] - z["x0"])
        self.type[at] = T.FLUID
        vin = torch.tensor([z["vx"], z["vy"]], dtype=new.dtype, device=new.device).expand(len(at), 2)
        zero, rest = torch.zeros_like(new), torch.full_like(new[:, 0], 1000.0)
        for k, x in (("r", new), ("v", vin), ("a", zero), ("ro", new), ("vo", vin), ("gnr", zero), ("n", zero), ("rho", rest), ("rhoo", rest),
                     ("p", zero[:, 0]), ("drho", zero[:, 0]), ("type", torch.full_like(at, z["btype"]).to(self.type.dtype))):
            setattr(self, k, torch.cat([getattr(self, k), x]))

    def outlet(self, z):
        gone = (self.type == z["btype"]) & ((self.r[:, 0] > z["x0"] + abs(z["xm"] - z["x0"])) | (self.r[:, 1] < self.dp / 2))
        conv = (self.type == T.FLUID) & (self.r[:, 0] > z["x0"])
        # the reference erases inside its loop: the particle after an erased one is not looked at
        run = torch.zeros(len(gone) + 1, dtype=torch.long)
        for s in torch.nonzero(gone)[:, 0].tolist():
            run[s + 1] = run[s] + 1
        odd = (run[:-1] % 2 == 1).to(gone.device)
        gone, conv = gone & ~odd, conv & ~odd & ~gone
        self.type[conv], self.a[conv], self.drho[conv] = z["btype"], 0.0, 0.0
        if bool(gone.any()):
            for k in ("r", "v", "a", "ro", "vo", "gnr", "n", "rho", "rhoo", "p", "drho", "type"):
                setattr(self, k, getattr(self, k)[~gone])

    def symplectic(self, zones=False):
        dt = self.dt
        self.walls()
        self.ro, self.vo, self.rhoo = self.r, self.v, self.rho.clone()
        self.rho = self.rho + self.drho * dt * 0.5
        self.r, self.v = self.r + self.v * dt * 0.5, self.v + self.a * dt * 0.5
        if zones:
            self.inlet(self.zones[0])
            self.outlet(self.zones[1])
        self.eos()
        self.forces()
        e = -self.drho / self.rho * dt
        self.rho, v = self.rhoo * ((2 - e) / (2 + e)), self.vo + self.a * dt
        self.r, self.v = self.ro + (v + self.vo) * dt * 0.5, v
        self.eos()
        self.forces()

    # ---- the ALE forms
    def ale_start(self):
        w = torch.full_like(self.rho, self.dp * self.dp)
        self.om, self.omr, self.omv = w, self.rho * w, self.v * w[:, None]
        self.dom, self.domr, self.domv = torch.zeros_like(w), torch.zeros_like(w), torch.zeros_like(self.v)
        self.grad = torch.zeros(len(w), 3, 2, dtype=w.dtype, device=w.device)  # rho, vx, vy

    def states(self, i, j, dr):
        """Left and right {rho, vx, vy} of a pair, reconstructed with the minmod weight."""
        u = torch.cat([self.rho[:, None], self.v], 1)
        a, b, ga, gb = u[i][:, None], u[j], self.grad[i][:, None], self.grad[j]
        sa, sb = (ga * dr[..., None, :]).sum(-1), (gb * dr[..., None, :]).sum(-1)

        def weight(c, d, s):
            flat = d - c == 0
            return torch.where(flat, 0.0, (2 * s / torch.where(flat, 1.0, d - c) - 1).clamp(0.0, 1.0))

        return a + weight(a, b, -sa) * 0.5 * sa, b - weight(b, a, sb) * 0.5 * sb

    def riemann(self, L, R, dn, c, rho_i, rho_j, v_i, v_j):
        vl, vr = (L[..., 1:] * dn).sum(-1), (R[..., 1:] * dn).sum(-1)
        avg, d = 0.5 * (L[..., 0] + R[..., 0]), vl - vr
        beta = torch.minimum(3 * d.clamp(min=0.0), c)
        rhos = avg + 0.5 * beta * d * avg / (c * c)
        vss = 0.5 * (vl + vr) - 0.5 * (rho_j - rho_i) * c / avg
        return rhos, dn * (vss - (vl + vr) * 0.5)[..., None] + (v_i + v_j) * 0.5

    def ale_pass(self, what):
        fluid, wall, c0 = self.type == T.FLUID, self.type == T.WALL, torch.as_tensor(self.cs, dtype=self.r.dtype, device=self.r.device)
        for i, j, ok in self.pairs():
            dr, drs, w, f, ok = self.geometry(i, j, ok)
            wj, act, dW = wall[j], fluid[i], dr * f[..., None]
            rho, nrho, om, v, nv = self.rho[i][:, None], self.rho[j], self.om[j], self.v[i][:, None], self.v[j]
            nb, ww, fl = -self.n[j], torch.where(wj, w, 0.0), (~wj).double()
            if what == "gradient":
                d = torch.stack([nrho - rho, nv[..., 0] - v[..., 0], nv[..., 1] - v[..., 1]], 2)[..., None]
                t = d * ((nb * ww[..., None] * self.dp) + dW * (om * fl)[..., None])[:, :, None]
                self.new[i[act]] = (2 * t.sum(1))[act]
                continue
            dn = -dr / drs[..., None]
            if what == "first":
                L, R = torch.cat([rho[..., None], v], 2).expand(-1, j.shape[1], -1), torch.cat([nrho[..., None], nv], 2)
            else:
                L, R = self.states(i, j, dr)
            c = c0 if what != "acceleration" else self.cs * ((rho / self.rho0).sqrt() + (nrho / self.rho0).sqrt())
            rhos, vs = self.riemann(L, R, dn, c, rho if what == "acceleration" else L[..., 0], nrho if what == "acceleration" else R[..., 0], v, nv)
            e = vs - v
            if what in ("density", "first"):
                dom = -(((v - nv) * nb).sum(2) * ww).sum(1) * self.dp
                if what == "first":
                    dom = dom - (((v - nv) * dW).sum(2) * om * fl).sum(1)
                domr = -2 * (rhos * om * (e * dW).sum(2) * fl).sum(1)
                self.dom[i[act]], self.domr[i[act]] = (dom * self.om[i])[act], (domr * self.om[i])[act]
            if what in ("acceleration", "first"):
                first = what == "first"
                ps = self.cs ** 2 * self.rho0 / 7.0 * ((rhos / self.rho0) ** 7 - 1) if first else self.cs ** 2 * (rhos - self.rho0)
                rw = L[..., 0] + (L[..., 1:] * nb).sum(2) * L[..., 0] / self.cs
                pw = self.cs ** 2 * (rw - (self.rho0 if first else 1000.0))
                flux = rhos[..., None] * vs * (e * dW).sum(2)[..., None] + ps[..., None] * dW
                acc = -2 * (flux * (om * fl)[..., None] + nb * (ww * self.dp * pw)[..., None]).sum(1) * self.om[i][:, None]
                acc[:, 1] -= self.g * self.om[i] * self.rho[i]
                self.domv[i[act]] = acc[act]

    def ale(self, step):
        dt, fl = self.dt, self.type == T.FLUID
        on, on2 = fl.double(), fl.double()[:, None]
        if step > 1:
            self.omv = self.omv + self.domv * dt * 0.5 * on2
            self.v = torch.where(fl[:, None], self.omv / (self.rho * self.om)[:, None], self.v)
        self.ale_pass("density")
        self.new = self.grad.clone()
        self.ale_pass("gradient")
        self.grad = self.new
        self.om, self.omr = self.om + self.dom * dt * on, self.omr + self.domr * dt * on
        self.rho = torch.where(fl, self.omr / self.om, self.rho)
        self.p = torch.where(fl, (self.cs ** 2 * (self.rho - self.rho0)).clamp(min=0.0), self.p)
        self.ale_pass("acceleration")
        k = 0.5 if step == 1 else 1.0
        self.omv = self.omv + self.domv * dt * k * on2
        self.v = torch.where(fl[:, None], self.omv / (self.rho * self.om)[:, None], self.v)
        self.r = self.r + self.v * dt * k * on2

    def rale(self, step):
        dt, on = self.dt, (self.type == T.FLUID).double()
        on2 = on[:, None]
        was = (self.om, self.omr, self.omv)

        def move(base, k):
            self.om, self.omr = base[0] + self.dom * dt * k * on, base[1] + self.domr * dt * k * on
            self.omv = base[2] + self.domv * dt * k * on2
            self.rho = torch.where(on > 0, self.omr / self.om, self.rho)
            self.v = torch.where(on2 > 0, self.omv / (self.rho * self.om)[:, None], self.v)

        if step > 1:
            move(was, 0.5)
        self.eos()
        self.ale_pass("first")
        if step == 1:
            move(was, 0.5)
            self.r = self.r + self.v * dt * 0.5 * on2
        else:
            self.r = self.r + self.v * dt * on2
            move(was, 1.0)


def exact(case, seed):
    kind, frames = case["kind"], []
    for c in _inputs(case, seed):
        X = Exact(c)
        if kind in ("ale", "rale"):
            X.ale_start()
            for s in range(1, case["steps"] + 1):
                getattr(X, kind)(s)
        else:
            X.eos()
            X.forces()
            for _ in range(case["steps"]):
                X.symplectic(kind == "inflow")
        frames.append(X)
    out = {k: torch.cat([getattr(X, k) for X in frames]).cpu().numpy() for k in FIELDS}
    if kind == "driver":  # a gauge marches in steps of its own, a sensor averages over the reference's stencil: no plain value
        out["gauges"], out["sensors"] = [None] * len(GAUGES), None
    return out
