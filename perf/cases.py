"""Performance cases of the SPH cutting solver: what a program asks of it through pymfc.

A pass of most cases is what the solver's callers do between two dumps: queue a block of steps,
then read the tool-force log and the particle fields that a dump holds (storage order, with the
creation ids). The batch and reverse-mode cases are the calibration workloads. Launch settings
are the library's defaults. Lattices carry a 1 % jitter (the rings: perturbed velocities), which
is what a seed changes.

exact() restates the step in plain torch FP64 (no single-precision truncations), from the initial
particles and the tool that the configuration describes.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "mfree_iwf-ul_cut_gpu_amd"))
import pymfc  # noqa: E402

DUMP = ("id", "pos", "vel", "S", "T", "eps_pl")  # the fields a dump reads
PREC = {"fp64": pymfc.PREC_FP64, "fp32c": pymfc.PREC_FP32C}


def _cut(name, nx, ny, dx_um, thermal, speed, prec, steps, kind="cut"):
    return {"name": name, "kind": kind, "nx": nx, "ny": ny, "dx_um": dx_um, "thermal": thermal, "speed": speed,
            "prec": prec, "steps": steps}


def listed():
    return [
        # a monitor loop: one step, then its tool force, velocities and temperatures (6k adiabatic cut);
        # the smallest call, where launches and latency count
        _cut("report_6k_fp64", 150, 40, 10.0, "adiabatic", 70.0, "fp64", 1, kind="report"),
        # the reference main()'s own cut (setup_ref_cut, ny = 30, 7.6k particles with the tool's)
        {"name": "ref_cut_30_fp64", "kind": "ref", "ny": 30, "prec": "fp64", "steps": 100},
        # the 6k adiabatic benchmark cut on the fast path
        _cut("cut_6k_fp32c", 150, 40, 10.0, "adiabatic", 70.0, "fp32c", 200),
        # the calibration cut at 1000 m/min, yielding within the first steps
        _cut("hot_37k_fp64", 375, 100, 4.0, "adiabatic", 1000.0, "fp64", 150),
        # the headline cut (150k workpiece + 47k tool particles, thermal contact), both precisions
        _cut("contact_150k_fp32c", 750, 200, 2.0, "contact", 70.0, "fp32c", 250),
        _cut("contact_150k_fp64", 750, 200, 2.0, "contact", 70.0, "fp64", 150),
        # an odd-sized cut with PSE conduction
        _cut("pse_odd_fp64", 331, 97, 4.0, "pse", 120.0, "fp64", 150),
        # the large PSE cut, the largest state
        _cut("pse_500k_fp32c", 1250, 400, 1.2, "pse", 120.0, "fp32c", 100),
        # colliding rings (setup_rings on a 200 x 200 lattice, 27k particles): elastic, no tool
        {"name": "rings_200_fp64", "kind": "rings", "nbox": 200, "prec": "fp64", "steps": 150},
        # a parameter sweep: 32 uneven cuts stepped together
        {"name": "batch_32_fp32c", "kind": "batch", "n": 32, "prec": "fp32c", "steps": 100},
        # calibration gradients: taped forward and backward pass, small and ordinary
        {"name": "vjp_6k", "kind": "vjp", "nx": 150, "ny": 40, "dx_um": 10.0, "steps": 60, "every": 20},
        {"name": "vjp_37k", "kind": "vjp", "nx": 375, "ny": 100, "dx_um": 4.0, "steps": 100, "every": 50},
    ]


def _log(rng, a, b):
    return math.exp(rng.uniform(math.log(a), math.log(b)))


def draw(rng):
    kind = rng.choice(["cut", "cut", "cut", "cut", "report", "ref", "rings", "batch", "vjp"])
    prec = rng.choice(["fp64", "fp32c"])
    if kind in ("cut", "report"):
        n = _log(rng, 2e3, 4e5 if kind == "cut" else 2e4)
        ny = max(13, int(math.sqrt(n / rng.uniform(2.5, 4.5))))
        thermal, speed = rng.choice([("adiabatic", 70.0), ("adiabatic", 1000.0), ("contact", 70.0), ("contact", 150.0),
                                     ("pse", 120.0)])
        if thermal == "contact":
            ny = min(ny, 200)
        nx = max(31, int(n / ny))
        # the workpiece keeps a height of 0.4 mm, so that the tool's depth of cut fits it
        dx_um = round(400.0 / ny, 2)
        steps = 1 if kind == "report" else max(40, min(250, int(8e6 / n)))
        return {"kind": kind, "nx": nx, "ny": ny, "dx_um": dx_um, "thermal": thermal, "speed": speed, "prec": prec,
                "steps": steps}
    if kind == "ref":
        return {"kind": "ref", "ny": rng.randrange(12, 90), "prec": prec, "steps": rng.randrange(60, 160)}
    if kind == "rings":
        return {"kind": "rings", "nbox": int(_log(rng, 60, 600)), "prec": prec, "steps": rng.randrange(60, 120)}
    if kind == "batch":
        return {"kind": "batch", "n": rng.randrange(2, 25), "prec": prec, "steps": rng.randrange(40, 100)}
    ny = int(_log(rng, 20, 100))
    return {"kind": "vjp", "nx": int(ny * rng.uniform(2.5, 4.0)), "ny": ny, "dx_um": round(400.0 / ny, 2),
            "steps": rng.randrange(30, 90), "every": rng.randrange(10, 40)}


def _configs(case, seed):
    """The solver configurations of a case (several for a batch)."""
    kind = case["kind"]
    prec = PREC[case.get("prec", "fp64")]
    if kind == "rings":
        return [pymfc.config_rings(case["nbox"], prec)]
    if kind == "ref":
        c = pymfc.config_ref_cut(ny=case["ny"])
        c.precision, c.jitter, c.seed = prec, 0.01, seed
        return [c]
    if kind == "batch":
        cfgs = pymfc.batch_configs(case["n"], precision=prec)
        for i, c in enumerate(cfgs):
            c.jitter, c.seed = 0.01, seed * 64 + i
        return cfgs
    c = pymfc.cut_config(case["nx"], case["ny"], case["dx_um"], thermal=case.get("thermal", "adiabatic"),
                         speed_m_min=case.get("speed", 1000.0), jitter=0.01, seed=seed, precision=prec)
    if kind == "vjp":
        c.promote_fp64, c.secant_tol = 1, 1e-14
    return [c]


def _ring_velocities(cfg, seed):
    x = pymfc.scenario(cfg)["pos"][:, 0]
    u = np.random.default_rng(seed).uniform(-1.0, 1.0, (x.size, 2))
    return np.stack([np.where(x < 0, 200.0, -200.0), np.zeros_like(x)], axis=1) + u


def prepare(case, seed):
    cfgs = _configs(case, seed)
    if case["kind"] == "batch":
        sim = pymfc.Batch(cfgs)
    else:
        sim = pymfc.Sim(cfgs[0])
    if case["kind"] == "rings":
        sim.set_field("vel", _ring_velocities(cfgs[0], seed))
    return {"case": case, "sim": sim}


def run(state):
    case, sim = state["case"], state["sim"]
    kind, steps = case["kind"], case["steps"]
    if kind == "report":
        sim.step(1)
        return {"F": sim.tool_force(), "vel": sim.field("vel"), "T": sim.field("T")}
    if kind == "batch":
        for s in sim.instances:
            s.reset_force_history()
        sim.step(steps)
        out = {"F": np.stack([s.force_history() for s in sim.instances])}
        for f in ("pos", "vel", "S"):
            out[f] = np.concatenate([s.field(f) for s in sim.instances])
        return out
    if kind == "vjp":
        sim.reset_force_history()
        F = sim.vjp_forward(steps, case["every"], steps // 2, steps)
        g = sim.vjp_backward(np.array([1.0, 0.5]))
        return {"F": F, "grad": g, "pos": sim.field("pos"), "vel": sim.field("vel")}
    sim.reset_force_history()
    sim.step(steps)
    out = {f: sim.field(f) for f in DUMP}
    if kind != "rings":
        out["F"] = sim.force_history()
    return out


def work(case):
    # per particle and step: the mutable state read and written once with its cell ids and
    # neighbour data, 492 bytes (the benchmark's count); about 26 pairs of some 110 floating-point
    # operations and the particle's own update
    steps = case["steps"] * (3 if case["kind"] == "vjp" else 1)
    n = sum(pymfc.scenario(c)["info"].n_particles for c in _configs(case, 1))
    return {"bytes": 492.0 * n * steps, "flops": 3500.0 * n * steps}


# ------------------------------------------------------------------ the step in plain FP64
PI_FAC = 10.0 / (7.0 * math.pi)
BIG = 3.4028234663852886e38


class _Exact:
    def __init__(self, cfg, vel=None):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        s = pymfc.scenario(cfg)  # the initial particles, grid and tool
        i = s["info"]
        self.c, self.i, self.dev = cfg, i, dev
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), dtype=torch.float64, device=dev)
        N = self.N = i.n_particles
        z = lambda: torch.zeros(N, dtype=torch.float64, device=dev)
        fl = torch.as_tensor(s["flags"], device=dev)
        pos = t(s["pos"])
        self.s = {k: z() for k in ("u", "v", "sxx", "sxy", "syy", "szz", "eps", "epsd", "fcx", "fcy", "ftx", "fty",
                                   "ptx", "pty", "vtx", "vty", "rt", "txx", "txy", "tyy", "tzz", "Tt")}
        self.s.update(x=pos[:, 0].clone(), y=pos[:, 1].clone(), rho=t(s["rho"]), h=t(s["h"]), T=t(s["T"]),
                      tool=(fl & 4) != 0, fixed=(fl & 1) != 0, id=torch.arange(N, device=dev))
        if vel is not None:
            self.s["u"], self.s["v"] = t(vel)[:, 0].clone(), t(vel)[:, 1].clone()
        self.nx, self.ny = z(), z()
        self.tl = s["tool"]
        self.G = cfg.E / (2.0 * (1.0 + cfg.nu))
        self.K = 2.0 * self.G * (1 + cfg.nu) / (3 * (1 - 2 * cfg.nu))
        self.c0 = math.sqrt(self.K / cfg.rho0)
        self.mass = i.mass
        self.a_wp = cfg.k_wp / (cfg.rho0 * cfg.cp)
        rc = cfg.rho_tool * cfg.cp_tool
        self.a_tool = cfg.k_tool / rc if rc > 0 else 0.0
        dx = math.sqrt(i.mass / cfg.rho0)
        q = 1.0 / cfg.hdx
        self.wdp = PI_FAC / (cfg.hdx * dx) ** 2 * (1 - 1.5 * q * q * (1 - 0.5 * q))
        self.hastool = len(self.tl["left"]) > 0
        self.speed = float(self.tl["vel"][0]) if self.hastool else 0.0
        self.tol = cfg.secant_tol if cfg.secant_tol > 0 else 1e-6
        self.F = []

    def move_tool(self):
        t, d = self.tl, self.i.dt * self.tl["vel"]
        t["left"], t["right"] = t["left"] + d, t["right"] + d
        t["fillet"][:2] += d
        for k, (l, r) in enumerate(zip(t["left"], t["right"])):
            det = l[0] - r[0]
            t["vertical"][k] = abs(det) < 1e-12
            t["line_a"][k] = 0.0 if abs(det) < 1e-12 else (l[1] - r[1]) / det
            t["line_b"][k] = l[0] if abs(det) < 1e-12 else (r[1] * l[0] - r[0] * l[1]) / det

    def contact(self, x, y):
        t, n = self.tl, len(self.tl["left"])
        fx, fy, fr, f1, f2 = t["fillet"]
        inside = torch.ones_like(x, dtype=torch.bool)
        for k in range(n):
            inside &= ((t["left"][k][0] - x) * t["n"][k][0] + (t["left"][k][1] - y) * t["n"][k][1]) < 0
        if n == 5:
            inside |= torch.hypot(fx - x, fy - y) < fr
        depth = torch.full_like(x, BIG)
        cx, cy, nx, ny = (torch.zeros_like(x) for _ in range(4))
        for k in range(n):
            if t["vertical"][k]:
                dd = t["left"][k][0] - x
                new = (dd.abs(), torch.full_like(x, t["left"][k][0]), y, torch.sign(dd), torch.zeros_like(x))
            elif n == 5 and k == 2:
                vx, vy = x - fx, y - fy
                r = torch.hypot(vx, vy)
                ax, ay = vx / r, vy / r
                qx, qy = fx + fr * ax, fy + fr * ay
                a = torch.atan2(fy - qy, fx - qx)
                a = torch.where(a > 0, a, a + 2 * math.pi)
                ok = (a > min(f1, f2)) & (a < max(f1, f2))
                new = (torch.where(ok, torch.hypot(qx - x, qy - y), torch.full_like(x, BIG)), qx, qy, ax, ay)
            else:
                a, b = t["line_a"][k], t["line_b"][k]
                px = (x + a * y - a * b) / (a * a + 1)
                py = (a * (x + a * y) + b) / (a * a + 1)
                new = (torch.hypot(px - x, py - y), px, py, torch.full_like(x, -t["n"][k][0]),
                       torch.full_like(x, -t["n"][k][1]))
            near = new[0] < depth
            depth, cx, cy, nx, ny = (torch.where(near, p, q) for p, q in zip(new, (depth, cx, cy, nx, ny)))
        return inside, cx, cy, nx, ny

    def flow(self, e, ed, tc):
        c = self.c
        r = ed / c.jc_eps_dot_ref
        tb = torch.where(r > 1, 1 + c.jc_C * torch.log(r.clamp(min=1.0)), (1 + r) ** c.jc_C)
        return (c.jc_A + c.jc_B * e ** c.jc_n) * tb * tc

    def step(self):
        c, i, s, dt = self.c, self.i, self.s, self.i.dt
        gny, gnx, mass = i.grid_ny, i.grid_nx, self.mass
        cell = (((s["x"] - i.bbmin_x) / i.cell_size).long() * gny + ((s["y"] - i.bbmin_y) / i.cell_size).long())
        cell = cell.clamp(0, i.num_cell - 1)
        order = torch.argsort(cell, stable=True)
        for k in s:
            s[k] = s[k][order]
        cell = cell[order]
        off = torch.searchsorted(cell, torch.arange(i.num_cell + 1, device=self.dev))
        # predictor
        g = lambda a, b: s[a] + 0.5 * dt * s[b]
        x, y, u, v = g("x", "ptx"), g("y", "pty"), g("u", "vtx"), g("v", "vty")
        sxx, sxy, syy, szz = g("sxx", "txx"), g("sxy", "txy"), g("syy", "tyy"), g("szz", "tzz")
        rho, T = g("rho", "rt"), g("T", "Tt")
        tool, h = s["tool"], s["h"]
        p = torch.where(tool, torch.zeros_like(rho), self.c0 ** 2 * (rho - c.rho0))
        r2i = 1.0 / rho ** 2
        a, b = (sxx - syy), 2 * sxy
        d = torch.hypot(a, b)
        cc = torch.where(d > 0, a / d.clamp(min=1e-300), torch.ones_like(d))
        sn = torch.where(d > 0, b / d.clamp(min=1e-300), torch.zeros_like(d))
        mid = 0.5 * (sxx + syy) - p
        q1 = -c.stress_eps * (mid + 0.5 * d).clamp(min=0) * r2i
        q2 = -c.stress_eps * (mid - 0.5 * d).clamp(min=0) * r2i
        R = (0.5 * (1 + cc) * q1 + 0.5 * (1 - cc) * q2, 0.5 * sn * (q1 - q2),
             0.5 * (1 - cc) * q1 + 0.5 * (1 + cc) * q2)
        A = ((sxx - p) * r2i, sxy * r2i, (syy - p) * r2i)
        cs, vol = torch.sqrt(self.K / rho), mass / rho
        # candidates of the 5 x 5 cell windows, then the pairs in support
        gi, gj = cell // gny, cell % gny
        lo, hi = (gj - 2).clamp(min=0), (gj + 3).clamp(max=gny)
        I, J = [], []
        me = torch.arange(self.N, device=self.dev)
        for q in range(-2, 3):
            col = gi + q
            ok = (col >= 0) & (col < gnx)
            col = col.clamp(0, gnx - 1)
            b0, b1 = off[col * gny + lo], off[col * gny + hi]
            n = torch.where(ok, b1 - b0, torch.zeros_like(b0))
            ii = torch.repeat_interleave(me, n)
            st = torch.cumsum(n, 0) - n
            I.append(ii)
            J.append(torch.arange(ii.numel(), device=self.dev) - st[ii] + b0[ii])
        I, J = torch.cat(I), torch.cat(J)
        dx, dy = x[I] - x[J], y[I] - y[J]
        rr = dx * dx + dy * dy
        add = lambda idx, val: torch.zeros(self.N, dtype=torch.float64, device=self.dev).index_add_(0, idx, val)
        pse = c.thermal_solver == pymfc.THERMAL_PSE
        tp = None
        if pse and self.a_wp != 0:
            h2 = h[I] ** 2
            tp = add(I, (T[J] - T[I]) * (4.0 / (h2 * h2 * math.pi)) * torch.exp(-rr / h2) * mass / rho[J])
        keep = (rr < 4 * h[I] ** 2) & (rr >= 1e-8)
        if pse:
            keep &= ~tool[I]
        I, J, dx, dy, rr = I[keep], J[keep], dx[keep], dy[keep], rr[keep]
        h1 = 1.0 / h[I]
        rad = torch.sqrt(rr)
        q = rad * h1
        far = q > 1
        m = 2 - q
        fac = PI_FAC * h1 * h1
        w = torch.where(far, 0.25 * m ** 6, 1 - 1.5 * q * q * (1 - 0.5 * q)) * fac
        der = torch.where(far, -0.75 * m * m, -3.0 * q * (1 - 0.75 * q)) * h1 / rad * fac
        tl = add(I, 2.0 * vol[J] * (T[I] - T[J]) * der)
        mm = ~tool[I] & ~tool[J]
        I, J, dx, dy, rr, w, der = I[mm], J[mm], dx[mm], dy[mm], rr[mm], w[mm], der[mm]
        wx, wy = der * dx, der * dy
        du, dv = u[J] - u[I], v[J] - v[I]
        vd = [add(I, t * vol[J]) for t in (du * wx, du * wy, dv * wx, dv * wy)]
        fab = (w / self.wdp) ** 4
        S3 = [A[k][I] + A[k][J] + fab * (R[k][I] + R[k][J]) for k in range(3)]
        rij = 0.5 * (rho[I] + rho[J])
        vx = -(du * dx + dv * dy)
        hij = 0.5 * (h[I] + h[J])
        mu = torch.where(vx < 0, hij * vx / (rr + c.av_eta ** 2 * hij * hij), torch.zeros_like(vx))
        pi = (-c.av_alpha * 0.5 * (cs[I] + cs[J]) * mu + c.av_beta * mu * mu) / rij
        ax = add(I, mass * (S3[0] * wx + S3[1] * wy - pi * wx))
        ay = add(I, mass * (S3[1] * wx + S3[2] * wy - pi * wy))
        xs0, xs1 = add(I, c.xsph_eps * w * mass / rij * du), add(I, c.xsph_eps * w * mass / rij * dv)
        # update
        run = ~tool if pse else torch.ones_like(tool)
        pick = lambda cond, new, old: torch.where(cond, new, old)
        ptx, pty = pick(run, xs0, s["ptx"]), pick(run, xs1, s["pty"])
        zero = torch.zeros_like(x)
        vtx, vty = pick(run, zero, s["vtx"]), pick(run, zero, s["vty"])
        Tt = s["Tt"]
        if pse:
            Tt = torch.where(tool, self.a_tool, self.a_wp) * tp if tp is not None else Tt
        else:
            al = torch.where(tool, zero + self.a_tool, zero + self.a_wp)
            Tt = pick(al != 0, al * tl, Tt)
        exy, om, tr = 0.5 * (vd[1] + vd[2]), 0.5 * (vd[2] - vd[1]), vd[0] + vd[3]
        wt = -om
        jau = (2 * self.G * (vd[0] - tr / 3) + 2 * wt * sxy, 2 * self.G * exy + om * sxx + wt * syy,
               2 * self.G * (vd[3] - tr / 3) + 2 * om * sxy, -2 * self.G * tr / 3)
        wp = ~tool
        txx, txy, tyy, tzz = (pick(wp, n, s[o]) for n, o in zip(jau, ("txx", "txy", "tyy", "tzz")))
        rt = pick(wp, -rho * tr, s["rt"])
        vtx = pick(wp, vtx + ax + (s["fcx"] + s["ftx"]) / mass, vtx)
        vty = pick(wp, vty + ay + (s["fcy"] + s["fty"]) / mass, vty)
        ptx, pty = pick(wp, ptx + u, ptx), pick(wp, pty + v, pty)
        x, y, u, v = s["x"] + dt * ptx, s["y"] + dt * pty, s["u"] + dt * vtx, s["v"] + dt * vty
        sxx, sxy, syy, szz = s["sxx"] + dt * txx, s["sxy"] + dt * txy, s["syy"] + dt * tyy, s["szz"] + dt * tzz
        rho, T = s["rho"] + dt * rt, s["T"] + dt * Tt
        if c.eta != 0 and self.hastool:
            f = torch.hypot(s["ftx"], s["fty"])
            dvx, dvy = u - self.speed, v
            dvn = dvx * self.nx + dvy * self.ny
            T = T + torch.where(wp & (f != 0), c.eta * dt * f * torch.hypot(dvx - dvn, dvy - dvn) / (c.cp * mass), zero)
        eps, epsd = s["eps"], s["epsd"]
        if not c.elastic:
            norm = torch.sqrt(sxx ** 2 + syy ** 2 + szz ** 2 + sxy ** 2)
            a, b, d = sxx - p, syy - p, szz - p
            svm = torch.sqrt(((a * a + b * b + d * d) - a * b - a * d - b * d + 3 * sxy * sxy).clamp(min=0))
            tc = 1 - ((T - c.jc_Tref) / (c.jc_Tmelt - c.jc_Tref)).clamp(min=0) ** c.jc_m
            need = wp & (svm >= self.flow(eps, epsd, tc))
            s23 = math.sqrt(2.0 / 3.0)
            if bool(need.any()):
                k = torch.nonzero(need)[:, 0]
                e0, nk, tk = eps[k], norm[k], tc[k]
                dl = (epsd[k] * dt * s23).clamp(min=1e-8)
                live = torch.ones_like(k, dtype=torch.bool)

                def res(z):
                    zz = s23 * z.clamp(min=0)
                    return nk - 2 * self.G * z - s23 * self.flow(e0 + zz, zz / dt, tk)

                for _ in range(102):
                    g0, g1 = res(dl), res(1.01 * dl)
                    new = dl - g0 / ((g0 - g1) / (dl - 1.01 * dl))
                    new = torch.where(new < 0, -0.1 * new, new)
                    moved = (new - dl).abs() >= self.tol
                    dl = torch.where(live, new, dl)
                    live = live & moved
                    if not bool(live.any()):
                        break
                inc = s23 * dl.clamp(min=0)
                scale = 1 - dl * 2 * self.G / nk
                sxx, sxy, syy, szz = (t.index_put((k,), t[k] * scale) for t in (sxx, sxy, syy, szz))
                T = T.index_put((k,), T[k] + c.tq / (c.cp * rho[k]) * inc * self.flow(e0 + inc, inc / dt, tk))
                eps = eps.index_put((k,), e0 + inc)
            epsd_new = zero.clone()
            if bool(need.any()):
                epsd_new[k] = inc / dt
            epsd = pick(wp, epsd_new, epsd)
        x = pick(tool, x + dt * self.speed, x)
        fcx, fcy, ftx, fty = s["fcx"], s["fcy"], s["ftx"], s["fty"]
        if self.hastool:
            self.move_tool()
            ins, cx, cy, nx, ny = self.contact(x, y)
            gn = (x - cx) * nx + (y - cy) * ny
            ax, ay = -mass * gn * nx / dt ** 2 * c.contact_alpha, -mass * gn * ny / dt ** 2 * c.contact_alpha
            rx, ry = u - self.speed, v
            km = c.contact_alpha * mass / dt
            bx, by = ftx - km * (rx - rx * nx), fty - km * (ry - ry * ny)
            sl, fy = torch.hypot(bx, by), c.mu * torch.hypot(ax, ay)
            lim = torch.where(sl > fy, fy / sl.clamp(min=1e-300), torch.ones_like(sl)) if c.mu != 0 else zero
            pin = lambda new, old: torch.where(tool, old, torch.where(ins, new, zero))
            fcx, fcy, ftx, fty = pin(ax, fcx), pin(ay, fcy), pin(bx * lim, ftx), pin(by * lim, fty)
            self.nx, self.ny = pin(nx, self.nx), pin(ny, self.ny)
        fx = wp & s["fixed"]
        u, v, fcx, fcy, ptx, pty, vtx, vty = (torch.where(fx, zero, t) for t in (u, v, fcx, fcy, ptx, pty, vtx, vty))
        if self.a_tool != 0:
            T = torch.where(s["fixed"], zero + c.T_init, T)
        s.update(x=x, y=y, u=u, v=v, sxx=sxx, sxy=sxy, syy=syy, szz=szz, rho=rho, T=T, eps=eps, epsd=epsd, fcx=fcx,
                 fcy=fcy, ftx=ftx, fty=fty, ptx=ptx, pty=pty, vtx=vtx, vty=vty, rt=rt, txx=txx, txy=txy, tyy=tyy,
                 tzz=tzz, Tt=Tt)
        self.F.append(torch.stack([fcx.sum() + ftx.sum(), fcy.sum() + fty.sum()]))

    def forces(self):
        return torch.stack(self.F).cpu().numpy()

    def field(self, f):
        s = self.s
        if f == "pos":
            return torch.stack([s["x"], s["y"]], 1).cpu().numpy()
        if f == "vel":
            return torch.stack([s["u"], s["v"]], 1).cpu().numpy()
        if f == "S":
            return torch.stack([s["sxx"], s["sxy"], s["syy"], s["szz"]], 1).cpu().numpy()
        return s[{"T": "T", "eps_pl": "eps"}[f]].cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    cfgs = _configs(case, seed)
    if kind == "batch" and case["n"] * case["steps"] > 1000:
        return None  # a python loop over the instances' steps: more than 20 seconds
    runs = []
    for c in cfgs:
        e = _Exact(c, _ring_velocities(c, seed) if kind == "rings" else None)
        for _ in range(case["steps"]):
            e.step()
        runs.append(e)
    e = runs[0]
    if kind == "report":
        return {"F": e.forces()[-1], "vel": e.field("vel"), "T": e.field("T")}
    if kind == "batch":
        out = {"F": np.stack([r.forces() for r in runs])}
        for f in ("pos", "vel", "S"):
            out[f] = np.concatenate([r.field(f) for r in runs])
        return out
    if kind == "vjp":  # the gradient of the converged return has no plain counterpart here
        return {"F": e.forces()[case["steps"] // 2:].mean(0), "grad": None, "pos": e.field("pos"),
                "vel": e.field("vel")}
    out = {f: (None if f == "id" else e.field(f)) for f in DUMP}
    if kind != "rings":
        out["F"] = e.forces()
    return out
