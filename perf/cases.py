"""The work a user has this framework do, as measured cases.

A case is one call sequence of a user's program on data it already holds:

kind "run"        resident members advance by `steps` large steps as captured
                  graphs and their fields come back to the host: one history
                  interval (about a simulated minute) of a simulation
                  (`nimbus_hip_step`, then `nimbus_hip_member_download` of
                  every member).
kind "transport"  the conservative WENO5 transport contract, on host arrays as
                  the adapter calls it, or on device arrays as a caller that
                  cannot allocate does.
kind "acoustic"   the batched acoustic substep contract on host arrays.

The states are storms in progress, not resting air: updrafts of up to 18 m/s,
saturated cloud, rain shafts and cold pools over a few per cent of the domain,
on the analytic sounding with seeded theta noise.

`exact` evaluates the same equations in plain torch in 64 bits. Two parts of
the scheme are defined in 32 bits whatever the storage and are taken so there
too: the radiating boundary velocity and the limiter ratio.
"""
import ctypes
import math

import numpy as np
import torch

from nimbus_amd import lib as L
from nimbus_amd import workloads as W

SIDES = {"open": L.BC_RADIATIVE, "periodic": L.BC_PERIODIC, "walls": L.BC_RIGID_SLIP, "gradient": L.BC_ZERO_GRADIENT}


def _run(name, nx, ny, nz, dx, dz, dt, substeps, steps, fp64=False, hevi=True, sides="open", sgs="2d", coriolis=0.0,
         diffusion=0.0, members=1):
    c = {"kind": "run", "nx": nx, "ny": ny, "nz": nz, "dx": dx, "dz": dz, "dt": dt, "substeps": substeps,
         "steps": steps, "fp64": fp64, "hevi": hevi, "sides": sides, "sgs": sgs, "coriolis": coriolis,
         "diffusion": diffusion, "members": members}
    return dict(c, name=name) if name else c


def _transport(name, nx, ny, nz, device, supplied):
    c = {"kind": "transport", "nx": nx, "ny": ny, "nz": nz, "dx": 500.0, "dz": 250.0, "dt": 3.0, "device": device,
         "supplied": supplied}
    return dict(c, name=name) if name else c


def _acoustic(name, nx, ny, nz, substeps, hevi, sides):
    c = {"kind": "acoustic", "nx": nx, "ny": ny, "nz": nz, "dx": 500.0, "dz": 250.0, "dt": 3.0, "substeps": substeps,
         "hevi": hevi, "sides": sides}
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest serving request: launches and latency
        _run("48x48x40 mixed", 48, 48, 40, 1000.0, 500.0, 3.0, 6, 20),
        # the plain all-FP64 explicit method on the smallest named grid
        _run("64x64x40 fp64 explicit", 64, 64, 40, 1000.0, 500.0, 3.0, 6, 20, fp64=True, hevi=False),
        # the named 500 m storm
        _run("160x160x80 mixed", 160, 160, 80, 500.0, 250.0, 3.0, 6, 20),
        # the headline domain: three storms at 250 m
        _run("400x400x100 mixed", 400, 400, 100, 250.0, 200.0, 1.5, 8, 40),
        # the plain reference method in mixed precision on a mid-size domain
        _run("192x192x60 mixed explicit", 192, 192, 60, 500.0, 1000.0 / 3.0, 1.5, 6, 40, hevi=False),
        # the largest serving grid in FP64 with the vertically implicit method (accuracy reruns)
        _run("256x256x80 fp64", 256, 256, 80, 500.0, 250.0, 1.5, 6, 40, fp64=True),
        # ragged sizes with the options on: f-plane, periodic sides, 3-D closure, explicit
        # diffusion, an odd substep count
        _run("147x93x57 mixed options", 147, 93, 57, 700.0, 350.0, 2.1, 7, 30, sides="periodic", sgs="3d",
             coriolis=1.0e-4, diffusion=50.0),
        # more than 129 levels
        _run("100x120x140 mixed deep", 100, 120, 140, 500.0, 150.0, 0.9, 6, 40, sides="walls"),
        # the uneven ensemble as one batch (six of its members)
        _run("ensemble of 6 mixed", 0, 0, 0, 0.0, 0.0, 0.0, 6, 20, members=6),
        # the adapter's transport call: host arrays both ways
        _transport("transport, host arrays", 160, 160, 80, False, True),
        # the same contract where the caller's arrays are on the device
        _transport("transport, device arrays", 128, 128, 60, True, False),
        # the adapter's acoustic call: one large step's substeps, host arrays both ways
        _acoustic("acoustic, host arrays", 128, 128, 60, 6, True, "open"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "run", "transport", "acoustic"])
    if kind == "transport":
        device = rng.random() < 0.5
        n = _log(rng, 32, 130 if device else 230)
        m = max(16, min(250, int(n * rng.uniform(0.7, 1.3))))
        nz = min(rng.randint(24, 100), (1 << 20) // (n * m)) if device else rng.randint(24, 100)
        return _transport(None, n, m, nz, device, rng.random() < 0.5)
    if kind == "acoustic":
        n = _log(rng, 32, 200)
        return _acoustic(None, n, max(16, min(250, int(n * rng.uniform(0.7, 1.3)))), rng.randint(24, 100),
                         rng.randint(5, 8), rng.random() < 0.6, rng.choice(list(SIDES)))
    n = _log(rng, 40, 320)
    m = max(32, min(400, int(n * rng.uniform(0.7, 1.3))))
    nz = rng.randint(36, 140) if n * m < 25000 else rng.randint(36, 100)
    dz = round(20000.0 / nz, 1)
    dx = round(rng.uniform(250.0, 1000.0), 1)
    fp64 = rng.random() < 0.25 and n * m * nz < 4_000_000
    return _run(None, n, m, nz, dx, dz, round(W.long_run_dt(dx, dz), 2), rng.randint(5, 8), rng.randint(8, 20), fp64,
                rng.random() < 0.7, rng.choice(list(SIDES)), rng.choice(["2d", "2d", "3d", "off"]),
                rng.choice([0.0, 1.0e-4]), rng.choice([0.0, 0.0, 50.0]))


# ---------------------------------------------------------------- inputs

def _members(case):
    """The grids and settings of the case's members: one, or those of the uneven ensemble."""
    if case.get("members", 1) == 1:
        return [dict(case, sounding={})]
    return [dict(case, nx=w.nx, ny=w.ny, nz=w.nz, dx=w.dx, dz=w.dz, dt=w.dt, sounding=w.sounding)
            for w in W.ensemble_c3()[:case["members"]]]


def _grid(m):
    return L.make_grid(m["nx"], m["ny"], m["nz"], m["dx"], m["dx"], m["dz"])


def _base(m):
    return L.base_state(_grid(m), L.default_sounding(**m.get("sounding", {})))


def _qvs(T, p):
    Tc = T.clamp(150.0, 400.0) - 273.15
    es = (611.21 * torch.exp((18.678 - Tc / 234.5) * Tc / (257.14 + Tc))).clamp(min=0.0)
    pp = p.clamp(100.0, 200000.0)
    return (0.62198 * es / (pp - es).clamp(min=1.0)).clamp(0.0, 0.2)


def _storms(m, base, seed, fp64):
    """A storm state on the device, fields (nx, ny, nz) in the storage type."""
    nx, ny, nz = m["nx"], m["ny"], m["nz"]
    gen = torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + 17)

    def rnd(*s):
        return torch.rand(*s, generator=gen, device="cuda", dtype=torch.float64)

    prof = {k: torch.from_numpy(v).cuda() for k, v in base.items()}
    x = (torch.arange(nx, device="cuda", dtype=torch.float64) * m["dx"]).view(-1, 1, 1)
    y = (torch.arange(ny, device="cuda", dtype=torch.float64) * m["dx"]).view(1, -1, 1)
    z = ((torch.arange(nz, device="cuda", dtype=torch.float64) + 0.5) * m["dz"]).view(1, 1, -1)
    core = torch.zeros(nx, ny, nz, device="cuda", dtype=torch.float64)
    rain, pool = torch.zeros_like(core), torch.zeros_like(core)
    n = 1 + (nx * m["dx"] > 60000.0) + (nx * m["dx"] > 90000.0)
    radius = min(5000.0, 0.12 * min(nx, ny) * m["dx"])
    for q in range(n):
        a, b, c = (0.8 + 0.4 * rnd(3)).tolist()
        cx = nx * m["dx"] * ((q + 0.5) / n + 0.04 * (a - 1.0))
        cy = ny * m["dx"] * (0.5 + 0.1 * (b - 1.0))
        r2 = ((x - cx) ** 2 + (y - cy) ** 2) / (radius * c) ** 2
        s2 = ((x - cx - 0.6 * radius) ** 2 + (y - cy) ** 2) / (radius * c) ** 2
        core += torch.exp(-r2) * torch.sin(math.pi * (z / 14000.0).clamp(0.0, 1.0))
        rain += torch.exp(-1.5 * s2) * (1.0 - z / 8000.0).clamp(0.0, 1.0)
        pool += torch.exp(-0.7 * s2) * (1.0 - z / 1500.0).clamp(0.0, 1.0)
    core, rain, pool = core.clamp(max=1.0), rain.clamp(max=1.0), pool.clamp(max=1.0)
    cloud = ((core - 0.25) / 0.75).clamp(min=0.0) * (z > 1000.0)
    p = prof["p0"].expand(nx, ny, nz).clone()
    theta = prof["theta0"] + 3.0 * core - 3.0 * pool + 0.2 * (rnd(nx, ny, nz) - 0.5)
    T = theta * (p / 100000.0) ** (287.0 / 1004.0)
    qs = _qvs(T, p)
    qv = torch.where(cloud > 0.0, qs * (1.0 + 0.02 * cloud), torch.minimum(prof["qv0"] * (1.0 + 0.2 * core), qs))
    st = {"u": prof["u0"] + 4.0 * core * (rnd(nx, ny, 1) - 0.5), "v": prof["v0"] + 4.0 * core * (rnd(nx, ny, 1) - 0.5),
          "w": 18.0 * core * (1.0 - 0.4 * rain), "rho": p / (287.0 * T), "p": p, "theta": theta, "qv": qv,
          "qc": 2.5e-3 * cloud, "qr": 5.0e-3 * ((rain - 0.05) / 0.95).clamp(min=0.0)}
    st["w"][:, :, -1] = 0.0
    return {k: v.expand(nx, ny, nz).to(torch.float64 if fp64 else torch.float32).contiguous() for k, v in st.items()}


def _config(m):
    sgs = None if m["sgs"] == "off" else dict(L.sgs_preset(), mode=L.SGS_3D if m["sgs"] == "3d" else L.SGS_HORIZONTAL)
    return L.step_config(m["dt"], m["substeps"], L.ACOUSTIC_HEVI if m["hevi"] else L.ACOUSTIC_EXPLICIT,
                         coriolis_f=m["coriolis"], lateral=SIDES[m["sides"]], sponge=L.sponge_preset(m["dx"]), sgs=sgs,
                         diffusion={"kh": m["diffusion"], "kv": 0.2 * m["diffusion"]} if m["diffusion"] else None)


def _seed(seed, k):
    return int(seed) + 7919 * k


def _transport_inputs(case, seed):
    """Begin density, winds or retained fluxes and end density, and the four scalars, float32 on the device."""
    base = _base(case)
    st = _storms(case, base, seed, False)
    out = {k: st[k] for k in ("rho", "u", "v", "w")}
    if case["supplied"]:
        r = st["rho"].double()

        def face(v, d):
            return (0.5 * (r + torch.roll(r, -1, d)) * v.double()).float()

        out.update(mfx=face(st["u"], 0), mfy=face(st["v"], 1), mfz=face(st["w"], 2))
        out["mfz"][:, :, -1] = 0.0
        div = ((out["mfx"].double() - torch.roll(out["mfx"], 1, 0).double()) / case["dx"] +
               (out["mfy"].double() - torch.roll(out["mfy"], 1, 1).double()) / case["dx"] +
               (out["mfz"].double() - torch.roll(out["mfz"], 1, 2).double()) / case["dz"])
        out["rho_end"] = (r - case["dt"] * div).clamp(0.5 * r.min(), 2.0).float()
    return out, [st[k] for k in ("theta", "qv", "qc", "qr")]


# ---------------------------------------------------------------- prepare and run

def prepare(case, seed):
    state = {"kind": case["kind"], "ctx": L.Context(0)}
    ctx = state["ctx"]
    if case["kind"] == "run":
        ctx.set_graphs(True)
        state["steps"] = case["steps"]
        state["members"] = []
        for k, m in enumerate(_members(case)):
            base = _base(m)
            st = {n: v.cpu().numpy() for n, v in _storms(m, base, _seed(seed, k), case["fp64"]).items()}
            member = ctx.member(_grid(m), _config(m), base, L.PRECISION_FP64 if case["fp64"] else L.PRECISION_MIXED)
            member.upload(dict(st, rain_mm=None))
            state["members"].append(member)
        return state
    if case["kind"] == "acoustic":
        base = _base(case)
        st = _storms(case, base, seed, False)
        state["case"] = case
        state["base"] = base
        state["in"] = {k: st[k].cpu().numpy() for k in ("u", "v", "w", "rho", "p", "theta")}
        return state
    fields, scalars = _transport_inputs(case, seed)
    if case["device"]:
        # the caller's own device arrays, in and out
        state["keep"] = (fields, scalars)
        state["out"] = [torch.empty_like(q) for q in scalars]

        def ptr(t):
            return ctypes.cast(t.data_ptr(), ctypes.POINTER(ctypes.c_float))
        call = ctx.lib.nimbus_hip_advect_scalars_conservative_noalloc
    else:
        fields, scalars = {k: v.cpu().numpy() for k, v in fields.items()}, [q.cpu().numpy() for q in scalars]
        state["keep"] = (fields, scalars)
        state["out"] = [np.empty_like(q) for q in scalars]
        ptr = L.fptr
        call = ctx.lib.nimbus_hip_dispatch_advect_scalars_conservative_cartesian_cgrid
    null = ctypes.POINTER(ctypes.c_float)()
    at = {k: ptr(v) for k, v in fields.items()}
    n, sup = len(scalars), case["supplied"]
    pf = ctypes.POINTER(ctypes.c_float)
    qin, qout = (pf * n)(*[ptr(q) for q in scalars]), (pf * n)(*[ptr(q) for q in state["out"]])
    kappa, pd = (ctypes.c_float * n)(), (ctypes.c_int * n)(0, 1, 1, 1)
    inv, iz = 1.0 / case["dx"], 1.0 / case["dz"]
    state["d"] = L.ConservativeTransportDispatch(
        at["u"], at["v"], at["w"], at["rho_end"] if sup else at["rho"], qin, qout, kappa, pd, n, case["nx"],
        case["ny"], case["nz"], inv, inv, iz, inv * inv, inv * inv, iz * iz, case["dt"], 0.05,
        at["rho"] if sup else null, at.get("mfx", null), at.get("mfy", null), at.get("mfz", null), int(sup), 0.0, 0.0,
        1, 0)
    state["arrays"] = (at, qin, qout, kappa, pd)
    state["call"] = call
    return state


def run(state):
    ctx = state["ctx"]
    if state["kind"] == "run":
        ctx.step(state["members"], state["steps"])
        return [m.download() for m in state["members"]]
    if state["kind"] == "transport":
        L.check(state["call"](ctx.handle, ctypes.byref(state["d"])), "transport")
        return state["out"]
    case, base = state["case"], state["base"]
    a = {k: v.copy() for k, v in state["in"].items()}  # the contract updates its arrays in place
    mf = [np.zeros_like(a["u"]) for _ in range(3)]
    side = SIDES[case["sides"]]
    d = L.AcousticBatchedDispatch(
        *[L.fptr(a[k]) for k in ("u", "v", "w", "rho", "p", "theta")], L.dptr(base["rho0"]), L.dptr(base["p0"]),
        case["nx"], case["ny"], case["nz"], case["dx"], case["dx"], case["dz"], case["dt"] / case["substeps"],
        case["substeps"], L.ACOUSTIC_HEVI if case["hevi"] else L.ACOUSTIC_EXPLICIT, 0.1, side, side, side, side,
        L.BOTTOM_FREE_SLIP, L.TOP_RIGID, *[L.fptr(x) for x in mf], 1, 1.0 / case["substeps"])
    L.check(ctx.lib.nimbus_hip_dispatch_acoustic_substeps_batched(ctx.handle, ctypes.byref(d)), "acoustic")
    return {"u": a["u"], "v": a["v"], "w": a["w"], "rho": a["rho"], "p": a["p"], "mfx": mf[0], "mfy": mf[1],
            "mfz": mf[2]}


def work(case):
    """Bytes: the 9 fields of a large step's stages, each read and written once per stage that the stencils
    force apart (68 + 17 per acoustic substep, in storage elements per cell), the closure's 2 x 7 and the
    diffusion's 11 where they are on, and the download. Flops: counted from the formulas per cell."""
    if case["kind"] == "run":
        e = 8 if case["fp64"] else 4
        b = f = 0.0
        for m in _members(case):
            cells = float(m["nx"] * m["ny"] * m["nz"])
            nsub = _substeps(m, _base(m))
            n_sgs = 0 if m["sgs"] == "off" else math.ceil(m["dt"] / 1.0 - 1e-9)
            per = 68 + 17 * nsub + 14 * n_sgs + (11 if m["diffusion"] else 0)
            b += cells * e * (case["steps"] * per + 9)
            f += cells * case["steps"] * (2 * 160 + nsub * (130 if m["hevi"] else 70) + 1100 + 80 + 200 * n_sgs +
                                          (200 if m["diffusion"] else 0))
        return {"bytes": b, "flops": f}
    cells = float(case["nx"] * case["ny"] * case["nz"])
    if case["kind"] == "transport":
        return {"bytes": cells * 4 * ((5 if case["supplied"] else 4) + 8), "flops": cells * 1300}
    return {"bytes": cells * 4 * (9 + 8), "flops": cells * case["substeps"] * (130 if case["hevi"] else 70)}


# ---------------------------------------------------------------- the same equations in 64 bits

G0, RD, RV, CP, LV, P00 = 9.81, 287.0, 461.5, 1004.0, 2.5e6, 1.0e5
GAMMA, KAPPA = CP / (CP - RD), RD / CP
X, Y, Z = 2, 1, 0  # axes of the (k, j, i) arrays below


def _substeps(m, base):
    c = float(np.sqrt(GAMMA * base["p0"] / base["rho0"]).max())
    d = m["dx"] if m["hevi"] else min(m["dx"], m["dz"])
    return max(m["substeps"], int(math.ceil(m["dt"] * c / (0.5 * d))) + 1, 2)


def _at(f, axis, idx):
    return f.index_select(axis, idx)


def _sh(f, axis, o):
    """f at offset o along an axis, clamped to the domain."""
    n = f.shape[axis]
    return f.index_select(axis, (torch.arange(n, device=f.device) + o).clamp(0, n - 1))


def _pos(f, axis):
    shape = [1, 1, 1]
    shape[axis] = -1
    return torch.arange(f.shape[axis], device=f.device).view(shape)


def _col(v):
    return v.view(-1, 1, 1)


def _eos(rho, theta):
    return P00 * (rho * RD * theta / P00) ** GAMMA


def _upwind(f, axis, a, inv):
    n = f.shape[axis]
    pos = _pos(f, axis)
    half = torch.minimum(pos, n - 1 - pos)
    m3, m2, m1, p1, p2, p3 = (_sh(f, axis, o) for o in (-3, -2, -1, 1, 2, 3))
    up = a >= 0
    d5 = torch.where(up, -2 * m3 + 15 * m2 - 60 * m1 + 20 * f + 30 * p1 - 3 * p2,
                     2 * p3 - 15 * p2 + 60 * p1 - 20 * f - 30 * m1 + 3 * m2) * (inv / 60.0)
    d3 = torch.where(up, 2 * p1 + 3 * f - 6 * m1 + m2, -p2 + 6 * p1 - 3 * f - 2 * m1) * (inv / 6.0)
    d1 = torch.where(up, f - m1, p1 - f) * inv
    return torch.where(half >= 3, d5, torch.where(half == 2, d3, torch.where(half == 1, d1, torch.zeros_like(f))))


class _Model:
    """One member in 64 bits: fields (k, j, i), rho and p as perturbations of the base state."""

    def __init__(self, m, base, config=None):
        self.m = m
        self.b = {k: _col(torch.from_numpy(np.asarray(v)).double().cuda()) for k, v in base.items()}
        self.dx, self.dz = m["dx"], m["dz"]
        self.nx, self.ny, self.nz = m["nx"], m["ny"], m["nz"]
        side = SIDES[m.get("sides", "open")]
        self.side, self.wrap = side, side == L.BC_PERIODIC

    def load(self, st):
        s = {k: v.double().permute(2, 1, 0).contiguous() for k, v in st.items()}
        s["rho"] = s["rho"] - self.b["rho0"]
        s["p"] = s["p"] - self.b["p0"]
        self.s = s
        self.rain = torch.zeros(self.ny, self.nx, device="cuda", dtype=torch.float64)
        f = s["u"]
        k, j, i = _pos(f, Z), _pos(f, Y), _pos(f, X)
        self.k, self.j, self.i = k, j, i
        self.inner = (i >= 1) & (i <= self.nx - 2) & (j >= 1) & (j <= self.ny - 2)
        self.below_lid = k <= self.nz - 2

    def host(self, v):
        return v.permute(2, 1, 0)

    # -- slow tendencies
    def slow(self, u, v, w):
        s, h = self.s, 0.25
        inv, iz, f = 1.0 / self.dx, 1.0 / self.dz, self.m["coriolis"]
        g0 = self.k == 0
        zero = torch.zeros_like(u)
        vx, wx, wy, uy = _sh(v, X, 1), _sh(w, X, 1), _sh(w, Y, 1), _sh(u, Y, 1)
        vy = h * (_sh(v, Y, -1) + v + _sh(vx, Y, -1) + vx)
        wz = torch.where(g0, h * (w + wx), h * (_sh(w, Z, -1) + w + _sh(wx, Z, -1) + wx))
        dz_ = torch.where(g0, torch.where(wz >= 0, zero, (_sh(u, Z, 1) - u) * iz), _upwind(u, Z, wz, iz))
        du = -u * _upwind(u, X, u, inv) - vy * _upwind(u, Y, vy, inv) - wz * dz_ + f * (vy - self.b["v0"])
        ux = h * (_sh(u, X, -1) + u + _sh(uy, X, -1) + uy)
        wz = torch.where(g0, h * (w + wy), h * (_sh(w, Z, -1) + w + _sh(wy, Z, -1) + wy))
        dz_ = torch.where(g0, torch.where(wz >= 0, zero, (_sh(v, Z, 1) - v) * iz), _upwind(v, Z, wz, iz))
        dv = -ux * _upwind(v, X, ux, inv) - v * _upwind(v, Y, v, inv) - wz * dz_ - f * (ux - self.b["u0"])
        uz, vz = _sh(u, Z, 1), _sh(v, Z, 1)
        ux = h * (_sh(u, X, -1) + u + _sh(uz, X, -1) + uz)
        vy = h * (_sh(v, Y, -1) + v + _sh(vz, Y, -1) + vz)
        dz_ = torch.where(g0, torch.where(w >= 0, w * iz, (_sh(w, Z, 1) - w) * iz), _upwind(w, Z, w, iz))
        dw = -ux * _upwind(w, X, ux, inv) - vy * _upwind(w, Y, vy, inv) - w * dz_
        rp, r0 = s["rho"], self.b["rho0"]
        qv0 = self.b["qv0"].float().double()
        rpf = 0.5 * (rp + _sh(rp, Z, 1))
        rf = 0.5 * (r0 + _sh(r0, Z, 1)) + rpf
        load = s["qc"] + s["qr"]
        dw = (dw - G0 * rpf / rf + G0 * 0.608 * (0.5 * (s["qv"] + _sh(s["qv"], Z, 1)) - 0.5 * (qv0 + _sh(qv0, Z, 1))) -
              G0 * 0.5 * (load + _sh(load, Z, 1)))
        on = self.inner & self.below_lid
        return [torch.where(on, d, zero) for d in (du, dv, dw)]

    def slow_rk2(self):
        s, dt = self.s, self.m["dt"]
        old = [s[n] for n in "uvw"]
        k1 = self.slow(*old)
        k2 = self.slow(*[a + dt * b for a, b in zip(old, k1)])
        for n, a, p, q in zip("uvw", old, k1, k2):
            s[n] = a + dt * 0.5 * (p + q)

    # -- boundary closure
    def seed(self):
        s = self.s
        self.stash = {"w": s["u"][:, :, 0].float(), "e": s["u"][:, :, self.nx - 2].float(),
                      "s": s["v"][:, 0, :].float(), "n": s["v"][:, self.ny - 2, :].float()}

    def _pair(self, axis, n, t, lo, hi, dts):
        s, size, bc = self.s, self.s["u"].shape[axis], self.side
        others = t + ["w", "rho", "p"]

        def get(f, c):
            return s[f].select(axis, c).clone()

        inn, a = {f: get(f, 1) for f in [n] + others}, {f: get(f, size - 2) for f in [n] + others}
        am = get(n, size - 3)

        def put(f, c, v):
            s[f].select(axis, c).copy_(v)

        if bc == L.BC_PERIODIC:
            for f in [n] + others:
                put(f, 0, a[f])
                put(f, size - 1, inn[f])
            return
        if bc == L.BC_RADIATIVE and dts > 0:
            h, inv = torch.tensor(dts, device="cuda").float(), torch.tensor(1.0, device="cuda") / torch.tensor(
                self.dx, device="cuda").float()
            p = self.stash[lo]
            ph = p - 30.0
            self.stash[lo] = torch.where(ph >= 0, p, p - ((h * ph) * (inn[n].float() - p)) * inv)
            put(n, 0, self.stash[lo].double())
            p = self.stash[hi]
            ph = p + 30.0
            self.stash[hi] = torch.where(ph <= 0, p, p - ((h * ph) * (p - am.float())) * inv)
            put(n, size - 2, self.stash[hi].double())
            put(n, size - 1, self.stash[hi].double())
        elif bc == L.BC_RADIATIVE:
            put(n, size - 1, a[n])
        elif bc == L.BC_ZERO_GRADIENT:
            put(n, 0, inn[n])
            put(n, size - 2, am)
            put(n, size - 1, am)
        else:
            for c in (0, size - 2, size - 1):
                put(n, c, torch.zeros_like(am))
        for f in others:
            put(f, 0, inn[f])
            put(f, size - 1, a[f])

    def close(self, dts=0.0):
        s = self.s
        for f in ("u", "v", "w", "rho", "p"):
            s[f] = s[f].clone()
        self._pair(X, "u", ["v"], "w", "e", dts)
        self._pair(Y, "v", ["u"], "s", "n", dts)
        s["w"][-1] = 0.0
        s["u"][-1] = s["u"][-2]
        s["v"][-1] = s["v"][-2]

    # -- acoustic substep
    def substep(self, dts, weight, hevi, first):
        s, b, nz = self.s, self.b, self.nz
        inv, iz = 1.0 / self.dx, 1.0 / self.dz
        u, v, w, th = s["u"], s["v"], s["w"], s["theta"]
        r0 = b["rho0"]
        rc = r0 + s["rho"]
        zero = torch.zeros_like(u)
        fx = torch.where(self.i < self.nx - 1, 0.5 * (rc + _sh(rc, X, 1)) * u, zero)
        fy = torch.where(self.j < self.ny - 1, 0.5 * (rc + _sh(rc, Y, 1)) * v, zero)
        rb = torch.where(self.below_lid, 0.5 * (rc + _sh(rc, Z, 1)), zero)
        if first:
            self.mf = [zero, zero, zero]
            self.rho_begin = s["rho"]
        div = (fx - _sh(fx, X, -1)) * inv + (fy - _sh(fy, Y, -1)) * inv
        if hevi:
            al, a1 = 0.55, 0.45
            rstar = torch.where(self.inner, rc - dts * div, rc)
            ps = _eos(rstar, th)
            C = GAMMA * ps / rstar
            fo = rb * w
            e = -a1 * dts * iz * (fo - torch.where(self.k > 0, _sh(fo, Z, -1), zero))
            Bc = al * dts * iz
            up = lambda f: f[1:]  # noqa: E731
            lo = lambda f: f[:-1]  # noqa: E731
            rbr = lo(rb)
            Ak = Bc / rbr
            Aa = -Ak * Bc * lo(C) * torch.cat([torch.zeros_like(rb[:1]), rbr[:-1]])
            U = -Ak * Bc * up(C) * up(rb)
            D = 1.0 + Ak * Bc * (up(C) + lo(C)) * rbr
            psp = ps - b["p0"]
            G = (al * (up(psp) - lo(psp)) + a1 * (up(s["p"]) - lo(s["p"]))) * iz
            R = lo(w) - dts / rbr * G - Ak * (up(C) * up(e) - lo(C) * lo(e))
            c_, d_ = [], []
            for r in range(nz - 1):
                piv = D[r] - (Aa[r] * c_[-1] if r else 0.0)
                c_.append(U[r] / piv)
                d_.append((R[r] - (Aa[r] * d_[-1] if r else 0.0)) / piv)
            x = [None] * (nz - 1)
            for r in range(nz - 2, -1, -1):
                x[r] = d_[r] - (c_[r] * x[r + 1] if r < nz - 2 else 0.0)
            x.append(torch.zeros_like(x[0]))
            wn = torch.where(self.inner & self.below_lid, torch.stack(x).clamp(-120.0, 120.0), w)
            F = torch.where(self.inner, rb * (al * wn + a1 * w), zero)
            rn = torch.where(self.inner, rstar - dts * iz * (F - torch.where(self.k > 0, _sh(F, Z, -1), zero)), rc)
            fz, s["w"] = F, wn
        else:
            fz = torch.where(self.below_lid, rb * w, zero)
            ft = torch.where(self.below_lid, fz, rc * w)
            div = div + (ft - torch.where(self.k > 0, _sh(fz, Z, -1), zero)) * iz
            rn = torch.where(self.inner, rc - dts * div, rc)
        self.mf = [a + weight * f for a, f in zip(self.mf, (fx, fy, fz))]
        rn = rn.clamp(0.05, 2.0)
        p = _eos(rn, th).clamp(1000.0, 200000.0) - b["p0"]
        on = self.inner & self.below_lid
        s["rho"], s["p"] = rn - r0, p
        du = -(_sh(p, X, 1) - p) * inv / (0.5 * (rn + _sh(rn, X, 1)))
        dv = -(_sh(p, Y, 1) - p) * inv / (0.5 * (rn + _sh(rn, Y, 1)))
        s["u"] = (u + dts * torch.where(on, du, zero)).clamp(-180.0, 180.0)
        s["v"] = (v + dts * torch.where(on, dv, zero)).clamp(-180.0, 180.0)
        dw = zero if hevi else torch.where(on, -(_sh(p, Z, 1) - p) * iz / (0.5 * (rn + _sh(rn, Z, 1))), zero)
        s["w"] = (s["w"] + dts * dw).clamp(-120.0, 120.0)

    def acoustic(self, n, dts, weight, hevi):
        self.seed()
        for q in range(n):
            self.substep(dts, weight, hevi, q == 0)
            self.close(dts)

    # -- transport
    @staticmethod
    def _face(q, axis, m):
        n = q.shape[axis]
        pos = _pos(q, axis)
        up = m >= 0
        v = [_sh(q, axis, o) for o in (-2, -1, 0, 1, 2, 3)]
        a, b, c, d, e = (torch.where(up, v[x], v[5 - x]) for x in range(5))
        fits = torch.where(up, (pos >= 2) & (pos + 2 <= n - 1), (pos >= 1) & (pos + 3 <= n - 1))
        has_mc = torch.where(up, pos >= 1, pos + 1 <= n - 2)
        q0 = a / 3 - 7 * b / 6 + 11 * c / 6
        q1 = -b / 6 + 5 * c / 6 + d / 3
        q2 = c / 3 + 5 * d / 6 - e / 6
        s0 = 13 / 12 * (a - 2 * b + c) ** 2 + 0.25 * (a - 4 * b + 3 * c) ** 2
        s1 = 13 / 12 * (b - 2 * c + d) ** 2 + 0.25 * (b - d) ** 2
        s2 = 13 / 12 * (c - 2 * d + e) ** 2 + 0.25 * (3 * c - 4 * d + e) ** 2
        m2 = torch.stack([t.abs() for t in (a, b, c, d, e)]).amax(0) ** 2
        eps = 1.0e-6 * m2 + 1.0e-40
        w0, w1, w2 = 0.1 / (eps + s0) ** 2, 0.6 / (eps + s1) ** 2, 0.3 / (eps + s2) ** 2
        ws = w0 + w1 + w2
        weno = (w0 * q0 + w1 * q1 + w2 * q2) / ws
        weno = torch.where(torch.isfinite(weno) & (ws > 0), weno, c)
        r, l = d - c, c - b
        x = torch.minimum((0.5 * (r + l)).abs(), 2 * torch.minimum(r.abs(), l.abs()))
        slope = torch.where((r > 0) & (l > 0), x, torch.where((r < 0) & (l < 0), -x, torch.zeros_like(x)))
        return m * torch.where(fits, weno, c + 0.5 * torch.where(has_mc, slope, torch.zeros_like(slope)))

    def transport(self, q, mf, rho_b, rho_e, dt, pd):
        inv = {X: 1.0 / self.dx, Y: 1.0 / self.dx, Z: 1.0 / self.dz}
        zero = torch.zeros_like(q)
        last = {X: self.nx - 1, Y: self.ny - 1, Z: self.nz - 1}
        hi = {a: torch.where(_pos(q, a) < last[a], self._face(q, a, m), zero) for a, m in zip((X, Y, Z), mf)}
        lo = {a: torch.where(_pos(q, a) > 0, _sh(f, a, -1), zero) for a, f in hi.items()}
        if pd:
            out = sum((hi[a].clamp(min=0.0) - lo[a].clamp(max=0.0)) * inv[a] for a in hi)
            r = torch.where(out > 0, (rho_b * q.clamp(min=0.0) / dt / out).clamp(max=1.0), torch.ones_like(q))
            small = torch.nextafter(r.float() * (1.0 - 32.0 * 2.0 ** -23), torch.zeros_like(r, dtype=torch.float32))
            r = torch.where((r > 0) & (r < 1), small, r.float()).double()
            hi = {a: f * torch.where(f > 0, r, _sh(r, a, 1)) for a, f in hi.items()}
            lo = {a: torch.where(_pos(q, a) > 0, _sh(f, a, -1), zero) for a, f in hi.items()}
        div = sum((hi[a] - lo[a]) * inv[a] for a in hi)
        return torch.where(self.inner, (rho_b * q - dt * div) / rho_e.clamp(min=0.05), q)

    # -- microphysics
    @staticmethod
    def _slope(T, qs, p):
        e = qs * p / (0.62198 + qs)
        Tc = T - 273.15
        den, num = 257.14 + Tc, (18.678 - Tc / 234.5) * Tc
        d = ((18.678 - 2 * Tc / 234.5) * den - num) / (den * den)
        ok = (T > 150) & (T < 400) & (qs > 0) & (qs < 0.2)
        return torch.where(ok, qs * p / (p - e).clamp(min=1.0) * d, torch.zeros_like(T))

    def _adjust(self, T, p, qv, qc):
        lv = LV / CP
        T = T.clamp(150.0, 400.0)
        qs = _qvs(T, p)
        most = torch.where(qv > qs, torch.minimum(qv, ((400.0 - T) / lv).clamp(min=0.0)),
                           torch.minimum(qc, ((T - 150.0) / lv).clamp(min=0.0)))
        sign = torch.where(qv > qs, 1.0, -1.0)  # condensing or evaporating by c >= 0
        f_end = sign * (qv - sign * most - _qvs(T + lv * sign * most, p))
        lo, hi = torch.zeros_like(T), most.clone()
        c = torch.minimum((sign * (qv - qs) / (1.0 + lv * self._slope(T, qs, p))).clamp(min=0.0), hi)
        for _ in range(40):
            Ta = T + lv * sign * c
            qa = _qvs(Ta, p)
            f = sign * (qv - sign * c - qa)
            lo, hi = torch.where(f > 0, c, lo), torch.where(f > 0, hi, c)
            n = c + f / (1.0 + lv * self._slope(Ta, qa, p))
            c = torch.where((n > lo) & (n < hi), n, torch.where(f == 0, c, 0.5 * (lo + hi)))
        c = torch.where(f_end <= 0, c, most)
        c = torch.where((qv > qs) | ((qv < qs) & (qc > 0)), c, torch.zeros_like(c)) * sign
        return T + lv * c, (qv - c).clamp(min=0.0), (qc + c).clamp(min=0.0)

    def kessler(self):
        s, b, dt, dz = self.s, self.b, self.m["dt"], self.dz
        p, rho = b["p0"] + s["p"], b["rho0"] + s["rho"]
        th, qv, qc, qr = s["theta"], s["qv"].clamp(min=0.0), s["qc"].clamp(min=0.0), s["qr"]
        pp = p.clamp(100.0, 200000.0)
        T0 = th.clamp(150.0, 700.0) * (pp / P00) ** KAPPA
        T, qvs_, qcs = self._adjust(T0, pp, qv, qc)
        rate = (qcs - s["qc"]) / dt
        zero = torch.zeros_like(th)
        dqc, dqv, dT, dqr = rate, -rate, LV / CP * rate, zero
        qr0 = qr.clamp(min=0.0)
        factor = 1.0 / (1.0 + 2.2 * dt * qr0 ** 0.875)
        prod = torch.minimum((qcs * (1 - factor) + factor * 1.0e-3 * dt * (qcs - 1.0e-3).clamp(min=0.0)).clamp(min=0.0),
                             qcs) / dt
        prod = torch.where(qcs > 0, prod, zero)
        dqc, dqr = dqc - prod, dqr + prod
        qsat = _qvs(T, pp)
        av = qr + prod * dt
        rcgs = 1.0e-3 * rho
        rc = rcgs * av.clamp(min=0.0)
        vent = (1.6 + 124.9 * rc ** 0.2046) * rc ** 0.525
        raw = vent / (2.55e8 / (p * qsat) + 5.4e5) * ((qsat - qvs_) / (rcgs * qsat))
        bound = (qsat - qvs_) / (1.0 + LV * LV * qsat / (CP * RV * (T * T).clamp(min=1.0)))
        ev = torch.minimum(raw.clamp(min=0.0), torch.minimum(bound, av) / dt)
        ev = torch.where(((qr > 0) | (prod > 0)) & (qsat > 0) & (qvs_ < qsat), ev, zero)
        dqv, dqr, dT = dqv + ev, dqr - ev, dT - LV / CP * ev
        V = torch.where(qr0 < 1.0e-9, zero, 36.34 * (1.0e-3 * rho * qr0) ** 0.1346) * (1.2 / rho).sqrt()
        fall = V.clamp(max=20.0) * qr0
        dqr = dqr - fall / dz + torch.where(self.below_lid, _sh(rho, Z, 1) / rho * _sh(fall, Z, 1) / dz, zero)
        self.rain += torch.where(self.inner[0], fall[0] * rho[0] * dt, torch.zeros_like(fall[0]))
        dth = dT * (P00 / pp) ** KAPPA
        new = {"theta": (th + (dth * dt).clamp(-50.0, 50.0)).clamp(200.0, 700.0)}
        for n, d in (("qv", dqv), ("qc", dqc), ("qr", dqr)):
            new[n] = (s[n] + d * dt).clamp(0.0, 0.05)
        for n, v in new.items():
            s[n] = torch.where(self.inner, v, s[n])

    def project(self):
        s = self.s
        s["p"] = _eos(self.b["rho0"] + s["rho"], s["theta"]).clamp(1000.0, 200000.0) - self.b["p0"]

    # -- closure and diffusion
    def _near(self, axis):
        n = self.s["u"].shape[axis]
        a = torch.arange(n, device="cuda")
        if self.wrap:
            return (torch.where(a <= 1, torch.full_like(a, n - 2), (a - 1).clamp(max=n - 2)),
                    torch.where(a >= n - 2, torch.ones_like(a), (a + 1).clamp(min=1)))
        return (a - 1).clamp(min=0), (a + 1).clamp(max=n - 1)

    def closure(self, h, mode3):
        s = self.s
        u, v, w = s["u"], s["v"], s["w"]
        ip, im = self._near(X)[1], self._near(X)[0]
        jp, jm = self._near(Y)[1], self._near(Y)[0]
        E, Wd = (lambda f: _at(f, X, ip)), (lambda f: _at(f, X, im))
        N, Sd = (lambda f: _at(f, Y, jp)), (lambda f: _at(f, Y, jm))
        T, B = (lambda f: _sh(f, Z, 1)), (lambda f: torch.where(self.k > 0, _sh(f, Z, -1), torch.zeros_like(f)))
        inv, iz = 1.0 / self.dx, 1.0 / self.dz
        zero = torch.zeros_like(u)
        s12 = 0.5 * ((N(u) - u) * inv + (E(v) - v) * inv)
        face = self.below_lid
        xb, yb = torch.where(face, (E(w) - w) * inv, zero), torch.where(face, (N(w) - w) * inv, zero)

        def four(f, side):
            return 0.25 * (side(f) + f)

        q12 = s12 * s12
        S12 = 0.25 * (q12 + Wd(q12) + Sd(q12) + Sd(Wd(q12)))
        S11, S22 = (u - Wd(u)) * inv, (v - Sd(v)) * inv
        if mode3:
            S33 = (w - B(w)) * iz
            xa, ya = torch.where(face, (T(u) - u) * iz, zero), torch.where(face, (T(v) - v) * iz, zero)
            q13, q23 = (0.5 * (xa + xb)) ** 2, (0.5 * (ya + yb)) ** 2
            S13 = 0.25 * (q13 + Wd(q13) + B(q13) + B(Wd(q13)))
            S23 = 0.25 * (q23 + Sd(q23) + B(q23) + B(Sd(q23)))
            strain = 2 * (S11 ** 2 + S22 ** 2 + S33 ** 2) + 4 * (S12 + S13 + S23)
        else:
            q13, q23 = xb * xb, yb * yb
            strain = (2 * (S11 ** 2 + S22 ** 2) + 4 * S12 + 0.25 * (q13 + Wd(q13) + B(q13) + B(Wd(q13))) +
                      0.25 * (q23 + Sd(q23) + B(q23) + B(Sd(q23))))
        delta = (self.dx * self.dx * self.dz) ** (1.0 / 3.0)
        nu = ((0.18 * delta) ** 2 * strain.sqrt()).clamp(max=1000.0)
        K = (3.0 * nu).clamp(max=1000.0)
        R = self.b["rho0"] + s["rho"]
        M = R * nu
        on = self.inner & self.below_lid
        edge = 2 if self.wrap else 3
        on_u, on_v = on & (self.i <= self.nx - edge), on & (self.j <= self.ny - edge)
        # u
        corner = 0.25 * (M + E(M) + N(M) + N(E(M))) * ((N(u) - u) * inv + (E(v) - v) * inv)
        t13 = 0.5 * (0.5 * (M + E(M)) + 0.5 * (T(M) + T(E(M)))) * ((E(w) - w) * inv + ((T(u) - u) * iz if mode3 else 0.0))
        t23 = 0.5 * (0.5 * (M + N(M)) + 0.5 * (T(M) + T(N(M)))) * ((N(w) - w) * inv + ((T(v) - v) * iz if mode3 else 0.0))
        n11, n22 = 2 * M * (u - Wd(u)) * inv, 2 * M * (v - Sd(v)) * inv
        du = (E(n11) - n11) * inv + (corner - Sd(corner)) * inv
        dv = (N(n22) - n22) * inv + (corner - Wd(corner)) * inv
        fw = (t13 - Wd(t13)) * inv + (t23 - Sd(t23)) * inv
        if mode3:
            du, dv = du + (t13 - B(t13)) * iz, dv + (t23 - B(t23)) * iz
            n33 = 2 * M * (w - B(w)) * iz
            fw = fw + (T(n33) - n33) * iz
        du, dv, dw = du / (0.5 * (R + E(R))), dv / (0.5 * (R + N(R))), fw / (0.5 * (R + T(R)))
        # theta, qv: a closed side has no flux
        open_ = self.side in (L.BC_RADIATIVE, L.BC_ZERO_GRADIENT)
        TK = R * K
        new = {}
        for n, lo, hi in (("theta", 200.0, 700.0), ("qv", 0.0, 0.05)):
            f = s[n]
            fe, fn = 0.5 * (TK + E(TK)) * (E(f) - f) * inv, 0.5 * (TK + N(TK)) * (N(f) - f) * inv
            fw_, fs = 0.5 * (TK + Wd(TK)) * (f - Wd(f)) * inv, 0.5 * (TK + Sd(TK)) * (f - Sd(f)) * inv
            if not open_ and not self.wrap:
                fe = torch.where(self.i == self.nx - 2, zero, fe)
                fw_ = torch.where(self.i == 1, zero, fw_)
                fn = torch.where(self.j == self.ny - 2, zero, fn)
                fs = torch.where(self.j == 1, zero, fs)
            d = (fe - fw_) * inv + (fn - fs) * inv
            if mode3:
                ft = torch.where(self.below_lid, 0.5 * (TK + T(TK)) * (T(f) - f) * iz, zero)
                d = d + (ft - B(ft)) * iz
            new[n] = (f + h * torch.where(self.inner, d / R, zero)).clamp(lo, hi)
        for n, d, m, c in (("u", du, on_u, 180.0), ("v", dv, on_v, 180.0), ("w", dw, on, 120.0)):
            new[n] = (s[n] + h * torch.where(m, d, zero)).clamp(-c, c)
        s.update(new)

    def diffuse(self, kh, kv):
        s, dt, nz = self.s, self.m["dt"], self.nz
        rho = self.b["rho0"] + s["rho"]
        inv2, dz = 1.0 / (self.dx * self.dx), self.dz
        zero = torch.zeros_like(rho)
        new = {}
        for n, loc in (("u", 1), ("v", 2), ("w", 3), ("theta", 0), ("qv", 0)):
            f = s[n]
            last = {X: self.nx - 2, Y: self.ny - 2}
            if loc in (1, 2) and not self.wrap:
                last[X if loc == 1 else Y] -= 1
            k1 = nz if loc == 0 else nz - 1

            def step(g, axis, o):
                size = g.shape[axis]
                a = torch.arange(size, device="cuda")
                t = a + o
                if self.wrap:
                    t = torch.where((a == 1) & (o < 0), torch.full_like(a, size - 2), t)
                    t = torch.where((a == size - 2) & (o > 0), torch.ones_like(a), t)
                return _at(g, axis, t.clamp(0, size - 1))

            cv = {0: lambda: rho, 1: lambda: 0.5 * (rho + step(rho, X, 1)), 2: lambda: 0.5 * (rho + step(rho, Y, 1)),
                  3: lambda: 0.5 * (rho + _sh(rho, Z, 1))}[loc]()
            if loc == 3:
                down = torch.where(self.k > 0, rho * kv * (f - _sh(f, Z, -1)) / dz, zero)
                up = torch.where(self.k < k1 - 1, _sh(rho, Z, 1) * kv * (_sh(f, Z, 1) - f) / dz, zero)
            else:
                up = torch.where(self.k < k1 - 1, 0.5 * (cv + _sh(cv, Z, 1)) * kv * (_sh(f, Z, 1) - f) / dz, zero)
                down = torch.where(self.k > 0, 0.5 * (cv + _sh(cv, Z, -1)) * kv * (f - _sh(f, Z, -1)) / dz, zero)
            t = (up - down) / (cv * dz)
            for axis in (X, Y):
                hi = 0.5 * (cv + step(cv, axis, 1)) * (step(f, axis, 1) - f)
                lo = 0.5 * (cv + step(cv, axis, -1)) * (f - step(f, axis, -1))
                if not self.wrap:
                    hi = torch.where(_pos(f, axis) >= last[axis], zero, hi)
                    lo = torch.where(_pos(f, axis) <= 1, zero, lo)
                t = t + kh * (hi - lo) * inv2 / cv
            on = ((self.i >= 1) & (self.i <= last[X]) & (self.j >= 1) & (self.j <= last[Y]) & (self.k < k1))
            c = {"u": 180.0, "v": 180.0, "w": 120.0}.get(n)
            v = f + dt * torch.where(on, t, zero)
            new[n] = v.clamp(-c, c) if c else v.clamp(*((200.0, 700.0) if n == "theta" else (0.0, 0.05)))
        s.update(new)

    # -- sponges
    def sponge(self):
        s, b, dt, nz = self.s, self.b, self.m["dt"], self.nz
        k = torch.arange(nz, device="cuda", dtype=torch.float64)

        def factor(alpha):
            return -torch.expm1(-alpha * dt)

        depth = nz * self.dz - 12000.0

        def alpha(z):
            if depth <= 0.0:
                return torch.zeros_like(z)
            return 0.05 * torch.sin(0.5 * math.pi * ((z - 12000.0) / depth).clamp(0.0, 1.0)) ** 2

        fu, fw = _col(factor(alpha((k + 0.5) * self.dz))), _col(factor(alpha((k + 1.0) * self.dz)))
        n = min(8, nz)
        d = (nz - 1) - k
        fwo = _col(factor(torch.where(d < n, 0.2 * torch.sin(0.5 * math.pi * (1.0 - d / (n - 1)).clamp(min=0.0)) ** 2,
                                      torch.zeros_like(d))))
        width = max(0, min(int(round(10000.0 / self.dx)), max(self.nx, self.ny)))
        dist = torch.minimum(torch.minimum(self.i, self.nx - 1 - self.i), torch.minimum(self.j, self.ny - 1 - self.j))
        fl = torch.where(dist < width, factor(0.05 * torch.sin(0.5 * math.pi * (1.0 - dist.double() / width)) ** 2),
                         torch.zeros_like(dist, dtype=torch.float64)) if width else 0.0
        for name, target, facs in (("u", b["u0"], (fu, fl)), ("v", b["v0"], (fu, fl)), ("w", 0.0, (fw, fwo, fl)),
                                   ("theta", b["theta0"], (fu, fl))):
            for f in facs:
                s[name] = s[name] + f * (target - s[name])

    def step(self):
        m, s = self.m, self.s
        self.slow_rk2()
        self.close()
        n = _substeps(m, {q: v.flatten().cpu().numpy() for q, v in self.b.items()})
        self.acoustic(n, m["dt"] / n, 1.0 / n, m["hevi"])
        rb, re = self.b["rho0"] + self.rho_begin, self.b["rho0"] + s["rho"]
        for name in ("theta", "qv", "qc", "qr"):
            s[name] = self.transport(s[name], self.mf, rb, re, m["dt"], name != "theta")
        self.kessler()
        done = 0.0
        while m["sgs"] != "off" and m["dt"] - done > 1.0e-12:
            h = min(m["dt"] - done, 1.0)
            self.closure(h, m["sgs"] == "3d")
            done += h
        if m["diffusion"]:
            self.diffuse(m["diffusion"], 0.2 * m["diffusion"])
        self.project()
        self.sponge()
        self.close()


def _exact_run(case, seed):
    out = []
    for k, m in enumerate(_members(case)):
        base = _base(m)
        model = _Model(m, base)
        model.load(_storms(m, base, _seed(seed, k), case["fp64"]))
        for _ in range(case["steps"]):
            model.step()
        s = dict(model.s, rho=model.s["rho"] + model.b["rho0"], p=model.s["p"] + model.b["p0"])
        out.append({**{n: model.host(s[n]) for n in L.FIELDS}, "rain_mm": model.rain.t()})
        del model, s
    return out


def exact(case, seed):
    if case["kind"] == "run":
        return _exact_run(case, seed)
    base = _base(case)
    model = _Model(case, base)
    if case["kind"] == "acoustic":
        st = _storms(case, base, seed, False)
        model.load({k: st[k] for k in ("u", "v", "w", "rho", "p", "theta")})
        n = case["substeps"]
        model.acoustic(n, case["dt"] / n, 1.0 / n, case["hevi"])
        s = model.s
        out = {"u": s["u"], "v": s["v"], "w": s["w"], "rho": s["rho"] + model.b["rho0"], "p": s["p"] + model.b["p0"],
               "mfx": model.mf[0], "mfy": model.mf[1], "mfz": model.mf[2]}
        return {k: model.host(v) for k, v in out.items()}
    fields, scalars = _transport_inputs(case, seed)
    f = {k: v.double().permute(2, 1, 0).contiguous() for k, v in fields.items()}
    model.load({k: fields[k] for k in ("u", "rho")} | {"p": fields["rho"]})
    if case["supplied"]:
        mf, rb, re = [f["mfx"], f["mfy"], f["mfz"]], f["rho"], f["rho_end"]
    else:
        rb = f["rho"]
        zero = torch.zeros_like(rb)
        mf = [torch.where(_pos(rb, a) < rb.shape[a] - 1, 0.5 * (rb + _sh(rb, a, 1)) * f[n], zero)
              for a, n in ((X, "u"), (Y, "v"), (Z, "w"))]
        re = rb - case["dt"] * sum((m - torch.where(_pos(rb, a) > 0, _sh(m, a, -1), zero)) / d
                                   for m, a, d in zip(mf, (X, Y, Z), (case["dx"], case["dx"], case["dz"])))
    return [model.host(model.transport(q.double().permute(2, 1, 0).contiguous(), mf, rb, re, case["dt"], n > 0))
            for n, q in enumerate(scalars)]
