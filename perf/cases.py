"""The work that users of this framework have it do, as cases of a measurement.

listed() names the cases, draw() gives others of the same ranges, prepare() makes what a program
holds before the call (inputs from a seed, the plan, its workspace), run() is one pass through the
public entry points, work() what a pass cannot do without, and exact() the same outputs from plain
torch in 64 bits (automatic differentiation through the scheme, none of this package's code).

Fields of a case: kind (see run), nx x ny interior cells, nstep time steps, shots, dtype "f32" or
"f64", kernel (PropagatorKernel of the acoustic scheme; 0 for elastic cases), npml, layout
("surface": sources and receivers on a line below the top edge; "well": both on vertical lines
inside the model), uneven (records and spreads of different lengths), gb (device memory for the
plan's workspace: the checkpoint schedule follows from it).
"""
import math

import numpy as np
import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

import __graft_entry__

ads = __graft_entry__.load_package()

DT = {"f32": torch.float32, "f64": torch.float64}


def _case(kind, nx, ny, nstep, shots, dtype, kernel=0, npml=20, layout="surface", uneven=False, gb=8.0):
    return {"kind": kind, "nx": int(nx), "ny": int(ny), "nstep": int(nstep), "shots": int(shots),
            "dtype": dtype, "kernel": int(kernel), "npml": int(npml), "layout": layout,
            "uneven": bool(uneven), "gb": float(gb)}


def listed():
    c = [
        # the reference's per-step custom op, called level by level from a user's own time loop:
        # the smallest call, where latency counts
        ("step_200x200_f64", _case("step", 200, 200, 1, 1, "f64", 1)),
        # the same op on a 1000 x 1000 grid with its gradient, as automatic differentiation calls it
        ("step_vjp_1000x1000_f64", _case("step_vjp", 1000, 1000, 1, 1, "f64", 1)),
        # the plain solver on one shot of a teaching-size model: full wavefield history, misfit,
        # gradient; the reference's own way to work (64 bits, its default propagator kernel)
        ("solver_200x200_f64", _case("solver", 200, 200, 1000, 1, "f64", 0)),
        # batched FWI gradient of a small shallow model with eight shots in 64 bits: the shipped
        # FWI example's sizes, many steps on a grid that does not fill the chip
        ("gradient_200x66_8_f64", _case("gradient", 200, 66, 1678, 8, "f64", 0, 12)),
        # velocity from a network: traces and their pullback through autograd, default kernel
        ("traces_400x800_24_f32", _case("traces", 400, 800, 500, 24, "f32", 0, 20, gb=24)),
        # the ordinary batched FWI gradient, with checkpoints
        ("gradient_1000x1000_32_f32", _case("gradient", 1000, 1000, 400, 32, "f32", 1, 40, gb=24)),
        # the largest: 64 shots of uneven record length and spread, checkpointed
        ("gradient_2000x2000_64_f32", _case("gradient", 2000, 2000, 240, 64, "f32", 1, 40, uneven=True, gb=60)),
        # cross-well survey on an odd grid: sources and receivers inside the model
        ("gradient_well_517x389_6_f32", _case("gradient", 517, 389, 700, 6, "f32", 1, 15, layout="well")),
        # modelling one observed record of a long, shallow section
        ("modelling_1501x401_1_f32", _case("modelling", 1501, 401, 1000, 1, "f32", 0, 20)),
        # batched elastic gradient for density and the Lame parameters
        ("elastic_600x600_16_f32", _case("elastic_gradient", 600, 600, 300, 16, "f32", 0, 30, gb=60)),
        # a small elastic survey in 64 bits
        ("elastic_134x97_4_f64", _case("elastic_gradient", 134, 97, 500, 4, "f64", 0, 12)),
        # the plain elastic solver on one shot: full histories, misfit, gradient
        ("elastic_solver_100x100_f64", _case("elastic_solver", 100, 100, 400, 1, "f64", 0, 12)),
    ]
    return [dict(v, name=k) for k, v in c]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "step_vjp", "solver", "gradient", "gradient", "gradient", "traces",
                       "modelling", "elastic_gradient", "elastic_gradient", "elastic_solver"])
    dtype = rng.choice(["f32", "f64"])
    kernel = rng.choice([0, 1])
    npml = rng.choice([8, 10, 12, 20, 30, 40])
    lo = 2 * npml + 20
    if kind in ("step", "step_vjp"):
        return _case(kind, _log(rng, 60, 1500), _log(rng, 60, 1500), 1, 1, dtype, 1, 12)
    if kind in ("solver", "elastic_solver"):
        npml = min(npml, 20)
        nx, ny = _log(rng, 60, 300), _log(rng, 60, 300)
        lim = 4e7 if kind == "solver" else 1.2e7
        n = max(60, min(rng.randint(200, 1200), int(lim / (nx * ny))))
        return _case(kind, nx, ny, n, 1, dtype, kernel if kind == "solver" else 0, npml)
    if kind == "elastic_gradient":
        nx, ny, shots = _log(rng, max(lo, 80), 700), _log(rng, max(lo, 80), 700), _log(rng, 1, 16)
        n = max(60, min(rng.randint(100, 800), int(1.5e9 / (nx * ny * shots))))
        return _case(kind, nx, ny, n, shots, dtype, 0, npml, gb=24)
    shots = 1 if kind == "modelling" else _log(rng, 1, 32)
    nx, ny = _log(rng, max(lo, 80), 1600), _log(rng, max(lo, 66), 1600)
    n = max(60, min(rng.randint(100, 1600), int(6e9 / (nx * ny * shots))))
    return _case(kind, nx, ny, n, shots, dtype, kernel, npml, rng.choice(["surface", "surface", "well"]),
                 rng.random() < 0.3, 24)


# ---------------------------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _spacing(case):
    """(h, dt): 10 m and 1 ms, or 5 m and 0.5 ms on the larger grids (CFL 0.64 at 4500 m/s)."""
    return (10.0, 1e-3) if case["nx"] < 900 else (5.0, 5e-4)


def _smooth(g, nx, ny, dev):
    """Smooth noise in [0, 1] on the padded grid."""
    a = torch.rand((1, 1, 9, 11), generator=g, dtype=torch.float64).to(dev)
    a = F.interpolate(a, size=(nx + 2, ny + 2), mode="bicubic", align_corners=True)[0, 0]
    return (a - a.min()) / (a.max() - a.min())


def _velocity(g, nx, ny, dev):
    """1500 .. 4500 m/s, growing with depth (the second axis), with smooth lateral changes."""
    d = torch.linspace(0.0, 1.0, ny + 2, dtype=torch.float64, device=dev)[None, :]
    return 1500.0 + 3000.0 * (0.45 * _smooth(g, nx, ny, dev) + 0.55 * d)


def _ricker(f, dt, n, dev, delay=1.2):
    t = torch.arange(n, dtype=torch.float64, device=dev) * dt
    a = (math.pi * f * (t - delay / f)) ** 2
    return (1.0 - 2.0 * a) * torch.exp(-a)


def _survey(case, seed):
    """Shots of a case: per shot a dict of si, sj, ri, rj (1-based, host), n (record length) and w
    (wavelet, device, 64 bits), and the generator that the model comes from."""
    dev = _device()
    g = torch.Generator().manual_seed(1000003 * int(seed) + 17)
    nx, ny, S, N, m = case["nx"], case["ny"], case["shots"], case["nstep"], case["npml"]
    h, dt = _spacing(case)
    elastic = case["kind"].startswith("elastic")
    shots = []
    for s in range(S):
        f = 8.0 + 4.0 * float(torch.rand((), generator=g))
        shift = float(torch.rand((), generator=g))
        n, nr = N, nx
        if case["uneven"]:
            n = max(2, int(N * (0.6 + 0.4 * float(torch.rand((), generator=g)))))
            nr = max(1, int(nx * (0.2 + 0.8 * float(torch.rand((), generator=g)))))
            if s == 0:
                n = N
        if case["layout"] == "well":
            ii = max(m + 2, nx // 4)
            jj = m + 3 + int((s + shift) * max(1, ny - 2 * m - 4) / S)
            rj = np.arange(m + 2, ny + 1 - m, dtype=np.int64)
            ri = np.full(len(rj), min(nx - m, 3 * nx // 4), np.int64)
        else:
            depth = m + 3 if elastic else 3
            ii = m + 2 + int((s + shift) * max(1, nx - 2 * m - 2) / S)
            jj = depth
            lo = min(max(2, ii - nr // 2), nx + 2 - nr)
            ri = np.arange(lo, lo + nr, dtype=np.int64)
            rj = np.full(nr, depth, np.int64)
        shots.append({"si": ii, "sj": jj, "ri": ri, "rj": rj, "n": n, "w": _ricker(f, dt, n, dev), "f": f})
    return shots, g, dev


def _observed(case, sh, scale):
    """A record (n + 1, receivers) of two arrivals with hyperbolic moveout."""
    h, dt = _spacing(case)
    dev = sh["w"].device
    x = torch.as_tensor(np.hypot(sh["ri"] - sh["si"], sh["rj"] - sh["sj"]) * h, device=dev)
    t = torch.arange(sh["n"] + 1, dtype=torch.float64, device=dev)[:, None] * dt
    out = 0.0
    for t0, v, a in ((0.02, 1700.0, 1.0), (0.25, 2400.0, 0.4)):
        arr = torch.sqrt(t0 * t0 + (x / v) ** 2)[None, :]
        q = (math.pi * sh["f"] * (t - arr - 1.2 / sh["f"])) ** 2
        out = out + a * (1.0 - 2.0 * q) * torch.exp(-q) / torch.sqrt(1.0 + x / (10.0 * h))[None, :]
    return scale * out


AMP = {False: 1e4, True: 1e6}      # wavelet peak, acoustic / elastic
OBS = {False: 5e-3, True: 5e-2}    # observed amplitudes of the size that these wavelets give


def _elastic_model(g, nx, ny, dev):
    vp = _velocity(g, nx, ny, dev) + 500.0
    vs = vp / 1.73
    rho = 310.0 * vp ** 0.25
    return rho, rho * (vp * vp - 2.0 * vs * vs), rho * vs * vs


def _fields(case, seed):
    """The per-step op's inputs: fields of a running simulation (smooth, of wave amplitude)."""
    dev = _device()
    g = torch.Generator().manual_seed(7919 * int(seed) + 5)
    nx, ny = case["nx"], case["ny"]
    h, dt = _spacing(case)
    c = _velocity(g, nx, ny, dev) ** 2
    k = torch.rand((12, 4), generator=g, dtype=torch.float64).tolist()
    x = torch.arange(nx + 2, dtype=torch.float64, device=dev)[:, None]
    y = torch.arange(ny + 2, dtype=torch.float64, device=dev)[None, :]
    wave = lambda r: 1e-2 * torch.sin(0.5 * r[0] * x + 0.4 * r[1] * y + 6.0 * r[2]) * (0.5 + r[3])
    w, wold, phi, psi = (sum(wave(k[3 * q + e]) for e in range(3)) for q in range(4))
    sx, ty = _acoustic_profiles(case)
    one = torch.ones((nx + 2, ny + 2), dtype=torch.float64, device=dev)
    s, t = one * sx.to(dev)[:, None], one * ty.to(dev)[None, :]
    ring = torch.zeros_like(one)
    ring[1:-1, 1:-1] = 1.0
    pml = ((s > 0) | (t > 0)).double() * ring
    f = [w * ring, wold * ring, 20.0 * phi * pml, 20.0 * psi * pml, s, t, c]
    cot = [wave(k[q]) * 100.0 for q in (0, 5, 9)]
    return [v.to(DT[case["dtype"]]) for v in f], [v.to(DT[case["dtype"]]) for v in cot]


def _params(case):
    h, dt = _spacing(case)
    if case["kind"].startswith("elastic"):
        return ads.ElasticPropagatorParams(NX=case["nx"], NY=case["ny"], NSTEP=case["nstep"], DELTAX=h,
                                           DELTAY=h, DELTAT=0.8 * dt, f0=12.0, vp_ref=4500.0,
                                           NPOINTS_PML=case["npml"])
    return ads.AcousticPropagatorParams(NX=case["nx"], NY=case["ny"], NSTEP=case["nstep"], DELTAX=h,
                                        DELTAY=h, DELTAT=dt, NPOINTS_PML=case["npml"], vp_ref=3000.0,
                                        PropagatorKernel=case["kernel"])


def prepare(case, seed):
    kind, dt = case["kind"], DT[case["dtype"]]
    p = _params(case)
    if kind in ("step", "step_vjp"):
        f, cot = _fields(case, seed)
        return {"case": case, "p": p, "f": f, "cot": cot}
    shots, g, dev = _survey(case, seed)
    el = kind.startswith("elastic")
    amp, obs = AMP[el], [_observed(case, sh, OBS[el]) for sh in shots]
    st = {"case": case, "p": p}
    if el:
        st["model"] = [m.to(dt) for m in _elastic_model(g, case["nx"], case["ny"], dev)]
        wl = [amp * torch.stack([sh["w"], sh["w"]], 1) for sh in shots]
        srcs = [ads.ElasticSource([sh["si"]] * 2, [sh["sj"]] * 2, [2, 3], w.to(dt)) for sh, w in zip(shots, wl)]
        rcvs = [ads.ElasticReceiver(np.concatenate([sh["ri"]] * 2), np.concatenate([sh["rj"]] * 2),
                                    np.repeat([0, 1], len(sh["ri"]))) for sh in shots]
        rec = [torch.cat([o, 0.7 * o], 1).T.contiguous().to(dt) for o in obs]
        if kind == "elastic_solver":
            st.update(src=srcs[0], rcv=rcvs[0], obs=rec[0])
            return st
        plan = ads.ElasticPlan(p, srcs, rcvs, dtype=dt)
    else:
        c = _velocity(g, case["nx"], case["ny"], dev)
        st["model"] = c.to(dt)
        srcs = [ads.AcousticSource([sh["si"]], [sh["sj"]], (amp * sh["w"])[:, None].to(dt)) for sh in shots]
        rcvs = [ads.AcousticReceiver(sh["ri"], sh["rj"]) for sh in shots]
        rec = [o.to(dt) for o in obs]
        if kind == "solver":
            st.update(src=srcs[0], rcv=rcvs[0], obs=rec[0])
            return st
        plan = ads.AcousticPlan(p, srcs, rcvs, dtype=dt, nstep=[sh["n"] for sh in shots])
    st["plan"], st["srcv"], st["obs"] = plan, plan.pack_srcv([s.srcv for s in srcs]), plan.pack_traces(rec)
    budget = int(case["gb"] * 1e9)
    st["K"] = plan.choose_interval(budget) if kind == "modelling" else plan.choose_schedule(budget)[0]
    plan.workspace(st["K"])
    return st


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------

def run(st):
    kind = st["case"]["kind"]
    if kind == "step":
        return ads.acoustic_one_step_customop(st["p"], *st["f"])
    if kind == "step_vjp":
        f = [x.detach().requires_grad_(q in (0, 1, 2, 3, 6)) for q, x in enumerate(st["f"])]
        out = ads.acoustic_one_step_customop(st["p"], *f)
        gr = torch.autograd.grad(out, [f[0], f[1], f[2], f[3], f[6]], st["cot"])
        return [o.detach() for o in out], list(gr)
    if kind == "solver":
        c = st["model"].detach().requires_grad_(True)
        ap = ads.AcousticPropagatorSolver(st["p"], st["src"], c)
        tr = ads.SimulatedObservation_(ap, st["rcv"])
        loss = torch.sum((tr - st["obs"]) ** 2)
        return {"traces": tr.detach(), "loss": loss.detach(), "grad": torch.autograd.grad(loss, c)[0]}
    if kind == "elastic_solver":
        m = [x.detach().requires_grad_(True) for x in st["model"]]
        ep = ads.ElasticPropagatorSolver(st["p"], st["src"], *m)
        tr = ads.SimulatedObservation_elastic(ep, st["rcv"])
        loss = torch.sum((tr - st["obs"]) ** 2)
        return {"traces": tr.detach(), "loss": loss.detach(), "grad": list(torch.autograd.grad(loss, m))}
    plan, srcv, K = st["plan"], st["srcv"], st["K"]
    if kind == "modelling":
        return {"traces": plan.forward(st["model"], srcv, K)}
    if kind == "traces":
        c = st["model"].detach().requires_grad_(True)
        tr = ads.acoustic_traces(plan, c, srcv, K)
        loss = torch.sum((tr - st["obs"]) ** 2)
        return {"traces": tr.detach(), "grad": torch.autograd.grad(loss, c)[0]}
    if kind == "gradient":
        loss, g, _ = plan.gradient(st["model"], srcv, st["obs"], K)
        return {"loss": loss, "grad": g}
    loss, g, _ = plan.gradient(*st["model"], srcv, st["obs"], K)
    return {"loss": loss, "grad": list(g)}


def work(case):
    """Bytes: every input read and every output written once, and for a gradient the wavefield that
    the reverse sweep reads, once written and once read.  Flops: of the scheme's formulas."""
    w = 4 if case["dtype"] == "f32" else 8
    cells = case["nx"] * case["ny"]
    n = float(case["nstep"]) * case["shots"] * (0.8 if case["uneven"] else 1.0)  # shot-levels
    nr = case["nx"] if case["layout"] == "surface" else case["ny"]
    if case["kind"] == "step":
        return {"bytes": 10.0 * w * cells, "flops": 30.0 * cells}
    if case["kind"] == "step_vjp":
        return {"bytes": 25.0 * w * cells, "flops": 100.0 * cells}
    if case["kind"] == "solver":  # u, phi, psi histories; u and its cotangent read back
        return {"bytes": 5.0 * w * cells * n, "flops": 45.0 * cells * n}
    if case["kind"] == "elastic_solver":
        return {"bytes": 15.0 * w * cells * n, "flops": 220.0 * cells * n}
    if case["kind"] == "modelling":
        return {"bytes": w * (cells + nr * n), "flops": 13.0 * cells * n}
    if case["kind"] == "elastic_gradient":
        return {"bytes": w * (10.0 * cells * n + 6.0 * cells + 4.0 * nr * n), "flops": 220.0 * cells * n}
    return {"bytes": w * (2.0 * cells * n + 2.0 * cells + 2.0 * nr * n), "flops": 38.0 * cells * n}


# ---------------------------------------------------------------------------------------------
# the same outputs in 64 bits, plain torch
# ---------------------------------------------------------------------------------------------

def _acoustic_profiles(case):
    """sigma(x), tau(y) on the padded axes."""
    h, _ = _spacing(case)
    out = []
    m = 12 if case["kind"] in ("step", "step_vjp") else case["npml"]
    for n in (case["nx"], case["ny"]):
        L = m * h
        xi = 3000.0 / L * math.log(1.0 / 0.001)
        x = torch.arange(n + 2, dtype=torch.float64) * h
        d = torch.where(x < L, L - x, torch.where(x > h * (n + 1) - L, x - (h * (n + 1) - L), torch.zeros_like(x)))
        out.append(xi * (d / L - torch.sin(2.0 * math.pi * d / L) / (2.0 * math.pi)))
    return out


def _ac_step(k0, dt, h, C, s, t, w, wold, phi, psi):
    """One level on padded arrays (..., nx + 2, ny + 2) whose ring is zero: u before sources, phi, psi."""
    I = (Ellipsis, slice(1, -1), slice(1, -1))
    ip, im = (Ellipsis, slice(2, None), slice(1, -1)), (Ellipsis, slice(None, -2), slice(1, -1))
    jp, jm = (Ellipsis, slice(1, -1), slice(2, None)), (Ellipsis, slice(1, -1), slice(None, -2))
    Ci, si, ti = C[1:-1, 1:-1], s[1:-1, 1:-1], t[1:-1, 1:-1]
    cx = (dt / h) ** 2
    lap = cx * (w[ip] + w[im] + w[jp] + w[jm] - 4.0 * w[I])
    e = dt * dt / (2.0 * h)
    u = ((2.0 - si * ti * dt * dt) * w[I] + Ci * lap + e * (phi[ip] - phi[im]) + e * (psi[jp] - psi[jm])
         - (1.0 - (si + ti) * dt / 2.0) * wold[I]) / (1.0 + (si + ti) * dt / 2.0)
    u = F.pad(u, (1, 1, 1, 1))
    v = u if k0 else w
    f = dt / (2.0 * h)
    phin = F.pad((1.0 - dt * si) * phi[I] + Ci * (ti - si) * f * (v[ip] - v[im]), (1, 1, 1, 1))
    psin = F.pad((1.0 - dt * ti) * psi[I] + Ci * (si - ti) * f * (v[jp] - v[jm]), (1, 1, 1, 1))
    return u, phin, psin


def _exact_steps(case, seed):
    f, cot = _fields(case, seed)
    f, cot = [x.double() for x in f], [x.double() for x in cot]
    h, dt = _spacing(case)
    w, wold, phi, psi, s, t, c = f
    if case["kind"] == "step":
        return _ac_step(False, dt, h, c, s, t, w, wold, phi, psi)
    leaf = [x.requires_grad_(True) for x in (w, wold, phi, psi, c)]
    out = _ac_step(False, dt, h, c, s, t, w, wold, phi, psi)
    # the ring of the outputs is a constant zero
    return [o.detach() for o in out], list(torch.autograd.grad(out, leaf, cot))


def _packed(shots, dev):
    S, R = len(shots), max(len(sh["ri"]) for sh in shots)
    N = max(sh["n"] for sh in shots)
    ri, rj = torch.zeros((2, S, R), dtype=torch.int64)
    ok = torch.zeros((S, R), dtype=torch.bool)
    w = torch.zeros((S, N), dtype=torch.float64, device=dev)
    for q, sh in enumerate(shots):
        k = len(sh["ri"])
        ri[q, :k], rj[q, :k], ok[q, :k] = torch.as_tensor(sh["ri"] - 1), torch.as_tensor(sh["rj"] - 1), True
        w[q, :sh["n"]] = sh["w"]
    si, sj = (torch.as_tensor([sh[k] - 1 for sh in shots], device=dev) for k in ("si", "sj"))
    return N, ri.to(dev), rj.to(dev), ok.to(dev), w, si, sj


def _sweep(N, first, state, step, seg):
    """Runs step(n, *state) -> state, row over first .. N with checkpoints; rows stacked by level."""
    rows, n = [], first

    def block(a, b, *st):
        out = []
        for q in range(a, b):
            st, r = step(q, *st)
            out.append(r)
        return (*st, torch.stack(out))

    while n <= N:
        e = min(N + 1, n + seg)
        *state, r = checkpoint(block, n, e, *state, use_reentrant=False)
        rows.append(r)
        n = e
    return torch.cat(rows)


def _exact_acoustic(case, seed):
    shots, g, dev = _survey(case, seed)
    el = False
    h, dt = _spacing(case)
    d = DT[case["dtype"]]
    nx, ny = case["nx"], case["ny"]
    c = _velocity(g, nx, ny, dev).to(d).double()
    obs = [_observed(case, sh, OBS[el]).to(d).double() for sh in shots]
    for sh in shots:
        sh["w"] = (AMP[el] * sh["w"]).to(d).double()
    sx, ty = _acoustic_profiles(case)
    one = torch.ones((nx + 2, ny + 2), dtype=torch.float64, device=dev)
    s, t = one * sx.to(dev)[:, None], one * ty.to(dev)[None, :]
    k0 = case["kernel"] == 0
    chunk = max(1, int(8e6 / (nx * ny)))
    want = case["kind"] != "modelling"
    grad, loss, traces = torch.zeros_like(c), 0.0, []
    for b in range(0, len(shots), chunk):
        part = shots[b:b + chunk]
        N, ri, rj, ok, w, si, sj = _packed(part, dev)
        S = len(part)
        q = torch.arange(S, device=dev)
        cc = c.clone().requires_grad_(want)

        def step(n, u1, u0, phi, psi):
            u, phi, psi = _ac_step(k0, dt, h, cc * cc, s, t, u1, u0, phi, psi)
            u = u.index_put((q, si, sj), dt * dt * w[:, n - 1], accumulate=True)
            return (u, u1, phi, psi), u[q[:, None], ri, rj]

        z = torch.zeros((S, nx + 2, ny + 2), dtype=torch.float64, device=dev)
        with torch.set_grad_enabled(want):
            rows = _sweep(N, 2, [z, z, z, z], step, max(4, int(math.sqrt(N))))  # levels 2 .. N: (level, shot, receiver)
            tr = torch.cat([torch.zeros_like(rows[:2]), rows])
            L = 0.0
            for e, sh in enumerate(part):
                one_tr = tr[:sh["n"] + 1, e, :len(sh["ri"])]
                traces.append(one_tr.detach().reshape(-1))
                L = L + torch.sum((one_tr - obs[b + e]) ** 2)
        if want:
            grad += torch.autograd.grad(L, cc)[0]
            loss = loss + L.detach()
    flat = torch.cat(traces)
    if case["kind"] == "modelling":
        return {"traces": flat}
    if case["kind"] == "traces":
        return {"traces": flat, "grad": grad}
    if case["kind"] == "solver":
        return {"traces": flat.reshape(case["nstep"] + 1, -1), "loss": loss, "grad": grad}
    return {"loss": loss.reshape(1), "grad": grad}


def _cpml(case, n, dt, h):
    """a, b on the full and the half grid of one axis (profile index 0 is the first interior cell)."""
    f0, vp = 12.0, 4500.0
    m = case["npml"]
    thick = m * h
    d0 = -3.0 * vp * math.log(0.001) / (2.0 * thick)
    amax = 2.0 * math.pi * (f0 / 2.0)
    out = []
    for half in (0.0, h / 2.0):
        x = torch.arange(n, dtype=torch.float64) * h + half
        lo, hi = thick - x, x - ((n - 0.5) * h - thick)
        q = torch.where(hi >= 0, hi, torch.where(lo >= 0, lo, torch.zeros_like(x))) / thick
        d, al = d0 * q ** 2, amax * q
        b = torch.exp(-(d + al) * dt)
        a = torch.where(d.abs() > 1e-6, d * (b - 1.0) / torch.where(d + al > 0, d + al, torch.ones_like(d)), torch.zeros_like(d))
        out += [a, b]
    return out


def _exact_elastic(case, seed):
    shots, g, dev = _survey(case, seed)
    d = DT[case["dtype"]]
    h, dt = _spacing(case)
    dt = 0.8 * dt
    nx, ny = case["nx"], case["ny"]
    model = [m.to(d).double() for m in _elastic_model(g, nx, ny, dev)]
    obs = []
    for sh in shots:
        o = _observed(case, sh, OBS[True])
        obs.append(torch.cat([o, 0.7 * o], 1).T.contiguous().to(d).double())
        sh["w"] = (AMP[True] * sh["w"]).to(d).double()
    px = [v.to(dev)[:, None] for v in _cpml(case, nx, dt, h)]  # a, b full; a, b half
    py = [v.to(dev)[None, :] for v in _cpml(case, ny, dt, h)]

    def sh_(f, lo_i, hi_i, lo_j, hi_j, di=0, dj=0):  # cells [lo, hi] shifted by (di, dj)
        return f[..., lo_i + di:hi_i + di + 1, lo_j + dj:hi_j + dj + 1]

    def diff(f, r, axis, back):  # 4th-order staggered difference, backward or forward half cell
        o = -1 if back else 0
        v = lambda k: sh_(f, *r, *((o + k, 0) if axis == 0 else (0, o + k)))
        return (27.0 * v(1) - 27.0 * v(0) - v(2) + v(-1)) / (24.0 * h)

    def pad(f, r):
        return F.pad(f, (r[2], ny + 1 - r[3], r[0], nx + 1 - r[1]))

    def damped(e, m, r, axis, half):
        a, b = (px if axis == 0 else py)[2 * half:2 * half + 2]
        a, b = (v[r[0] - 1:r[1]] if axis == 0 else v[:, r[2] - 1:r[3]] for v in (a, b))
        m = b * sh_(m, *r) + a * e
        return e + m, pad(m, r)

    R1, R2, R3, R4 = (1, nx - 1, 2, ny), (2, nx, 1, ny - 1), (2, nx, 2, ny), (1, nx - 1, 1, ny - 1)
    chunk = max(1, int(6e6 / (nx * ny)))
    grads, loss, traces = [torch.zeros_like(m) for m in model], 0.0, []
    for b0 in range(0, len(shots), chunk):
        part = shots[b0:b0 + chunk]
        N, ri, rj, ok, w, si, sj = _packed(part, dev)
        S = len(part)
        q = torch.arange(S, device=dev)
        rho, lam, mu = (m.clone().requires_grad_(True) for m in model)

        def step(n, vx, vy, sxx, syy, sxy, m1, m2, m3, m4, m5, m6, m7, m8):
            lb = 0.5 * (sh_(lam, *R1, 1, 0) + sh_(lam, *R1))
            mb = 0.5 * (sh_(mu, *R1, 1, 0) + sh_(mu, *R1))
            ex, m1 = damped(diff(vx, R1, 0, False), m1, R1, 0, 1)
            ey, m2 = damped(diff(vy, R1, 1, True), m2, R1, 1, 0)
            sxx = sxx + pad(((lb + 2 * mb) * ex + lb * ey) * dt, R1)
            syy = syy + pad(((lb + 2 * mb) * ey + lb * ex) * dt, R1)
            mb = 0.5 * (sh_(mu, *R2) + sh_(mu, *R2, 0, 1))
            ex, m3 = damped(diff(vy, R2, 0, True), m3, R2, 0, 0)
            ey, m4 = damped(diff(vx, R2, 1, False), m4, R2, 1, 1)
            sxy = sxy + pad(mb * (ex + ey) * dt, R2)
            ex, m5 = damped(diff(sxx, R3, 0, True), m5, R3, 0, 0)
            ey, m6 = damped(diff(sxy, R3, 1, True), m6, R3, 1, 0)
            vx = vx + pad((ex + ey) * dt / sh_(rho, *R3), R3)
            rb = 0.25 * (sh_(rho, *R4) + sh_(rho, *R4, 1, 0) + sh_(rho, *R4, 1, 1) + sh_(rho, *R4, 0, 1))
            ex, m7 = damped(diff(sxy, R4, 0, False), m7, R4, 0, 1)
            ey, m8 = damped(diff(syy, R4, 1, False), m8, R4, 1, 1)
            vy = vy + pad((ex + ey) * dt / rb, R4)
            sxx = sxx.index_put((q, si, sj), w[:, n - 1], accumulate=True)
            syy = syy.index_put((q, si, sj), w[:, n - 1], accumulate=True)
            row = torch.cat([vx[q[:, None], ri, rj], vy[q[:, None], ri, rj]], 1)
            return (vx, vy, sxx, syy, sxy, m1, m2, m3, m4, m5, m6, m7, m8), row

        z = torch.zeros((S, nx + 2, ny + 2), dtype=torch.float64, device=dev)
        rows = _sweep(N, 1, [z] * 13, step, max(4, int(math.sqrt(N) / 2)))
        tr = torch.cat([torch.zeros_like(rows[:1]), rows]).permute(1, 2, 0)  # shot, receiver, level
        L = 0.0
        for e in range(S):
            traces.append(tr[e].detach())
            L = L + torch.sum((tr[e] - obs[b0 + e]) ** 2)
        for a, x in zip(grads, torch.autograd.grad(L, (rho, lam, mu))):
            a += x
        loss = loss + L.detach()
    if case["kind"] == "elastic_solver":
        return {"traces": traces[0], "loss": loss, "grad": grads}
    return {"loss": loss.reshape(1), "grad": grads}


def exact(case, seed):
    cost = float(case["nx"]) * case["ny"] * case["shots"] * case["nstep"]
    if cost > (4e9 if case["kind"].startswith("elastic") else 2e10):
        return None  # longer than 20 seconds
    if case["kind"] in ("step", "step_vjp"):
        return _exact_steps(case, seed)
    return _exact_elastic(case, seed) if case["kind"].startswith("elastic") else _exact_acoustic(case, seed)
