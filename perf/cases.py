"""The work that a user of cfdx has the GPU do, as cases that can be timed and compared.

A case is one program: its blocks are set up once (grid, initial state, run parameters), and a pass
advances them through the public entry points and reads the state back, or evaluates the right-hand
side into a device array. The sizes are those of the benchmark workloads (package module
`workloads`), of the served C-grid ladder (`serve.C5_LADDER`) and of the tests, with ragged ones
between them.

Kinds:
  rhs      Block.rhs_noalloc into a device tensor (a caller with its own time integrator)
  step     Block.step, direct launches, then the state (a single solve)
  batch    Batch.step, replayed step graph, of periodic cubes, then every block's state
  monitor  the iteration loop of driver.Run: one step and its residual per iteration, then the state
  dropin   DropInSolver.step: the reference's three kernels and record layouts, then FLOW
C-grid blocks (kinds step, batch, monitor with "cgrid") carry side conditions and a wake cut.

Double-precision results are returned in double. A mixed-precision solve is accurate to about 1e-6
(its fluxes are 32-bit), so its state is returned, as such a program stores it, in 32 bits.
"""
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "high-order-accurate-cfd-solver-code-for-heterogenous-hardware-cpu-and-gpgpu-_amd")

_ctx = None


def _cfdx():
    """The package (imported after torch, whose HIP runtime the library then shares)."""
    if "cfdx" not in sys.modules:
        spec = importlib.util.spec_from_file_location("cfdx", os.path.join(PKG, "__init__.py"),
                                                      submodule_search_locations=[PKG])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["cfdx"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["cfdx"]


def _context():
    """One context for the process, on torch's current stream: library work and tensors in order."""
    global _ctx
    if _ctx is None:
        s = torch.cuda.Stream()
        torch.cuda.set_stream(s)
        _ctx = _cfdx().Ctx(0, stream=s.cuda_stream)
    return _ctx


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest call there is: one right-hand side of a block of 960 nodes (all launch latency)
        dict(name="rhs_12x10x8", kind="rhs", ni=12, nj=10, nk=8, precision="fp64", model="mts", flow="tgv", mach=0.3,
             reyl=1600.0),
        # the Euler validation run: isentropic vortex, 64^3, 100 steps
        dict(name="vortex_64_euler", kind="step", ni=64, nj=64, nk=64, precision="fp64", model="euler", flow="vortex",
             mach=0.5, reyl=1600.0, steps=100),
        # a small cube on its own, mixed precision: the replayed graph of short launches
        dict(name="cube_32_mixed", kind="batch", sizes="32x32x32", precision="mixed", model="mts", steps=200),
        # the Taylor-Green LES at 128^3 in double, one solve on its own
        dict(name="tgv_128_fp64", kind="step", ni=128, nj=128, nk=128, precision="fp64", model="mts", flow="tgv",
             mach=0.1, reyl=1600.0, steps=60),
        # the same solve in mixed precision
        dict(name="tgv_128_mixed", kind="step", ni=128, nj=128, nk=128, precision="mixed", model="mts", flow="tgv",
             mach=0.1, reyl=1600.0, steps=100),
        # the headline size: 256^3 in double, one block replaying its step graph
        dict(name="tgv_256_fp64", kind="batch", sizes="256x256x256", precision="fp64", model="mts", steps=40),
        # the Smagorinsky option on a ragged block, no size a multiple of a tile
        dict(name="smag_97x83x61", kind="step", ni=97, nj=83, nk=61, precision="fp64", model="smagorinsky", flow="tgv",
             mach=0.2, reyl=1600.0, steps=100),
        # an airfoil solve in double on the ladder's largest C-grid
        dict(name="cgrid_384_fp64", kind="step", cgrid=True, ni=384, nj=128, nk=32, precision="fp64", model="mts",
             steps=60),
        # one iteration after the other with its residual, on the ladder's smallest C-grid
        dict(name="cgrid_128_monitor", kind="monitor", cgrid=True, ni=128, nj=64, nk=16, precision="fp64", model="mts",
             steps=100),
        # a server's batch: the C-grid ladder in flight together, mixed precision
        dict(name="cgrids_batch_mixed", kind="batch", cgrid=True, sizes="128x64x16,192x96x24,256x128x32,384x128x32",
             precision="mixed", model="mts", steps=40),
        # uneven cubes (edges of the 64-cube workload) batched in mixed precision
        dict(name="cubes_batch_mixed", kind="batch", sizes="32x32x32,48x48x48,64x64x64,96x96x96,128x128x128,64x64x64,"
             "96x96x96,48x48x48", precision="mixed", model="mts", steps=60),
        # the reference's kernel boundary: its record layouts and its call sequence
        dict(name="dropin_48x40x36", kind="dropin", ni=48, nj=40, nk=36, precision="fp64", model="mts", flow="tgv",
             mach=0.3, reyl=1000.0, steps=10),
    ]


CGRIDS = ((128, 64, 16), (192, 96, 24), (256, 128, 32), (384, 128, 32))   # the served ladder


def draw(rng):
    """A case of the same ranges: blocks of 8 .. 192 nodes a side (log-uniform, odd sizes as they
    come), ladder C-grids and ragged ones between them, batches of 1 .. 8 blocks."""
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def steps(nodes):
        return max(10, min(200, int(1.2e8 / nodes)))

    def cgrid():
        if rng.random() < 0.5:
            return CGRIDS[rng.randrange(4)]
        return (2 * side(32, 192), side(24, 128), side(7, 32))

    kind = rng.choice(["rhs", "step", "step", "batch", "batch", "cgrid", "cgrid", "cgrids", "monitor", "dropin"])
    c = dict(precision=rng.choice(["fp64", "mixed"]), model=rng.choice(["mts", "mts", "smagorinsky"]))
    flow = dict(flow="tgv", mach=round(rng.uniform(0.1, 0.6), 3), reyl=round(rng.uniform(500.0, 5000.0), 1))
    if kind == "rhs":
        c.update(kind="rhs", ni=side(8, 112), nj=side(8, 112), nk=side(8, 112), **flow)
        c.update(precision="fp64", mach=round(rng.uniform(0.3, 0.6), 3))
    elif kind == "step":
        c.update(kind="step", ni=side(16, 192), nj=side(16, 160), nk=side(16, 160), **flow)
        if rng.random() < 0.3:
            c.update(model="euler", flow="vortex", mach=round(rng.uniform(0.4, 0.6), 3))
        c.update(steps=steps(c["ni"] * c["nj"] * c["nk"]))
    elif kind == "batch":
        e = [(side(24, 128),) * 3 if rng.random() < 0.5 else (side(24, 128), side(24, 128), side(24, 128))
             for _ in range(rng.randint(1, 8))]
        c.update(kind="batch", sizes=",".join("%dx%dx%d" % s for s in e), steps=steps(sum(a * b * k for a, b, k in e)))
    elif kind == "cgrid":
        s = cgrid()
        c.update(kind="step", cgrid=True, ni=s[0], nj=s[1], nk=s[2], steps=min(100, steps(s[0] * s[1] * s[2])))
    elif kind == "cgrids":
        e = [cgrid() for _ in range(rng.randint(2, 6))]
        c.update(kind="batch", cgrid=True, sizes=",".join("%dx%dx%d" % s for s in e),
                 steps=min(100, steps(sum(a * b * k for a, b, k in e))))
    elif kind == "monitor":
        s = cgrid()
        c.update(kind="monitor", cgrid=True, ni=s[0], nj=s[1], nk=s[2], precision="fp64",
                 steps=min(100, steps(s[0] * s[1] * s[2])))
    else:
        c.update(kind="dropin", ni=side(12, 64), nj=side(12, 64), nk=side(12, 64), precision="fp64", **flow)
        c.update(steps=rng.randint(5, 20))
    return c


def _sizes(case):
    if "sizes" in case:
        return [tuple(int(x) for x in s.split("x")) for s in case["sizes"].split(",")]
    return [(case["ni"], case["nj"], case["nk"])]


def _specs(case, seed):
    """Per block, what the seed draws: the map's phases; in a batch of cubes the flow, Mach and
    Reynolds number; for a C-grid the NACA section, the angle of attack, Mach and Reynolds number
    (the ranges of the 64-cube and the served workloads)."""
    rng = np.random.default_rng(seed)
    out = []
    for ni, nj, nk in _sizes(case):
        s = dict(ni=ni, nj=nj, nk=nk)
        if case.get("cgrid"):
            s.update(naca=(float(rng.uniform(0.0, 0.04)), 0.4, float(rng.uniform(0.08, 0.18))),
                     aoa=float(rng.uniform(-4.0, 10.0)), mach=float(rng.uniform(0.3, 0.7)), reyl=float(rng.uniform(1e5, 1e6)))
        else:
            s.update(phases=[float(x) for x in rng.uniform(0, 2 * math.pi, 3)])
            if "flow" in case:
                s.update(flow=case["flow"], mach=case["mach"], reyl=case["reyl"])
            else:
                s.update(flow="tgv" if rng.integers(2) else "vortex", mach=float(rng.uniform(0.1, 0.6)),
                         reyl=float(rng.uniform(500.0, 5000.0)))
                if max(ni, nj, nk) >= 192:   # the 256^3 run is the Taylor-Green LES
                    s.update(flow="tgv", mach=0.1, reyl=1600.0)
            L = 10.0 if s["flow"] == "vortex" else 2 * math.pi
            s.update(length=L, amp=0.05 * L / max(ni, nj, nk))
            if case["kind"] == "step" and s["flow"] == "vortex":
                # a Cartesian box, the vortex anywhere in it
                s.update(amp=0.0, center=(float(rng.uniform(3, 7)), float(rng.uniform(3, 7))))
            # a fixed step at a CFL number of about 0.4
            h = L / max(ni, nj, nk)
            speed = 2.0 if s["flow"] == "tgv" else 2.0 + 2.8 / s["mach"]
            s.update(dt=0.4 * h / (speed + 3.0 / s["mach"]))
        out.append(s)
    return out


def _params(case, s):
    X = _cfdx()
    if case["model"] == "euler":
        return X.euler_params()
    return X.default_params(mach=s["mach"], reyl=s["reyl"], sgs=case["model"])


def _block(case, s):
    """The block of one solve, initialised and configured; its parameters and time step."""
    X = _cfdx()
    prec = X.MIXED if case["precision"] == "mixed" else X.FP64
    p = _params(case, s)
    if case.get("cgrid"):
        d, g = X.cgrid_desc(s["ni"], s["nj"], s["nk"], prec, naca=s["naca"], aoa_deg=s["aoa"])
        b = X.Block.of(d, ctx=_context())
        b.set_geometry_soa(X.cgrid_geometry(d, g)[1])
        b.configure(s["mach"], 0.0, p)
        b.set_flow(X.freestream(b.n, s["mach"], s["aoa"]))
        dt = b.cfl_dt(0.5)
    else:
        b = X.Block(s["ni"], s["nj"], s["nk"], precision=prec, ctx=_context())
        b.init_case(grid="sinusoid", length=(s["length"],) * 3, amp=s["amp"], phases=s["phases"], init=s["flow"],
                    mach=s["mach"], center=s.get("center", (5.0, 5.0)))
        dt = s["dt"]
    b.configure(s["mach"], dt, p)
    return b, p, dt


class _Device:
    """A device tensor as the library's device-buffer arguments take it."""

    def __init__(self, t):
        self.tensor, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def prepare(case, seed):
    X = _cfdx()
    specs = _specs(case, seed)
    st = dict(kind=case["kind"], steps=case.get("steps", 1), single=case["precision"] == "mixed")
    if case["kind"] == "dropin":
        s = specs[0]
        host = X.periodic_case(s["ni"], s["nj"], s["nk"], grid="sinusoid", length=(s["length"],) * 3, amp=s["amp"],
                               phases=s["phases"], init=s["flow"], mach=s["mach"])
        st.update(solver=X.DropInSolver(host, ctx=_context()), mach=s["mach"], dt=s["dt"], params=_params(case, s))
        return st
    made = [_block(case, s) for s in specs]
    st.update(blocks=[m[0] for m in made], params=[m[1] for m in made], dt=[m[2] for m in made],
              mach=[s["mach"] for s in specs])
    if case["kind"] == "rhs":
        st.update(out=_Device(torch.zeros((5, made[0][0].n), dtype=torch.float64, device="cuda")))
    elif case["kind"] == "batch":
        q = X.Batch(precision=X.MIXED if case["precision"] == "mixed" else X.FP64, ctx=_context())
        for b in st["blocks"]:
            q.add(b)
        st.update(batch=q)
    elif case["kind"] == "monitor":
        st["blocks"][0].set_monitor(True)
    return st


def _fields(flow, single):
    """A FLOW record array as the fields a program keeps."""
    a = torch.from_numpy(flow.view(np.float64).reshape(-1, 9))
    if single:
        a = a.float()
    # record order: u, v, w, p, t, rho, mu, a, e
    return dict(velocity=a[:, 0:3], p=a[:, 3], t=a[:, 4], rho=a[:, 5], mu=a[:, 6], a=a[:, 7], e=a[:, 8])


def run(st):
    kind, n = st["kind"], st["steps"]
    if kind == "dropin":
        st["solver"].step(n, st["mach"], st["dt"], st["params"])
        return _fields(st["solver"].flow()[1:], False)
    b = st["blocks"][0]
    if kind == "rhs":
        b.rhs_noalloc(st["params"][0], st["out"])
        return st["out"].tensor
    if kind == "step":
        b.step(n, st["mach"][0], st["dt"][0], st["params"][0])
        return _fields(b.get_flow(), st["single"])
    if kind == "monitor":
        history = []
        for _ in range(n):
            b.step(1, st["mach"][0], st["dt"][0], st["params"][0])
            history.append(b.residual())
        return dict(_fields(b.get_flow(), False), history=np.array(history))
    st["batch"].step(n)
    return [_fields(x.get_flow(), st["single"]) for x in st["blocks"]]


def work(case):
    """What a pass cannot do without: per step the scheme's operations (three stages of three face
    fluxes, the viscous node fluxes and the update) and one reading of geometry and state with one
    writing of the state per stage, and the state read back."""
    nodes = sum(a * b * k for a, b, k in _sizes(case))
    flops = 10100 if case["model"] == "euler" else 11772
    if case["kind"] == "rhs":
        return dict(bytes=nodes * (22 + 5 + 5) * 8, flops=nodes * flops // 3)
    if case["kind"] == "dropin":   # per stage its records: FLOW, GRID, det, metric, deter, U in and out
        return dict(bytes=nodes * (72 + case["steps"] * 3 * (72 * 2 + 56 + 8 + 504 + 48 + 80)), flops=nodes * flops * case["steps"])
    # geometry 22, stage vector in and out 10, RK base 5 at two of three stages
    per_stage = 22 * (4 if case["precision"] == "mixed" else 8) + 10 * 8 + 5 * 8 * 2 // 3
    return dict(bytes=nodes * (72 + case["steps"] * 3 * per_stage), flops=nodes * flops * case["steps"])


# ---------------------------------------------------------------------------
# the periodic scheme in 64 bits, in plain tensor operations
# ---------------------------------------------------------------------------
def _at(a, d, o):
    """The values at offset o along direction d (0: i, the last axis)."""
    return a if o == 0 else torch.roll(a, -o, dims=a.dim() - 1 - d)


def _geometry(s, dev):
    """det, metric rows m[d][c] and the +1/2-face rows and dets of the sinusoidal map; coordinates."""
    n = (s["ni"], s["nj"], s["nk"])
    L, A, ph = s["length"], s["amp"], s["phases"]
    w = 2.0 * math.pi / L
    h = [L / q for q in n]
    i, j, k = (torch.arange(q, dtype=torch.float64, device=dev) for q in n)
    s1, s2, s3 = (i * h[0])[None, None, :], (j * h[1])[None, :, None], (k * h[2])[:, None, None]
    full = torch.zeros((n[2], n[1], n[0]), dtype=torch.float64, device=dev)
    S, C = torch.sin, torch.cos
    x = s1 + A * S(w * s2 + ph[0]) * S(w * s3 + ph[0]) + full
    y = s2 + A * S(w * s3 + ph[1]) * S(w * s1 + ph[1]) + full
    z = s3 + A * S(w * s1 + ph[2]) * S(w * s2 + ph[2]) + full
    J = [[h[0] + full, h[1] * A * w * C(w * s2 + ph[0]) * S(w * s3 + ph[0]) + full, h[2] * A * w * S(w * s2 + ph[0]) * C(w * s3 + ph[0]) + full],
         [h[0] * A * w * S(w * s3 + ph[1]) * C(w * s1 + ph[1]) + full, h[1] + full, h[2] * A * w * C(w * s3 + ph[1]) * S(w * s1 + ph[1]) + full],
         [h[0] * A * w * C(w * s1 + ph[2]) * S(w * s2 + ph[2]) + full, h[1] * A * w * S(w * s1 + ph[2]) * C(w * s2 + ph[2]) + full, h[2] + full]]
    cof = [[J[(c + 1) % 3][(d + 1) % 3] * J[(c + 2) % 3][(d + 2) % 3] - J[(c + 1) % 3][(d + 2) % 3] * J[(c + 2) % 3][(d + 1) % 3]
            for c in range(3)] for d in range(3)]
    D = sum(J[0][d] * cof[d][0] for d in range(3))
    m = [torch.stack([cof[d][c] / D for c in range(3)]) for d in range(3)]

    def half(f, d):
        return sum(c * _at(f, d, o) for o, c in zip(range(-2, 4), (3, -25, 150, 150, -25, 3))) / 256.0

    return (x, y, z), D, m, [half(m[d], d) for d in range(3)], [half(D, d) for d in range(3)]


def _initial(s, xyz):
    x, y, z = xyz
    M = s["mach"]
    pinf = 1.0 / (1.4 * M * M)
    if s["flow"] == "tgv":
        u, v = torch.sin(x) * torch.cos(y) * torch.cos(z), -torch.cos(x) * torch.sin(y) * torch.cos(z)
        p = pinf + (torch.cos(2 * x) + torch.cos(2 * y)) * (torch.cos(2 * z) + 2.0) / 16.0
        return torch.stack([1.4 * M * M * p, u, v, torch.zeros_like(u), p])
    beta, (xc, yc) = 5.0, s.get("center", (5.0, 5.0))
    dx, dy = x - xc, y - yc
    r2 = dx * dx + dy * dy
    e = beta / (2.0 * math.pi) * torch.exp(0.5 * (1.0 - r2)) / M
    T = 1.0 - 0.4 * beta * beta / (8.0 * 1.4 * math.pi ** 2) * torch.exp(1.0 - r2)
    rho = T ** 2.5
    return torch.stack([rho, 1.0 - e * dy, e * dx, torch.zeros_like(x), rho * T / (1.4 * M * M)])


def _conserved(P):
    rho, u, v, w, p = P
    return torch.stack([rho, rho * u, rho * v, rho * w, p / 0.4 + 0.5 * rho * (u * u + v * v + w * w)])


def _viscous(U, D, m, model, mach, reyl):
    """The viscous and sub-grid node fluxes along the three directions (5, ...) each, and mu."""
    Pr, Tinf, Cmts, Ct, Cs = 0.72, 273.0, 0.03, 10.0, 0.17
    iU = 1.0 / U[0]
    V = U[1:4] * iU
    e = U[4] * iU - 0.5 * (V * V).sum(0)
    gV, ge, KS = [], [], []
    for d in range(3):
        um, up = _at(U, d, -1), _at(U, d, 1)
        dU = (8.0 * (up - um) - (_at(U, d, 2) - _at(U, d, -2))) / 12.0
        g = (dU[1:4] - V * dU[0]) * iU
        gV.append(g)
        ge.append((dU[4] - U[4] * iU * dU[0]) * iU - (V * g).sum(0))
        f = 0.25 * um + 0.5 * U + 0.25 * up
        KS.append((V[d] - f[1 + d] / f[0]).abs())
    # Cartesian gradients: G[c][a] = d V_c / d x_a
    G = [[sum(gV[d][c] * m[d][a] for d in range(3)) for a in range(3)] for c in range(3)]
    E = [sum(ge[d] * m[d][a] for d in range(3)) for a in range(3)]
    T = 1.4 * mach * mach * 0.4 * e
    mu = T ** 1.5 * (1.0 + 110.4 / Tinf) / (T + 110.4 / Tinf)
    div = G[0][0] + G[1][1] + G[2][2]
    mr = mu / reyl
    tau = [[mr * (G[a][b] + G[b][a] - (2.0 / 3.0 * div if a == b else 0.0)) for b in range(3)] for a in range(3)]
    q = [-mu * 1.4 / (Pr * reyl) * E[a] for a in range(3)]
    Sh = [[0.5 * (G[a][b] + G[b][a]) for b in range(3)] for a in range(3)]
    diag = sum(Sh[a][a] ** 2 for a in range(3))
    off = Sh[0][1] ** 2 + Sh[1][2] ** 2 + Sh[0][2] ** 2
    delta = D ** (-1.0 / 3.0)
    if model == "smagorinsky":
        eddy = [Cs * Cs * delta * torch.sqrt(2.0 * diag + 4.0 * off)] * 3
    else:
        mod = torch.sqrt(2.0 * (off + 2.0 / 3.0 * diag))
        eddy = [torch.where(mod != 0, Cmts * delta * k * k / torch.where(mod != 0, k + delta * mod / Ct, 1.0), Cmts * delta * k) for k in KS]
    pair = {(0, 1): 0, (1, 2): 1, (0, 2): 2, (0, 0): 0, (1, 1): 1, (2, 2): 2}
    sgs = [[-2.0 * U[0] * eddy[pair[tuple(sorted((a, b)))]] * Sh[a][b] for b in range(3)] for a in range(3)]
    flux = []
    for a in range(3):
        if model == "smagorinsky":
            H = -1.4 / Pr * U[0] * eddy[0] * E[a] + sum(V[b] * sgs[a][b] for b in range(3))
        else:
            Q = -eddy[a] * E[a] / (1.4 * 0.4 * mach * mach)
            H = 1.4 * Q + (sgs[a][0] + sgs[a][1] + sgs[a][2]) * V[a]
        flux.append(torch.stack([torch.zeros_like(e)] + [sgs[a][b] - tau[a][b] for b in range(3)]
                                + [q[a] + H - sum(V[b] * tau[a][b] for b in range(3))]))
    return [D * sum(m[d][a] * flux[a] for a in range(3)) for d in range(3)], mu


def _flux(Q, k):
    """Inviscid flux of conserved states along the row k, and the velocity along it and the pressure."""
    r = 1.0 / Q[0]
    un = (Q[1] * k[0] + Q[2] * k[1] + Q[3] * k[2]) * r
    p = 0.4 * (Q[4] - 0.5 * (Q[1] ** 2 + Q[2] ** 2 + Q[3] ** 2) * r)
    return torch.stack([Q[0] * un, Q[1] * un + k[0] * p, Q[2] * un + k[1] * p, Q[3] * un + k[2] * p, (Q[4] + p) * un]), un, p


def _weno(a, b, c, q, d, eps):
    """Weighted mean of three candidates q with linear weights d; a, b, c: their indicators."""
    w = [di / (eps + i) ** 2 for di, i in zip(d, (a, b, c))]
    return (w[0] * q[0] + w[1] * q[1] + w[2] * q[2]) / (w[0] + w[1] + w[2])


def _face_flux(Q, F, d, kf, df, eps):
    """F-hat at the +1/2 faces along d: characteristic WCNS, local Lax-Friedrichs, midpoint correction."""
    kn = torch.sqrt((kf * kf).sum(0))
    k = kf / kn
    R = _at(Q, d, 1)
    sa, sb = torch.sqrt(Q[0]), torch.sqrt(R[0])

    def vel_h(q):
        v = q[1:4] / q[0]
        return torch.cat([v, ((1.4 * q[4] - 0.2 * q[0] * (v * v).sum(0)) / q[0])[None]])

    av = (sa * vel_h(Q) + sb * vel_h(R)) / (sa + sb)
    u, v, w, h = av
    rho = sa * sb
    q2 = u * u + v * v + w * w
    a = torch.sqrt(0.4 * (h - 0.5 * q2))
    th, phi = k[0] * u + k[1] * v + k[2] * w, 0.2 * q2
    c = [k[2] * v - k[1] * w, k[0] * w - k[2] * u, k[1] * u - k[0] * v]
    r2 = math.sqrt(0.5)
    al, be = rho / a * r2, r2 / (rho * a)
    W = []
    for o in range(-2, 4):
        x = _at(Q, d, o)
        mm = u * x[1] + v * x[2] + w * x[3] - x[4]
        E = (1.0 - phi / a ** 2) * x[0] + 0.4 / a ** 2 * mm
        nn = k[0] * x[1] + k[1] * x[2] + k[2] * x[3]
        A, B = be * (phi * x[0] - 0.4 * mm), be * a * (th * x[0] - nn)
        W.append(torch.stack([k[0] * E + (k[2] * x[2] - k[1] * x[3] - c[0] * x[0]) / rho,
                              k[1] * E + (k[0] * x[3] - k[2] * x[1] - c[1] * x[0]) / rho,
                              k[2] * E + (k[1] * x[1] - k[0] * x[2] - c[2] * x[0]) / rho, A - B, A + B]))

    def smooth(p, q, r, t):
        return 13.0 / 12.0 * (p - 2 * q + r) ** 2 + 0.25 * t ** 2

    mid = [(3 * W[2] + 6 * W[3] - W[4]) / 8, (-W[1] + 6 * W[2] + 3 * W[3]) / 8]
    pos = _weno(smooth(W[3], W[4], W[5], 3 * W[3] - 4 * W[4] + W[5]), smooth(W[2], W[3], W[4], W[4] - W[2]),
                smooth(W[1], W[2], W[3], W[1] - 4 * W[2] + 3 * W[3]),
                ((15 * W[3] - 10 * W[4] + 3 * W[5]) / 8, mid[0], mid[1]), (1 / 16, 5 / 8, 5 / 16), eps)
    neg = _weno(smooth(W[2], W[3], W[4], 3 * W[2] - 4 * W[3] + W[4]), smooth(W[1], W[2], W[3], W[3] - W[1]),
                smooth(W[0], W[1], W[2], W[0] - 4 * W[1] + 3 * W[2]),
                (mid[0], mid[1], (3 * W[0] - 10 * W[1] + 15 * W[2]) / 8), (5 / 16, 5 / 8, 1 / 16), eps)

    def back(x):
        X, Pp, Mm = k[0] * x[0] + k[1] * x[1] + k[2] * x[2], al * (x[3] + x[4]), al * a * (x[3] - x[4])
        return torch.stack([X + Pp, u * (X + Pp) + k[0] * Mm + rho * (k[1] * x[2] - k[2] * x[1]),
                            v * (X + Pp) + k[1] * Mm + rho * (k[2] * x[0] - k[0] * x[2]),
                            w * (X + Pp) + k[2] * Mm + rho * (k[0] * x[1] - k[1] * x[0]),
                            2.5 * phi * X + 2.5 * (phi + a * a) * Pp + th * Mm + rho * (c[0] * x[0] + c[1] * x[1] + c[2] * x[2])])

    qp, qn = back(pos), back(neg)
    fp, lp, pp = _flux(qp, k)
    fn, ln, pn = _flux(qn, k)
    lam = torch.maximum((lp + torch.sqrt(1.4 * pp / qp[0])).abs(), (ln + torch.sqrt(1.4 * pn / qn[0])).abs())
    mc = (57.0 * (_at(F, d, -2) + _at(F, d, 3)) - 411.0 * (_at(F, d, -1) + _at(F, d, 2)) + 354.0 * (F + _at(F, d, 1))) / 11520.0
    return 0.5 * df * kn * (fp + fn - lam * (qp - qn)) + mc


def _rhs(P, U, geo, model, mach, reyl):
    _, D, m, kf, df = geo
    Q = _conserved(P)
    L, mu = torch.zeros_like(U), None
    if model != "euler":
        Fv, mu = _viscous(U, D, m, model, mach, reyl)
    for d in range(3):
        f = _face_flux(Q, D * _flux(Q, m[d])[0], d, kf[d], df[d], 1e-7)
        L -= f - _at(f, d, -1)
        if model != "euler":
            L -= (8.0 * (_at(Fv[d], d, 1) - _at(Fv[d], d, -1)) - (_at(Fv[d], d, 2) - _at(Fv[d], d, -2))) / 12.0
    return L, mu


def _solve(s, model, steps, dev):
    """The fields after `steps` SSP-RK3 steps; steps = 0: the right-hand side of the initial state."""
    geo = _geometry(s, dev)
    D = geo[1]
    P = _initial(s, geo[0])
    if steps == 0:
        return _rhs(P, D * _conserved(P), geo, model, s["mach"], s["reyl"])[0].reshape(5, -1).cpu()
    dt, mu = s["dt"], None
    for _ in range(steps):
        U0 = U = D * _conserved(P)
        for a, b in ((0.0, 1.0), (0.75, 0.25), (1.0 / 3.0, 2.0 / 3.0)):
            L, mu = _rhs(P, U, geo, model, s["mach"], s["reyl"])
            U = a * U0 + b * (U + dt * L)
            q = U / D
            v = q[1:4] / q[0]
            P = torch.cat([q[0:1], v, 0.4 * (q[4:5] - 0.5 * q[0] * (v * v).sum(0, keepdim=True))])
    rho, p = P[0], P[4]
    out = dict(velocity=P[1:4].reshape(3, -1).T, p=p, t=1.4 * s["mach"] ** 2 * p / rho, rho=rho,
               mu=torch.zeros_like(p) if mu is None else mu, a=torch.sqrt(1.4 * p / rho), e=p / (0.4 * rho))
    return {key: (x if key == "velocity" else x.reshape(-1)).cpu() for key, x in out.items()}


def exact(case, seed):
    """The pass in 64 bits. None for a C-grid, whose metrics are the package's, and where the plain
    form takes too long."""
    if case.get("cgrid"):
        return None
    nodes = sum(a * b * k for a, b, k in _sizes(case))
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    if nodes * case.get("steps", 1) > (3e8 if dev == "cuda" else 3e5):
        return None
    steps = 0 if case["kind"] == "rhs" else case["steps"]
    got = [_solve(s, case["model"], steps, dev) for s in _specs(case, seed)]
    return got if case["kind"] == "batch" else got[0]
