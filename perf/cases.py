"""The measured cases of the solver: whole runs through the public entry points.

One pass is what a user's program does with a solver it keeps: load an initial state from
device tensors, advance it, read the fields and the populations back as device tensors; or, for
the differentiable solver, run forward and backward through autograd. The sizes are those of the
repository's benchmark scenarios and tests (64^2 .. 8192^2 and 3-D up to 256 x 128 x 96 and beyond), with
odd and ragged grids among them. `exact` restates the same runs in plain torch, in 64 bits.
"""
from __future__ import annotations

import ctypes
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "cuda-lbm_amd"))

from lbm_amd import Config, Config3D, Solver, Solver3D, abi as A  # noqa: E402
from lbm_amd.autograd import Simulation  # noqa: E402

DEV = "cuda"
COLL = {"bgk": A.LBM_BGK, "mrt": A.LBM_MRT, "cm": A.LBM_CM}
STORE = {"f32": A.LBM_F32, "f16": A.LBM_F16_SHIFTED, "bf16": A.LBM_BF16_SHIFTED}
# multiply-adds and other arithmetic of one node update, in flops: moments, equilibrium,
# relaxation and (where the operator has them) the moment transforms
FLOPS = {("2d", "bgk"): 110, ("2d", "mrt"): 150, ("2d", "cm"): 220,
         ("3d", "bgk"): 330, ("3d", "mrt"): 400, ("3d", "cm"): 420}
U_LID = 0.1
U_IN = 0.05
NU = 0.02


def listed():
    return [
        # the smallest call: a few steps of a validation-sized vortex; launches and latency count
        dict(name="vortex_64_bgk_f32", kind="d2q9", layout="periodic", nx=64, ny=64, coll="bgk", storage="f32", steps=20),
        # the 2-D Taylor-Green validation run
        dict(name="vortex_128_bgk_f32", kind="d2q9", layout="periodic", nx=128, ny=128, coll="bgk", storage="f32", steps=200),
        # the headline workload: lid-driven cavity 1024^2, MRT, single precision
        dict(name="cavity_1024_mrt_f32", kind="d2q9", layout="cavity", nx=1024, ny=1024, coll="mrt", storage="f32", steps=200),
        # a cavity of odd size with 16-bit storage and an odd number of steps
        dict(name="cavity_777x611_mrt_f16", kind="d2q9", layout="cavity", nx=777, ny=611, coll="mrt", storage="f16", steps=151),
        # the force-driven channel of the Poiseuille scenario, CM, 16-bit storage
        dict(name="channel_4096x1024_cm_bf16", kind="d2q9", layout="channel", nx=4096, ny=1024, coll="cm", storage="bf16", steps=60),
        # the same channel with the operator's adaptive rates (domain means in every step)
        dict(name="channel_4096x1024_adapter_f32", kind="d2q9", layout="adapter", nx=4096, ny=1024, coll="cm", storage="f32", steps=30),
        # the largest: a periodic box far beyond the caches
        dict(name="box_8192_bgk_f32", kind="d2q9", layout="periodic", nx=8192, ny=8192, coll="bgk", storage="f32", steps=40),
        # flow past a cylinder, immersed boundary
        dict(name="cylinder_2048x512_cm_f32", kind="cylinder", layout="cylinder", nx=2048, ny=512, coll="cm", storage="f32", steps=100),
        # the inverse problem's forward and backward
        dict(name="inverse_512_bgk", kind="adjoint", layout="periodic", nx=512, ny=512, coll="bgk", storage="f32", steps=200, every=50),
        # the 3-D Taylor-Green scenario
        dict(name="vortex3d_128_bgk_f32", kind="d3q27", layout="periodic", nx=128, ny=128, nz=128, coll="bgk", storage="f32", steps=20),
        # a ragged 3-D box, MRT, 16-bit storage, odd step count
        dict(name="box3d_250x201x150_mrt_f16", kind="d3q27", layout="periodic", nx=250, ny=201, nz=150, coll="mrt", storage="f16", steps=21),
        # the wind tunnel scenario: Guo inlet and outlet, walls, an immersed sphere
        dict(name="tunnel_256x128x96_sphere_cm_f32", kind="tunnel", layout="tunnel", nx=256, ny=128, nz=96, coll="cm", storage="f32", steps=20, markers=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    coll = rng.choice(["bgk", "mrt", "cm"])
    storage = rng.choice(["f32", "f32", "f16", "bf16"])
    if pick < 0.5:
        layout = rng.choice(["periodic", "periodic", "cavity", "channel", "adapter"])
        if layout == "adapter":
            coll = "cm"
        nx, ny = _log(rng, 40, 7000), _log(rng, 40, 7000)
        # about 10 ms of work at most, and a whole run's worth of steps on a small grid
        most = int(6.0e8 / (nx * ny))
        steps = max(5, min(most, rng.randint(40, 200) if layout != "adapter" else rng.randint(20, 40)))
        return dict(kind="d2q9", layout=layout, nx=nx, ny=ny, coll=coll, storage=storage, steps=steps)
    if pick < 0.6:
        return dict(kind="cylinder", layout="cylinder", nx=_log(rng, 300, 3000), ny=_log(rng, 160, 900), coll=rng.choice(["bgk", "cm"]),
                    storage=rng.choice(["f32", "f16"]), steps=rng.randint(20, 80))
    if pick < 0.7:
        every = rng.randint(10, 50)
        return dict(kind="adjoint", layout="periodic", nx=_log(rng, 60, 900), ny=_log(rng, 60, 900), coll=rng.choice(["bgk", "mrt"]), storage="f32",
                    steps=rng.randint(40, 120), every=every)
    nx, ny, nz = _log(rng, 20, 300), _log(rng, 20, 220), _log(rng, 20, 220)
    steps = max(3, min(40, int(1.5e8 / (nx * ny * nz))))
    layout = rng.choice(["periodic", "periodic", "duct", "tunnel"])
    if layout == "tunnel":
        nx, ny, nz = max(nx, 48), max(ny, 40), max(nz, 40)
        return dict(kind="tunnel", layout="tunnel", nx=nx, ny=ny, nz=nz, coll=coll, storage=storage, steps=steps, markers=rng.choice([0, 128, 256]))
    return dict(kind="d3q27", layout=layout, nx=nx, ny=ny, nz=nz, coll=coll, storage=storage, steps=steps)


# ---- set-up of a case: the same numbers for the solver and for the 64-bit restatement -----------


def _omega(nu):
    return float(torch.tensor(1.0, dtype=torch.float32) / (3.0 * torch.tensor(nu, dtype=torch.float32) + 0.5))


def _rates2(case, om):
    if case["coll"] == "mrt":
        return (0.0, 1.1, 1.2, 0.0, 1.4, 0.0, 1.4, om, om)
    if case["coll"] == "cm":
        return (0.0, 0.0, 0.0, 1.0, om, om, 1.0, 1.0, 1.0)
    return (0.0, om, om, 0.0, om, 0.0, om, om, om)


def _setup2(case):
    """Config fields, flags [ny, nx] (numpy uint8 or None) of a D2Q9 case."""
    nx, ny, lay = case["nx"], case["ny"], case["layout"]
    nu = {"cavity": U_LID * min(nx, ny) / 1000.0, "cylinder": U_IN * ny / 8.0 / 100.0}.get(lay, NU)
    om = _omega(nu)
    kw = dict(nx=nx, ny=ny, collision=COLL[case["coll"]], omega=om, S=_rates2(case, om), storage=STORE[case["storage"]])
    flags = torch.zeros(ny, nx, dtype=torch.uint8)
    if lay == "periodic":
        kw.update(periodic_x=True, periodic_y=True)
        flags = None
    elif lay == "cavity":
        flags[0] = flags[-1] = A.BOUNCE_BACK
        flags[:, 0] = flags[:, -1] = A.BOUNCE_BACK
        flags[-1, 1:-1] = A.MOVING_WALL_BOUNCE_BACK
        kw.update(wall_u=(U_LID, 0.0), u_lid=U_LID)
    elif lay in ("channel", "adapter"):
        flags[0] = flags[-1] = A.BOUNCE_BACK
        kw.update(periodic_x=True, force=(float(torch.tensor(1e-6, dtype=torch.float32)), 0.0))
        if lay == "adapter":
            kw.update(adapter=A.LBM_OPTIMAL_ADAPTER)
    else:  # cylinder: velocity inlet, zero-gradient outlet, walls
        flags[:, 0] = A.ZOU_HE_LEFT
        flags[:, -1] = A.ZG_OUTFLOW
        flags[0] = flags[-1] = A.BOUNCE_BACK
        kw.update(u_lid=U_IN)
    return kw, flags


def _setup3(case):
    nx, ny, nz, lay = case["nx"], case["ny"], case["nz"], case["layout"]
    om = _omega(NU)
    S = [1.0] * 27
    S[4:9] = [om] * 5
    kw = dict(nx=nx, ny=ny, nz=nz, collision=COLL[case["coll"]], omega=om, S=tuple(S), storage=STORE[case["storage"]])
    flags = None
    if lay == "periodic":
        kw.update(periodic_x=True, periodic_y=True, periodic_z=True)
    else:
        flags = torch.zeros(nz, ny, nx, dtype=torch.uint8)
        flags[0] = flags[-1] = A.BOUNCE_BACK
        flags[:, 0] = flags[:, -1] = A.BOUNCE_BACK
        if lay == "duct":
            kw.update(periodic_x=True)
        else:
            flags[:, :, 0] = A.GUO_VELOCITY_INLET
            flags[:, :, -1] = A.GUO_PRESSURE_OUTLET
            kw.update(u_inlet=U_IN)
    return kw, flags


def _waves(gen, shape, modes, amp):
    """A smooth random field of zero mean on the grid: `modes` Fourier modes of low wave number."""
    axes = [torch.arange(n, device=DEV, dtype=torch.float64) * (2 * math.pi / n) for n in shape]
    out = torch.zeros(shape, device=DEV, dtype=torch.float64)
    for _ in range(modes):
        k = torch.randint(1, 4, (len(shape),), generator=gen).tolist()
        ph = (2 * math.pi * torch.rand(len(shape), generator=gen)).tolist()
        term = None
        for d, ax in enumerate(axes):
            v = torch.sin(k[d] * ax + ph[d]).reshape([-1 if e == d else 1 for e in range(len(shape))])
            term = v if term is None else term * v
        out += term * amp
    return out


def _initial(case, seed):
    """rho [...], u [..., D], float32 on the GPU: a smooth flow with a little noise; the plug
    flow of the inlet under it where there is one, at rest at the walls of a closed box."""
    gen = torch.Generator().manual_seed(seed)
    dim = 3 if "nz" in case else 2
    shape = (case["nz"], case["ny"], case["nx"]) if dim == 3 else (case["ny"], case["nx"])
    noise = torch.Generator(device=DEV).manual_seed(seed)
    rho = 1.0 + _waves(gen, shape, 3, 0.002)
    comps = []
    for d in range(dim):
        v = _waves(gen, shape, 4, 0.012 if case["layout"] in ("periodic", "cavity") else 0.004)
        v += 2e-4 * torch.randn(shape, device=DEV, dtype=torch.float64, generator=noise)
        if case["layout"] in ("cavity", "channel", "adapter", "duct"):
            for a, n in enumerate(shape):
                wrapped = case["layout"] != "cavity" and a == dim - 1
                if not wrapped:
                    e = torch.sin(math.pi * torch.arange(n, device=DEV, dtype=torch.float64) / (n - 1))
                    v = v * e.reshape([-1 if b == a else 1 for b in range(dim)])
        if d == 0 and case["layout"] in ("cylinder", "tunnel"):
            v = v + U_IN
        comps.append(v)
    return rho.float().contiguous(), torch.stack(comps, -1).float().contiguous()


def _markers(case, seed):
    """Marker positions and their arc length or area, numpy float32; None without a body."""
    gen = torch.Generator().manual_seed(seed + 77)
    off = (torch.rand(3, generator=gen, dtype=torch.float64) - 0.5).tolist()
    if case["kind"] == "cylinder":
        d = max(16.0, case["ny"] / 8.0)
        n = int(d * math.pi)
        t = torch.arange(n, dtype=torch.float64) * (2 * math.pi / n)
        xy = torch.stack([case["nx"] * 0.25 + off[0] + 0.5 * d * torch.cos(t), case["ny"] * 0.5 + off[1] + 0.5 * d * torch.sin(t)], -1)
        return xy.float().numpy(), torch.full((n,), math.pi * d / n).float().numpy()
    n = case.get("markers", 0)
    if not n:
        return None
    d = min(case["ny"], case["nz"]) / 6.0
    i = torch.arange(n, dtype=torch.float64) + 0.5
    z = 1.0 - 2.0 * i / n
    r, t = torch.sqrt(1.0 - z * z), i * (math.pi * (3.0 - math.sqrt(5.0)))
    p = 0.5 * d * torch.stack([r * torch.cos(t), r * torch.sin(t), z], -1)
    p += torch.tensor([case["nx"] * 0.4 + off[0], case["ny"] * 0.5 + off[1], case["nz"] * 0.5 + off[2]], dtype=torch.float64)
    return p.float().numpy(), torch.full((n,), math.pi * d * d / n).float().numpy()


def _force_field(case, seed):
    gen = torch.Generator().manual_seed(seed + 5)
    shape = (case["ny"], case["nx"])
    return torch.stack([_waves(gen, shape, 8, 1e-5) for _ in range(2)], -1).float().contiguous()


def _cotangent(case, seed):
    noise = torch.Generator(device=DEV).manual_seed(seed + 9)
    return torch.randn(case["ny"], case["nx"], 2, device=DEV, generator=noise)


# ---- the measured interface ---------------------------------------------------------------------


def prepare(case, seed):
    rho, u = _initial(case, seed)
    if case["kind"] == "adjoint":
        kw, _ = _setup2(case)
        sim = Simulation(Config(**kw), case["steps"], case["every"], rho0=rho)
        return dict(kind="adjoint", sim=sim, u=u.requires_grad_(True), force=_force_field(case, seed).requires_grad_(True),
                    cot=_cotangent(case, seed))
    three = "nz" in case
    kw, flags = _setup3(case) if three else _setup2(case)
    s = Solver3D(Config3D(**kw)) if three else Solver(Config(**kw))
    s.set_stream(torch.cuda.current_stream().cuda_stream)
    if flags is not None:
        s.set_flags(flags.numpy())
    m = _markers(case, seed) if case["kind"] in ("cylinder", "tunnel") else None
    if m is not None:
        s.ibm_set_markers(m[0], m[1], 3)
    return dict(kind="d3q27" if three else "d2q9", s=s, rho=rho, u=u, steps=case["steps"])


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    if state["kind"] == "adjoint":
        u_end = state["sim"](state["force"], state["u"])
        g_force, g_u0 = torch.autograd.grad(u_end, (state["force"], state["u"]), grad_outputs=state["cot"])
        return {"u": u_end.detach(), "g_force": g_force, "g_u0": g_u0}
    s, lib = state["s"], state["s"].lib
    macros, pops = (lib.lbm3d_get_macros, lib.lbm3d_get_pops) if state["kind"] == "d3q27" else (lib.lbm_get_macros, lib.lbm_get_pops)
    s.init_from_macros(state["rho"], state["u"])
    s.step(state["steps"])
    rho, u = torch.empty_like(state["rho"]), torch.empty_like(state["u"])
    f = torch.empty((27 if state["kind"] == "d3q27" else 9,) + tuple(rho.shape), device=rho.device)
    s._check(macros(s.h, _ptr(rho), _ptr(u), 1))
    s._check(pops(s.h, _ptr(f), 1))
    return {"rho": rho, "u": u, "f": f}


def work(case):
    n, dim = case["nx"] * case["ny"] * case.get("nz", 1), 3 if "nz" in case else 2
    fl = FLOPS["3d" if dim == 3 else "2d", case["coll"]] * n * case["steps"]
    if case["kind"] == "adjoint":  # u0, force and the cotangent in; u, two gradients out; backward as two forwards
        return {"bytes": 6 * 8 * n, "flops": 3 * fl}
    return {"bytes": 4 * n * (2 * (1 + dim) + (27 if dim == 3 else 9)), "flops": fl}


# ---- the same runs in plain torch, 64 bits ------------------------------------------------------

C2 = [(0, 0), (1, 0), (0, 1), (-1, 0), (0, -1), (1, 1), (-1, 1), (-1, -1), (1, -1)]
C3 = [(0, 0, 0), (1, 0, 0), (-1, 0, 0), (0, 1, 0), (0, -1, 0), (0, 0, 1), (0, 0, -1)]
C3 += [(1, 1, 0), (-1, 1, 0), (1, -1, 0), (-1, -1, 0), (1, 0, 1), (-1, 0, 1), (1, 0, -1), (-1, 0, -1)]
C3 += [(0, 1, 1), (0, -1, 1), (0, 1, -1), (0, -1, -1)]
C3 += [(x, y, z) for z in (1, -1) for y in (1, -1) for x in (1, -1)]


def _w(c):
    n = sum(abs(k) for k in c)
    return ([4 / 9, 1 / 9, 1 / 36] if len(c) == 2 else [8 / 27, 2 / 27, 1 / 54, 1 / 216])[n]


def _opp(C):
    return [C.index(tuple(-k for k in c)) for c in C]


def _feq(C, q, rho, u, usq):
    cu = 0.0
    for a, k in enumerate(C[q]):
        if k:
            cu = cu + k * u[a]
    return _w(C[q]) * rho * (1 + 3 * cu + 4.5 * cu * cu - 1.5 * usq)


def _guo(C, q, u, F, uF):
    cu = cF = 0.0
    for a, k in enumerate(C[q]):
        if k:
            cu, cF = cu + k * u[a], cF + k * F[a]
    return _w(C[q]) * (3 * (cF - uF) + 9 * cu * cF)


def _moments(C, f):
    rho = f[0].clone()
    for q in range(1, len(C)):
        rho = rho + f[q]
    j = []
    for a in range(len(C[0])):
        s = 0.0
        for q, c in enumerate(C):
            if c[a]:
                s = s + c[a] * f[q]
        j.append(s)
    return rho, j


def _mrt_basis():
    """The orthogonal D2Q9 moment basis: density, energy, its square, and per axis momentum and
    energy flux, then the two stresses."""
    rows = []
    for m in range(9):
        row = []
        for x, y in C2:
            s = x * x + y * y
            row.append([1, 3 * s - 4, 4 - 10.5 * s + 4.5 * s * s, x, (3 * s - 5) * x, y, (3 * s - 5) * y, x * x - y * y, x * y][m])
        rows.append(row)
    return torch.tensor(rows, dtype=torch.float64)


def _axis_inv(m0, m1, m2, u):
    """Values at c = -1, 0, 1 whose moments about u are m0, m1, m2."""
    r1 = m1 + u * m0
    r2 = m2 + 2 * u * m1 + u * u * m0
    return 0.5 * (r2 - r1), m0 - r2, 0.5 * (r2 + r1)


def _collide2(case, kw, f, rho, u, F, means):
    """In place on the list f of nine planes."""
    usq = u[0] * u[0] + u[1] * u[1]
    om, S = kw["omega"], kw["S"]
    S = [float(torch.tensor(s, dtype=torch.float32)) for s in S]
    forced = F is not None
    uF = u[0] * F[0] + u[1] * F[1] if forced else None
    if case["coll"] == "bgk":
        return [(1 - om) * f[q] + om * _feq(C2, q, rho, u, usq) + ((1 - 0.5 * om) * _guo(C2, q, u, F, uF) if forced else 0.0) for q in range(9)]
    if case["coll"] == "mrt":
        M = _mrt_basis()
        Mi = torch.linalg.inv(M)
        X = (Mi @ torch.diag(torch.tensor(S, dtype=torch.float64)) @ M).tolist()
        Y = (Mi @ torch.diag(1 - 0.5 * torch.tensor(S, dtype=torch.float64)) @ M).tolist()
        d = [f[q] - _feq(C2, q, rho, u, usq) for q in range(9)]
        g = [_guo(C2, q, u, F, uF) for q in range(9)] if forced else None
        out = []
        for q in range(9):
            v = f[q].clone()
            for k in range(9):
                if X[q][k]:
                    v -= X[q][k] * d[k]
                if forced:
                    v += Y[q][k] * g[k]
            out.append(v)
        return out
    # central moments about u: density, momentum, trace and difference of the second, xy, two
    # third and the fourth; relaxed towards those of a Maxwellian with the forcing beside them
    K = {}
    for a in range(3):
        for b in range(3):
            s = 0.0
            for q, (x, y) in enumerate(C2):
                s = s + (x - u[0]) ** a * (y - u[1]) ** b * f[q]
            K[a, b] = s
    k = [K[0, 0], K[1, 0], K[0, 1], K[2, 0] + K[0, 2], K[2, 0] - K[0, 2], K[1, 1], K[2, 1], K[1, 2], K[2, 2]]
    keq = [rho, 0.0, 0.0, 2 * rho / 3, 0.0, 0.0, 0.0, 0.0, rho / 9]
    Fx, Fy = F if forced else (0.0, 0.0)
    R = [0.0, Fx, Fy, 0.0, 0.0, 0.0, Fy / 3, Fx / 3, 0.0]
    rate = list(S)
    if means is not None:
        t = 0.0003 * rho / means[0] - 0.00775 * rho * torch.sqrt(usq) / means[1] + 0.00016 * _stress(f) / means[2] + 0.0087
        t = torch.clamp(torch.where(t > 0, t, torch.full_like(t, 0.005)), max=1.5)
        rate[6] = rate[7] = rate[8] = 1 / (3 * t + 0.5)
    d = [-rate[i] * (k[i] - keq[i]) + (1 - 0.5 * rate[i]) * R[i] for i in range(9)]
    z = torch.zeros_like(rho)
    D = {(0, 0): d[0], (1, 0): d[1], (0, 1): d[2], (2, 0): 0.5 * (d[3] + d[4]), (0, 2): 0.5 * (d[3] - d[4]), (1, 1): d[5],
         (2, 1): d[6], (1, 2): d[7], (2, 2): d[8]}
    col = [_axis_inv(D[a, 0] + z, D[a, 1] + z, D[a, 2] + z, u[1]) for a in range(3)]
    row = [_axis_inv(col[0][j], col[1][j], col[2][j], u[0]) for j in range(3)]
    return [f[q] + row[C2[q][1] + 1][C2[q][0] + 1] for q in range(9)]


def _stress(f):
    xx = f[1] + f[3] + f[5] + f[6] + f[7] + f[8]
    yy = f[2] + f[4] + f[5] + f[6] + f[7] + f[8]
    xy = f[5] - f[6] + f[7] - f[8]
    return torch.sqrt(xx * xx + 2 * xy * xy + yy * yy)


def _collide3(case, kw, f, rho, u, F):
    usq = u[0] * u[0] + u[1] * u[1] + u[2] * u[2]
    om = kw["omega"]
    forced = F is not None
    if case["coll"] == "bgk":
        uF = sum(u[a] * F[a] for a in range(3)) if forced else None
        return [(1 - om) * f[q] + om * _feq(C3, q, rho, u, usq) + ((1 - 0.5 * om) * _guo(C3, q, u, F, uF) if forced else 0.0) for q in range(27)]

    def second(a, b):
        s = 0.0
        for q, c in enumerate(C3):
            if c[a] * c[b]:
                s = s + c[a] * c[b] * f[q]
        return s

    xx, yy, zz, xy, xz, yz = second(0, 0), second(1, 1), second(2, 2), second(0, 1), second(0, 2), second(1, 2)
    w = 1 - om
    if case["coll"] == "mrt":  # unforced here: product equilibrium plus the relaxed deviatoric stresses
        d4, d5, d6 = w * (xy - rho * u[0] * u[1]), w * (xz - rho * u[0] * u[2]), w * (yz - rho * u[1] * u[2])
        d7, d8 = w * (xx - yy - rho * (u[0] ** 2 - u[1] ** 2)), w * (xx - zz - rho * (u[0] ** 2 - u[2] ** 2))
        t = (d7 + d8) / 3
        T = {(1, 1, 0): d4, (1, 0, 1): d5, (0, 1, 1): d6, (2, 0, 0): t, (0, 2, 0): t - d7, (0, 0, 2): t - d8}
        phi = [{0: 2 / 3 - v * v, 1: 0.5 * (1 / 3 + v * v + v), -1: 0.5 * (1 / 3 + v * v - v)} for v in u]
        inv = {-1: {1: -0.5, 2: 0.5}, 0: {0: 1.0, 2: -1.0}, 1: {1: 0.5, 2: 0.5}}  # value at c from moments 0, 1, 2
        out = []
        for c in C3:
            v = rho * phi[0][c[0]] * phi[1][c[1]] * phi[2][c[2]]
            for m, x in T.items():
                k = 1.0
                for a in range(3):
                    k *= inv[c[a]].get(m[a], 0.0)
                if k:
                    v = v + k * x
            out.append(v)
        return out
    j = [rho * u[a] - (0.5 * F[a] if forced else 0.0) for a in range(3)]

    def central(raw, a, b):
        return raw - u[a] * j[b] - u[b] * j[a] + rho * u[a] * u[b]

    kxx, kyy, kzz = central(xx, 0, 0), central(yy, 1, 1), central(zz, 2, 2)
    e = [1.0, 0.0, 1 / 3]
    zero = torch.zeros_like(rho)
    K = {}
    for a in range(3):
        for b in range(3):
            for c in range(3):
                v = zero + rho * (e[a] * e[b] * e[c])
                if forced:
                    v = v + 0.5 * F[0] * ((a == 1) * e[b] * e[c]) + 0.5 * F[1] * ((b == 1) * e[a] * e[c]) + 0.5 * F[2] * ((c == 1) * e[a] * e[b])
                K[a, b, c] = v
    K[1, 1, 0], K[1, 0, 1], K[0, 1, 1] = w * central(xy, 0, 1), w * central(xz, 0, 2), w * central(yz, 1, 2)
    t = (rho + w * (2 * kxx - kyy - kzz)) / 3
    K[2, 0, 0], K[0, 2, 0], K[0, 0, 2] = t, t - w * (kxx - kyy), t - w * (kxx - kzz)
    for a in range(3):
        for b in range(3):
            K[a, b, 0], K[a, b, 1], K[a, b, 2] = _axis_inv(K[a, b, 0], K[a, b, 1], K[a, b, 2], u[2])
    for a in range(3):
        for c in range(3):
            K[a, 0, c], K[a, 1, c], K[a, 2, c] = _axis_inv(K[a, 0, c], K[a, 1, c], K[a, 2, c], u[1])
    for b in range(3):
        for c in range(3):
            K[0, b, c], K[1, b, c], K[2, b, c] = _axis_inv(K[0, b, c], K[1, b, c], K[2, b, c], u[0])
    return [K[c[0] + 1, c[1] + 1, c[2] + 1] for c in C3]


def _edge(shape, periodic, c):
    """Slices of the nodes whose neighbour at -c lies outside the domain (one per axis that has any)."""
    found, dim = [], len(shape)
    for a, k in enumerate(c):
        if k and not periodic[a]:
            sl = [slice(None)] * dim
            sl[dim - 1 - a] = 0 if k > 0 else -1
            found.append(tuple(sl))
    return found


def _stream(C, f, old, periodic):
    dim, out = len(C[0]), []
    for q, c in enumerate(C):
        g = torch.roll(f[q], [c[a] for a in reversed(range(dim))], list(range(dim)))
        for sl in _edge(g.shape, periodic, c):
            g[sl] = old[q][sl]
        out.append(g)
    return out


def _bounce(C, g, flags, periodic, wall):
    """Every direction that leaves the domain returns as its opposite, in order of the directions."""
    opp = _opp(C)
    still, moving = flags == A.BOUNCE_BACK, flags == A.MOVING_WALL_BOUNCE_BACK
    both = still | moving
    for q in range(1, len(C)):
        away = tuple(-k for k in C[q])  # nodes whose neighbour at +c is outside
        mask = torch.zeros_like(both)
        for sl in _edge(both.shape, periodic, away):
            mask[sl] = both[sl]
        if not mask.any():
            continue
        v = g[q]
        if wall is not None:
            v = v - 6 * _w(C[q]) * sum(k * wu for k, wu in zip(C[q], wall)) * moving
        g[opp[q]] = torch.where(mask, v, g[opp[q]])


def _zou_he_left(g, mask, ux):
    r = (g[0] + g[2] + g[4] + 2 * (g[3] + g[6] + g[7])) / (1 - ux)
    g1 = g[3] + 2 / 3 * r * ux
    g5 = g[7] - 0.5 * (g[2] - g[4]) + r * ux / 6
    g8 = g[6] + 0.5 * (g[2] - g[4]) + r * ux / 6
    for q, v in ((1, g1), (5, g5), (8, g8)):
        g[q] = torch.where(mask, v, g[q])


def _guo_plane(g, snap, inlet):
    """Guo velocity inlet (x = 0) or pressure outlet (x = nx - 1) of the 3-D tunnel."""
    x, xn, sgn = (0, 1, 1) if inlet else (-1, -2, -1)
    own = [v[..., x] for v in g]
    near = [v[..., xn] for v in snap]
    known = 0.0
    for q, c in enumerate(C3):
        if c[0] * sgn < 0:
            known = known + 2 * own[q]
        elif c[0] == 0:
            known = known + own[q]
    if inlet:
        ui = float(torch.tensor(U_IN, dtype=torch.float32))
        ub = [torch.full_like(known, ui), torch.zeros_like(known), torch.zeros_like(known)]
        rb = known / (1 - ui)
    else:
        rb = torch.ones_like(known)
        tr = [sum(c[a] * own[q] for q, c in enumerate(C3) if c[0] >= 0 and c[a]) for a in (1, 2)]
        ub = [known - 1, tr[0], tr[1]]
    rf, jf = _moments(C3, near)
    uf = [v / rf for v in jf]
    sb, sf = sum(v * v for v in ub), sum(v * v for v in uf)
    for q, c in enumerate(C3):
        if c[0] * sgn > 0:
            g[q][..., x] = _feq(C3, q, rb, ub, sb) + (near[q] - _feq(C3, q, rf, uf, sf))


def _delta(r):
    a = r.abs()
    near = (3 - 2 * a + torch.sqrt(torch.clamp(1 + 4 * a - 4 * a * a, min=0))) / 8
    far = (5 - 2 * a - torch.sqrt(torch.clamp(-7 + 12 * a - 4 * a * a, min=0))) / 8
    return torch.where(a < 1, near, torch.where(a < 2, far, torch.zeros_like(a)))


def _body(markers, shape):
    """Node indices [n, 4^D] and kernel weights of every marker's stencil."""
    p = torch.as_tensor(markers[0], device=DEV).double()
    dim = p.shape[1]
    base = torch.floor(p).long()
    idx, wts = torch.zeros(p.shape[0], 1, dtype=torch.long, device=DEV), torch.ones(p.shape[0], 1, dtype=torch.float64, device=DEV)
    for a in reversed(range(dim)):
        at = base[:, a:a + 1] + torch.arange(-1, 3, device=DEV)
        k = _delta(p[:, a:a + 1] - at.double())
        n = shape[dim - 1 - a]
        idx = (idx[:, :, None] * n + at.clamp(0, n - 1)[:, None, :]).reshape(p.shape[0], -1)
        wts = (wts[:, :, None] * (k * ((at >= 0) & (at < n)))[:, None, :]).reshape(p.shape[0], -1)
    return idx, wts, torch.as_tensor(markers[1], device=DEV).double()


def _body_force(body, rho, u, iters=3):
    """Multi-direct forcing: drive the interpolated velocity at the markers to zero."""
    idx, wts, ds = body
    flat = [v.reshape(-1).clone() for v in u]
    r = rho.reshape(-1)
    total = [torch.zeros_like(r) for _ in u]
    rl = (wts * r[idx]).sum(1)
    for _ in range(iters):
        step = []
        for v in flat:
            fl = -2 * rl * (wts * v[idx]).sum(1)
            step.append(torch.zeros_like(r).index_add_(0, idx.reshape(-1), (wts * (fl * ds)[:, None]).reshape(-1)))
        for a, s in enumerate(step):
            flat[a] += s / (2 * r)
            total[a] += s
    return [t.reshape(rho.shape) for t in total]


def _advance(case, seed):
    three = "nz" in case
    C, kw = (C3 if three else C2), (_setup3 if three else _setup2)(case)[0]
    flags = (_setup3 if three else _setup2)(case)[1]
    flags = None if flags is None else flags.to(DEV)
    periodic = [kw.get("periodic_" + a, False) for a in "xyz"][: 3 if three else 2]
    rho, u = _initial(case, seed)
    rho, u = rho.double(), [v.double() for v in u.unbind(-1)]
    f = [_feq(C, q, rho, u, sum(v * v for v in u)) for q in range(len(C))]
    old = list(f)
    m = _markers(case, seed) if case["kind"] in ("cylinder", "tunnel") else None
    body = _body(m, rho.shape) if m is not None else None
    const = kw.get("force")
    wall = [float(torch.tensor(v, dtype=torch.float32)) for v in kw["wall_u"]] if "wall_u" in kw else None
    for _ in range(case["steps"]):
        g = _stream(C, f, old, periodic)
        old = f
        if flags is not None:
            snap = [v.clone() for v in g] if case["layout"] == "tunnel" else list(g)
            _bounce(C, g, flags, periodic, wall)
            if case["layout"] == "cylinder":
                _zou_he_left(g, flags == A.ZOU_HE_LEFT, float(torch.tensor(U_IN, dtype=torch.float32)))
                out = flags[:, -1] == A.ZG_OUTFLOW
                for q, c in enumerate(C):
                    if c[0] < 0:
                        v = g[q].clone()
                        v[:, -1] = torch.where(out, snap[q][:, -2], v[:, -1])
                        g[q] = v
            elif case["layout"] == "tunnel":
                _guo_plane(g, snap, True)
                _guo_plane(g, snap, False)
            del snap
        rho, j = _moments(C, g)
        F = None
        if const is not None:
            F = [torch.full_like(rho, const[0]), torch.full_like(rho, const[1])]
        if body is not None:
            F = _body_force(body, rho, [v / rho for v in j])
        u = [(v + 0.5 * F[a]) / rho if F is not None else v / rho for a, v in enumerate(j)]
        if three:
            f = _collide3(case, kw, g, rho, u, F)
        else:
            means = None
            if case["layout"] == "adapter":
                means = [rho.mean(), (rho * torch.sqrt(u[0] ** 2 + u[1] ** 2)).mean(), _stress(g).mean()]
            f = _collide2(case, kw, g, rho, u, F, means)
    return {"rho": rho, "u": torch.stack(u, -1), "f": torch.stack(f)}


def _adjoint(case, seed):
    kw, _ = _setup2(case)
    rho0, u0 = _initial(case, seed)
    rho0, u0 = rho0.double(), u0.double().requires_grad_(True)
    force = _force_field(case, seed).double().requires_grad_(True)
    cot = _cotangent(case, seed).double()

    def state(u):
        v = u.unbind(-1)
        usq = v[0] * v[0] + v[1] * v[1]
        return torch.stack([_feq(C2, q, rho0, v, usq) for q in range(9)])

    def post(f, F):
        g = _stream(C2, f.unbind(0), None, [True, True])
        rho, j = _moments(C2, g)
        return g, rho, [(v + 0.5 * F[..., a]) / rho for a, v in enumerate(j)]

    def step(f, F):
        g, rho, u = post(f, F)
        return torch.stack(_collide2(case, kw, g, rho, u, F.unbind(-1), None))

    def ending(f, F):
        return torch.stack(post(f, F)[2], -1)

    from torch.utils.checkpoint import checkpoint

    f = state(u0)
    for _ in range(case["steps"] - 1):
        f = checkpoint(step, f, force, use_reentrant=False)
    u = ending(f, force)
    g_force, g_u0 = torch.autograd.grad(u, (force, u0), grad_outputs=cot)
    return {"u": u.detach(), "g_force": g_force, "g_u0": g_u0}


def exact(case, seed):
    if case["kind"] == "adjoint":
        return _adjoint(case, seed)
    with torch.no_grad():
        return _advance(case, seed)
