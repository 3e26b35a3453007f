"""The work a user of the framework has it do, as cases that can be timed.

A case is a dict of plain values.  `prepare` makes what a program has in hand
before the call (host or device arrays, the handle of a grid it made once),
`run` is one call through the public entry points of t-flows_amd/tflows_gpu.py,
`exact` gives the same results in plain torch at 64 bits, and `work` counts
what one call cannot do without.

Kinds, and what each stands for in a flow solver:
  dropin     Solve_Native on host arrays, as an unchanged host code calls it
             every time step: small grids, where latency and launches count
  pressure   the device-resident pressure solve (two-phase density, Jacobi),
             in FP64 or with FP32 sweeps in FP64 refinement
  icc        the pressure solve with the reference's default preconditioner
  momentum_solve  a non-symmetric convection-diffusion system, textbook methods
  knn        an unstructured system with random cell numbering (points, rows of
             11 to 20 entries), in FP64 or the FP32 form
  batch      many independent pressure systems of mixed size in one call
  assemble   pressure matrix and right-hand side from face data on the device
  momentum   one velocity component's matrix, right-hand side and v_m from
             face data on the device
  fluxes     Rhie-Chow volume fluxes on the device
"""
import ctypes
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "t-flows_amd"))
import tflows_cases as cases  # noqa: E402
import tflows_gpu as gpu  # noqa: E402

BATCH_RHO_MAX = 1000.0
SCHEMES = ("central", "upwind", "quick", "minmod", "smart", "superbee")


def listed():
    return [
        # the smallest grid of the tests, NRMS test over the x range: all latency
        dict(name="dropin-12x10x8", kind="dropin", nx=12, ny=10, nz=8, rho=1.0, tol=1e-8, norm=False),
        # the ordinary small solve: 40^3 Poisson, the pressure solves' NRMS with norm
        dict(name="dropin-40", kind="dropin", nx=40, ny=40, nz=40, rho=1.0, tol=1e-8, norm=True),
        # an odd box, two-phase: every side odd, so rows do not pair up
        dict(name="pressure-131x117x97", kind="pressure", nx=131, ny=117, nz=97, rho=1000.0, tol=1e-8,
             fp32=False),
        # the largest: 200^3 two-phase 1:1000, FP64
        dict(name="pressure-200", kind="pressure", nx=200, ny=200, nz=200, rho=1000.0, tol=1e-8, fp32=False),
        # the FP32 form on a large box
        dict(name="pressure-fp32-160", kind="pressure", nx=160, ny=160, nz=160, rho=1000.0, tol=1e-8,
             fp32=True),
        # the default preconditioner
        dict(name="icc-100", kind="icc", nx=100, ny=100, nz=100, rho=1000.0, tol=1e-8),
        # a momentum-like system: few iterations, launches and set-up count
        dict(name="bicgstab-upwind-120", kind="momentum_solve", n=120, solver="bcgs", tol=1e-8),
        # an unstructured system, a million points
        dict(name="knn-100", kind="knn", nx=100, ny=100, nz=100, tol=1e-10, fp32=False),
        # 48 systems of sides 20..64 in the FP32 form
        dict(name="batch-48", kind="batch", count=48, smin=20, smax=64, tol=1e-8, fp32=True),
        # assembly on the device, faces in grid order
        dict(name="assemble-128", kind="assemble", nx=128, ny=128, nz=128, order="grid", singular=True),
        dict(name="momentum-110x100x90", kind="momentum", nx=110, ny=100, nz=90, order="grid",
             scheme="minmod", td="parabolic", component=2),
        dict(name="fluxes-128x112x96", kind="fluxes", nx=128, ny=112, nz=96, order="grid", choi=True, gu=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(float(lo) * (float(hi) / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["dropin", "dropin", "pressure", "pressure", "icc", "momentum_solve", "knn", "batch",
                       "assemble", "momentum", "fluxes"])
    if kind == "dropin":
        side = [_log_int(rng, 6, 48) for _ in range(3)]
        return dict(kind=kind, nx=side[0], ny=side[1], nz=side[2], rho=float(rng.choice([1, 10, 1000])),
                    tol=rng.choice([1e-8, 1e-10]), norm=rng.random() < 0.5)
    if kind == "pressure":
        side = [_log_int(rng, 48, 160) for _ in range(3)]
        return dict(kind=kind, nx=side[0], ny=side[1], nz=side[2], rho=float(rng.choice([1, 100, 1000])),
                    tol=rng.choice([1e-8, 1e-10]), fp32=rng.random() < 0.4)
    if kind == "icc":
        side = [_log_int(rng, 16, 110) for _ in range(3)]
        return dict(kind=kind, nx=side[0], ny=side[1], nz=side[2], rho=float(rng.choice([1, 1000])),
                    tol=rng.choice([1e-8, 1e-10]))
    if kind == "momentum_solve":
        return dict(kind=kind, n=_log_int(rng, 16, 120), solver=rng.choice(["bcgs", "cgs"]),
                    tol=rng.choice([1e-8, 1e-10]))
    if kind == "knn":
        side = [_log_int(rng, 20, 100) for _ in range(3)]
        return dict(kind=kind, nx=side[0], ny=side[1], nz=side[2], tol=rng.choice([1e-8, 1e-10]),
                    fp32=rng.random() < 0.4)
    if kind == "batch":
        smin = rng.randint(8, 24)
        return dict(kind=kind, count=rng.randint(8, 48), smin=smin, smax=smin + rng.randint(8, 36),
                    tol=rng.choice([1e-8, 1e-10]), fp32=rng.random() < 0.6)
    side = [_log_int(rng, 12, 120) for _ in range(3)]
    case = dict(kind=kind, nx=side[0], ny=side[1], nz=side[2],
                order=rng.choice(["grid", "grid", "boundary_first", "shuffled"]))
    if kind == "assemble":
        return dict(case, singular=rng.random() < 0.5)
    if kind == "momentum":
        return dict(case, scheme=rng.choice(SCHEMES), td=rng.choice(["linear", "parabolic"]),
                    component=rng.randint(1, 3))
    return dict(case, choi=rng.random() < 0.6, gu=rng.random() < 0.5)


# ---- inputs ----------------------------------------------------------------

class _OnDevice:
    """A torch tensor as a device operand of the library."""

    def __init__(self, a, dtype=torch.float64):
        self.t = torch.as_tensor(a, dtype=dtype).to("cuda")
        self.ptr = ctypes.c_void_p(self.t.data_ptr())


def _matrix(case, seed):
    kind = case["kind"]
    if kind in ("dropin", "pressure", "icc"):
        return cases.hex_pressure(case["nx"], case["ny"], case["nz"], rho_out=case["rho"], seed=seed)
    if kind == "momentum_solve":
        return cases.upwind(case["n"], seed=seed)
    return cases.knn(case["nx"], case["ny"], case["nz"], seed=seed)


def _systems(case, seed):
    # the sizes are the batch's; the densities, interfaces and right-hand sides the seed's
    sides, _ = cases.batch_params(case["count"], case["smin"], case["smax"], BATCH_RHO_MAX)
    _, ratios = cases.batch_params(case["count"], case["smin"], case["smax"], BATCH_RHO_MAX, seed=seed)
    return [cases.hex_pressure(int(n), rho_out=float(q), seed=seed + 7 * k)
            for k, (n, q) in enumerate(zip(sides, ratios))]


def _faces(case, seed):
    """Face data: internal faces in grid order and then the boundary faces;
    the boundary regions first, side by side; or a random order."""
    order = case["order"]
    return cases.hex_faces(case["nx"], case["ny"], case["nz"], seed=seed, shuffle=order == "shuffled",
                           ambient=order == "boundary_first")


def _momentum_fields(case, f, seed):
    return cases.momentum_fields(f, seed=seed)


def _options(case):
    kind = case["kind"]
    relres = kind not in ("dropin",)
    return gpu.Options(precision=gpu.FP32_IR if case.get("fp32") else gpu.FP64,
                       criterion=gpu.CRIT_RELRES if relres else gpu.CRIT_NRMS)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": dict(case), "opt": _options(case)}
    if kind in ("dropin", "pressure", "icc", "momentum_solve", "knn"):
        m = _matrix(case, seed)
        s["nat"] = gpu.Native(m.row, m.col, m.dia)
        s["miter"] = 20 * max(1000, int(m.n ** (1.0 / 3.0)))
        if kind == "dropin":
            s.update(val=m.val, b=m.b, x0=np.zeros(m.n))
        else:
            s.update(val=_OnDevice(m.val), b=_OnDevice(m.b), x=_OnDevice(np.zeros(m.n)))
    elif kind == "batch":
        ms = _systems(case, seed)
        s["batch"] = gpu.Batch([(m.row, m.col, m.dia) for m in ms])
        s["x"] = _OnDevice(np.zeros(sum(m.n for m in ms)))
        s["val"] = _OnDevice(np.concatenate([m.val for m in ms]))
        s["b"] = _OnDevice(np.concatenate([m.b for m in ms]))
    else:
        f = _faces(case, seed)
        s["nat"] = gpu.Native(f.row, f.col, f.dia)
        s["faces"] = gpu.Faces(s["nat"], f.c1, f.c2, f.pos, f.diag_bc, f.b_region)
        if kind == "assemble":
            s.update({k: _OnDevice(getattr(f, k)) for k in ("fc", "fw", "vm", "vflux")})
            s["n_bnd"] = f.n_bnd
            s["pp"] = _OnDevice(f.pp) if f.pp is not None else None
        elif kind == "momentum":
            s["fields"] = gpu.Momentum(_momentum_fields(case, f, seed), component=case["component"],
                                       adv=case["scheme"], blend_matrix=True, td=case["td"])
            s["v_m"] = _OnDevice(np.zeros(f.n))
        else:
            rf = cases.rhie_chow_fields(f, case["nx"], case["ny"], case["nz"], seed=seed)
            s["fields"] = gpu.RhieChow(rf, choi=case["choi"], gu=case["gu"])
            s["flux"] = _OnDevice(f.vflux)
        if kind != "fluxes":
            s["val"], s["b"] = _OnDevice(np.zeros(len(f.col))), _OnDevice(np.zeros(f.n))
    torch.cuda.synchronize()
    return s


# ---- one call ----------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "dropin":
        x = s["x0"].copy()
        niter, fin = s["nat"].solve_native("cg", "jacobi", s["val"], x, s["b"], s["miter"], case["tol"],
                                           norm=1.0 if case["norm"] else None)
        return {"x": x, "niter": niter, "fin_res": fin}
    if kind in ("pressure", "icc", "momentum_solve", "knn", "batch"):
        s["x"].t.zero_()                            # the initial guess; the library has streams of its own
        torch.cuda.current_stream().synchronize()
        if kind == "batch":
            niter, fin, _ = s["batch"].solve("cg", "jacobi", s["val"], s["x"], s["b"], 20000, case["tol"],
                                             options=s["opt"], device=True)
        else:
            solver = case["solver"] if kind == "momentum_solve" else "cg"
            prec = "icc" if kind == "icc" else "jacobi"
            niter, fin = s["nat"].solve_native_device(solver, prec, s["val"], s["x"], s["b"], s["miter"],
                                                      case["tol"], options=s["opt"])
        return {"x": s["x"].t, "niter": niter, "fin_res": fin}
    if kind == "assemble":
        s["faces"].assemble(s["fc"], s["fw"], s["vm"], s["vflux"], s["val"], s["b"],
                            singular=case["singular"], dpp=s["pp"], n_bnd=s["n_bnd"])
        return {"val": s["val"].t, "b": s["b"].t}
    if kind == "momentum":
        s["faces"].momentum(s["fields"], s["val"], s["b"], s["v_m"])
        return {"val": s["val"].t, "b": s["b"].t, "v_m": s["v_m"].t}
    s["faces"].rhie_chow(s["fields"], s["flux"])
    return {"flux": s["flux"].t}


# ---- the same in plain torch at 64 bits ----------------------------------------

def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _t(a):
    return torch.as_tensor(np.ascontiguousarray(a)).to(_device())


def _csr(m):
    return torch.sparse_csr_tensor(_t(m.row.astype(np.int64) - 1), _t(m.col.astype(np.int64) - 1), _t(m.val),
                                   size=(m.n, m.n))


def _cg(m, tol, most):
    A, b, d = _csr(m), _t(m.b), _t(m.val[m.dia.astype(np.int64) - 1])
    x = torch.zeros_like(b)
    r, p, rho = b.clone(), torch.zeros_like(b), torch.ones((), dtype=b.dtype, device=b.device)
    stop = tol * float(b.norm())
    for k in range(most):
        z = r / d
        new = r @ z
        p = z + (new / rho) * p if k else z
        rho = new
        q = A @ p
        alpha = rho / (p @ q)
        x += alpha * p
        r -= alpha * q
        if k % 16 == 15 and float(r.norm()) < stop:
            break
    return x


def _bicgstab(m, tol, most):
    A, b, d = _csr(m), _t(m.b), _t(m.val[m.dia.astype(np.int64) - 1])
    x = torch.zeros_like(b)
    r, rt = b.clone(), b.clone()
    p, v = torch.zeros_like(b), torch.zeros_like(b)
    rho = alpha = omega = 1.0
    for _ in range(most):
        new = float(rt @ r)
        p = r + (new / rho) * (alpha / omega) * (p - omega * v)
        rho = new
        y = p / d
        v = A @ y
        alpha = rho / float(rt @ v)
        s = r - alpha * v
        z = s / d
        t = A @ z
        omega = float(t @ s) / float(t @ t)
        x += alpha * y + omega * z
        r = s - omega * t
        if float(r.norm()) < tol * float(b.norm()):
            break
    return x


def _scatter(n, index, values):
    return torch.zeros(n, dtype=torch.float64, device=values.device).index_add_(0, index, values)


def _cells(f):
    """Faces' cells as indices of arrays laid out (-n_bnd:n), and which faces are internal."""
    nb = f.n_bnd
    c1, c2 = _t(f.c1.astype(np.int64)), _t(f.c2.astype(np.int64))
    return nb, c1 - 1, c1 + nb, c2 + nb, c2 > 0


def _exact_assemble(case, f):
    n = f.n
    nb, own, _, e2, inner = _cells(f)
    c2 = torch.where(inner, _t(f.c2.astype(np.int64)) - 1, 0)
    fc, fw, vm, flux = _t(f.fc), _t(f.fw), _t(f.vm), _t(f.vflux)
    a12 = torch.where(inner, fc * (fw * vm[own] + (1.0 - fw) * vm[c2]), 0.0)
    at_bc = ~inner & (_t(f.diag_bc) > 0)
    diag = _scatter(n, own, a12 + torch.where(at_bc, fc * vm[own], 0.0)) + _scatter(n, c2[inner], a12[inner])
    b = _scatter(n, own, -flux) + _scatter(n, c2[inner], flux[inner])
    for region in range(1, 7):                       # regions in ascending order
        at = ~inner & (_t(f.region.astype(np.int64)) == region)
        if f.pp is not None:
            amb = at & (_t(f.b_region) == 2)
            b[own[amb]] = (fc * vm[own])[amb] * _t(f.pp)[e2[amb]]
        b[own[at & (_t(f.b_region) == 1)]] = 0.0
    if case["singular"]:
        diag = diag * (1.0 + 1.0e-6)
    val = torch.zeros(len(f.col), dtype=torch.float64, device=diag.device)
    pos = _t(f.pos.astype(np.int64)).reshape(-1, 2) - 1
    val[pos[inner, 0]] = -a12[inner]
    val[pos[inner, 1]] = -a12[inner]
    val[_t(f.dia.astype(np.int64)) - 1] = diag
    return {"val": val, "b": b}


def _exact_momentum(case, f, mf, dt=1e-2, urf=0.7, p_drop=0.5):
    n = f.n
    nb, own, e1, e2, inner = _cells(f)
    oth = e2[inner] - nb - 1
    phi, rho = _t(mf.phi_n), _t(mf.density)
    F, fi, fw = _t(mf.v_flux), _t(mf.f), _t(mf.fw)
    g = [_t(mf.gx), _t(mf.gy), _t(mf.gz)]
    s = [_t(mf.sx), _t(mf.sy), _t(mf.sz)]
    d = [_t(mf.dx), _t(mf.dy), _t(mf.dz)]
    scheme = case["scheme"]
    up = torch.where(F > 0, e1, e2)
    down = torch.where(F > 0, e2, e1)
    if scheme == "central":
        phif = fi * phi[e1] + (1.0 - fi) * phi[e2]
    elif scheme == "upwind":
        phif = phi[up]
    else:
        fj = torch.where(F > 0, 1.0 - fi, fi)
        sgn = torch.where(F > 0, 1.0, -1.0)
        gd = sum(g[k][up] * d[k] for k in range(3))
        star = phi[down] - 2.0 * sgn * gd
        mn, mx = phi.clone(), phi.clone()
        for a, b in ((e1, e2), (e2, e1)):
            mn.scatter_reduce_(0, a, phi[b], "amin")
            mx.scatter_reduce_(0, a, phi[b], "amax")
        phi_u = torch.maximum(mn[up], torch.minimum(star, mx[up]))
        den = phi[down] - phi[up]
        den = torch.where(den.abs() < 1e-15, den + torch.copysign(torch.full_like(den, 1e-15), den), den)
        rj = (phi[up] - phi_u) / den
        gdn, gup = 0.5 * fj * (1.0 + fj), 0.5 * fj * (1.0 - fj)
        if scheme == "quick":
            psi = gdn + gup * rj
        elif scheme == "minmod":
            psi = fj * rj.clamp(0.0, 1.0)
        elif scheme == "smart":
            psi = torch.minimum(2.0 * rj, gdn + gup * rj).clamp(max=1.0).clamp(min=0.0)
        else:
            psi = 0.5 * torch.maximum((2.0 * rj).clamp(max=1.0).clamp(min=0.0), rj.clamp(max=2.0))
        phif = phi[up] + psi * sgn * (phi[e2] - phi[e1])
    carried = F * phif - F * torch.where(F < 0, phi[e2], phi[e1])     # explicit minus implicit upwind
    rho_c = rho[nb + 1:]
    b = rho_c * (_scatter(n, oth, carried[inner]) - _scatter(n, own, carried))
    i = case["component"] - 1
    at = lambda a: fw * a[e1] + (1.0 - fw) * a[e2]  # noqa: E731
    ui, uj, uk = at(g[i]), at(g[(i + 1) % 3]), at(g[(i + 2) % 3])
    si, sj, sk = s[i], s[(i + 1) % 3], s[(i + 2) % 3]
    di, dj, dk = d[i], d[(i + 1) % 3], d[(i + 2) % 3]
    vis, fc, stress = _t(mf.vis_eff), _t(mf.fc), _t(mf.f_stress)
    cross = vis * ((ui + ui) * si + (uj + at(_t(mf.uj_i))) * sj + (uk + at(_t(mf.uk_i))) * sk)
    cross = cross - (ui * di + uj * dj + uk * dk) * vis * fc
    b = b + _scatter(n, own, cross) - _scatter(n, oth, cross[inner])
    b = b + rho_c * (_scatter(n, own, stress) - _scatter(n, oth, stress[inner]))
    m12 = vis * fc - F.clamp(max=0.0) * rho[e1]
    m21 = vis * fc + F.clamp(min=0.0) * rho[e2]
    wall = ~inner & (_t(mf.wall) > 0)
    diag = _scatter(n, own, torch.where(inner | wall, m12, 0.0)) + _scatter(n, oth, m21[inner])
    b = b + _scatter(n, own, torch.where(wall, m12 * phi[e2], 0.0))
    vol, o, oo = _t(mf.vol), _t(mf.phi_o), _t(mf.phi_oo)
    a0 = rho_c * vol / dt
    if case["td"] == "linear":
        diag, b = diag + a0, b + a0 * o
    else:
        diag, b = diag + 1.5 * a0, b + 2.0 * a0 * o - 0.5 * a0 * oo
    b = b + (p_drop + _t(mf.cell_f) - _t(mf.p_i)) * vol
    v_m = vol / diag
    diag = diag / urf
    b = b + diag * (1.0 - urf) * phi[nb + 1:]
    val = torch.zeros(len(f.col), dtype=torch.float64, device=diag.device)
    pos = _t(f.pos.astype(np.int64)).reshape(-1, 2) - 1
    val[pos[inner, 0]] = -m12[inner]
    val[pos[inner, 1]] = -m21[inner]
    val[_t(f.dia.astype(np.int64)) - 1] = diag
    return {"val": val, "b": b, "v_m": v_m}


def _exact_fluxes(case, f, rf, dt=1e-2):
    inner = _t(f.c2) > 0
    c1 = _t(f.c1.astype(np.int64))[inner] - 1
    c2 = _t(f.c2.astype(np.int64))[inner] - 1
    face = lambda k: _t(getattr(rf, k))[inner]  # noqa: E731
    fs, vm, p = face("f"), _t(rf.v_m), _t(rf.p)
    at = lambda a: fs * a[c1] + (1.0 - fs) * a[c2]  # noqa: E731
    vel = [_t(rf.u), _t(rf.v), _t(rf.w)]
    tm = vm * _t(rf.density) / dt
    if case["choi"]:                                  # w_o = 1, w_oo = 0: backward Euler
        vel = [a - _t(o) * tm for a, o in zip(vel, (rf.u_o, rf.v_o, rf.w_o_))]
    if case["gu"]:
        vel = [a - vm * _t(c) for a, c in zip(vel, (rf.cell_fx, rf.cell_fy, rf.cell_fz))]
    area = [face("sx"), face("sy"), face("sz")]
    fl = sum(at(a) * s for a, s in zip(vel, area))
    fl = fl + face("fc") * at(vm) * (p[c1] - p[c2])
    fl = fl + face("fc") * sum(at(_t(g) * vm) * face(d)
                               for g, d in ((rf.px, "dx"), (rf.py, "dy"), (rf.pz, "dz")))
    if case["choi"]:
        fl = fl + at(tm) * face("flux_o")
    if case["gu"]:
        fl = fl + at(vm) * sum(face(k) * s for k, s in zip(("face_fx", "face_fy", "face_fz"), area))
    out = _t(f.vflux).clone()                         # boundary faces keep what they held
    out[inner] = fl
    return {"flux": out}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("dropin", "pressure", "icc", "knn"):
        m = _matrix(case, seed)
        return {"x": _cg(m, 1e-12, 8000), "niter": None, "fin_res": None}
    if kind == "momentum_solve":
        return {"x": _bicgstab(_matrix(case, seed), 1e-13, 400), "niter": None, "fin_res": None}
    if kind == "batch":
        return {"x": torch.cat([_cg(m, 1e-12, 4000) for m in _systems(case, seed)]), "niter": None,
                "fin_res": None}
    f = _faces(case, seed)
    if kind == "assemble":
        return _exact_assemble(case, f)
    if kind == "momentum":
        return _exact_momentum(case, f, _momentum_fields(case, f, seed))
    return _exact_fluxes(case, f, cases.rhie_chow_fields(f, case["nx"], case["ny"], case["nz"], seed=seed))


# ---- what one call cannot do without --------------------------------------------

def work(case):
    """Inputs read once and outputs written once; for a solve also the
    operations of its iterations, whose number is about that of these systems
    at 1e-8 per cell along the longest side."""
    kind = case["kind"]
    if kind == "batch":
        side = 0.5 * (case["smin"] + case["smax"])
        n = case["count"] * side ** 3
        return {"bytes": 8.0 * (7 * n + 3 * n), "flops": 12.0 * side * (14 * n + 12 * n)}
    if kind == "momentum_solve":
        n = float(case["n"]) ** 3
        return {"bytes": 8.0 * 10 * n, "flops": 20.0 * (28 * n + 24 * n)}
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = float(nx) * ny * nz
    if kind in ("dropin", "pressure", "icc", "knn"):
        per_row = 16.0 if kind == "knn" else 7.0
        its = {"icc": 4.0, "knn": 10.0}.get(kind, 12.0 if case.get("rho", 1.0) > 1.0 else 9.0) * max(nx, ny, nz)
        each = 2 * per_row * n + 12 * n + (28 * n if kind == "icc" else 0)
        return {"bytes": 8.0 * (per_row * n + 3 * n), "flops": its * each}
    nnz = 7.0 * n
    nf = 3.0 * n
    if kind == "assemble":
        return {"bytes": 8.0 * (3 * nf + n + nnz + n), "flops": 8.0 * nf + 8 * n}
    if kind == "momentum":
        return {"bytes": 8.0 * (12 * nf + 13 * n + nnz + 2 * n), "flops": 100.0 * nf + 30 * n}
    per_face = 8 + (2 if case["choi"] else 0) + (3 if case["gu"] else 0) + 1
    per_cell = 8 + (7 if case["choi"] else 0) + (3 if case["gu"] else 0)
    return {"bytes": 8.0 * (per_face * nf + per_cell * n), "flops": 60.0 * nf}
