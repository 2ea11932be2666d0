"""Performance cases of libt3x: the calls a user of the library makes, over the
range of sizes, forms and domains it is made for.

Kinds of case (field "kind"):
  run      Problem.run: whole design iterations of TOP3D_XL (the solid solve,
           then nLoop iterations), GLOBAL or LOCAL; returns the densities and
           histories a user reads.
  solve    one finite-element analysis of a given design: set_modulus,
           assemble, pcg, compliance on host arrays.
  matvec   apply_K on a host vector: the operator inside a user's own solver.
  update   one design update of a user's own loop: PDE filter of the
           sensitivities, then the OC bisection, on host arrays.
  oc       oc_noalloc on device arrays: the design update of a loop that keeps
           its arrays on the GPU.
  serve    a batch of whole optimisations through the serving engine.

Forms (field "form"): "fp64" is the library's default (the reference's
arithmetic), "mixed" the precision form that bench.py runs.  Sizes are
(ny, nx, nz) voxels.  The load on the cantilever's free face has a direction
and a magnitude drawn per seed, as the serving workload's requests have.
"""
import functools
import math

import numpy as np
import torch

import top3d_xl_amd as t3x
from top3d_xl_amd import irregular

R_MIN = math.sqrt(3.0)
MIXED = dict(precision=2, vcycle=1, omega=0.4, coarsestControl=0)
E0, EMIN, NU, PENAL = 1.0, 1e-6, 0.3, 3.0


def _run(name, shape, form, mode="GLOBAL", V0=0.12, rHat=0.0, nLoop=1, domain="cuboid"):
    ny, nx, nz = shape
    return dict(name=name, kind="run", ny=ny, nx=nx, nz=nz, form=form, mode=mode, V0=V0, rHat=rHat, nLoop=nLoop,
                domain=domain)


def listed():
    return [
        # the smallest model the tests optimise whole: launches and waits only
        _run("run_12x24x12_fp64", (12, 24, 12), "fp64"),
        # the reference's default cuboid, GLOBAL and porous infill (LOCAL); 50 is padded to 56
        _run("run_50x100x50_fp64", (50, 100, 50), "fp64", nLoop=2),
        _run("run_50x100x50_local", (50, 100, 50), "fp64", mode="LOCAL", V0=0.5, rHat=6.0, nLoop=2),
        # an ordinary large FP64 model (the serving workload's 128)
        _run("run_128x256x128_fp64", (128, 256, 128), "fp64"),
        # the headline cuboid in the precision form: 101M DOFs, the largest call
        _run("run_256x512x256_mixed", (256, 512, 256), "mixed"),
        # a voxel model with void space (a third of its box) and explicit supports
        _run("run_irregular_128x256x128_mixed", (128, 256, 128), "mixed", V0=0.4, domain="irregular"),
        # several small requests at once on one GPU
        dict(name="serve_32_48_64", kind="serve", sizes="32,64,48,32,48,32", nLoop=1, active=4, form="mixed"),
        # a single analysis of a given design, ragged small FP64 and ordinary mixed
        dict(name="solve_45x91x37_fp64", kind="solve", ny=45, nx=91, nz=37, form="fp64"),
        dict(name="solve_96x192x96_mixed", kind="solve", ny=96, nx=192, nz=96, form="mixed"),
        # the operator alone, ragged
        dict(name="matvec_61x121x83", kind="matvec", ny=61, nx=121, nz=83, form="fp64"),
        # filter and OC of a user's own loop
        dict(name="update_100x200x100", kind="update", ny=100, nx=200, nz=100, rMin=R_MIN, V0=0.2, form="fp64"),
        # OC on device arrays at the headline size
        dict(name="oc_device_33.5M", kind="oc", n=256 * 512 * 256, V0=0.12),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _shape(rng, lo, hi):
    s = _log(rng, lo, hi)
    return tuple(max(8, int(round(s * f * rng.uniform(0.85, 1.15)))) for f in (1.0, 2.0, 1.0))


def draw(rng):
    kind = rng.choice(["run", "run", "run", "solve", "solve", "matvec", "update", "oc", "serve"])
    form = rng.choice(["fp64", "mixed"])
    if kind == "run":
        domain = rng.choice(["cuboid", "cuboid", "irregular"])
        mode = "GLOBAL" if domain == "irregular" else rng.choice(["GLOBAL", "GLOBAL", "LOCAL"])
        ny, nx, nz = _shape(rng, 32 if domain == "irregular" else 10, 96)
        glob = mode == "GLOBAL"
        return dict(kind=kind, ny=ny, nx=nx, nz=nz, form=form, mode=mode, domain=domain,
                    V0=round(rng.uniform(0.08, 0.4) if glob else rng.uniform(0.4, 0.6), 3),
                    rHat=0.0 if glob else float(rng.randint(4, 8)), nLoop=1)
    if kind == "serve":
        return dict(kind=kind, sizes=",".join(str(rng.choice([32, 48, 64])) for _ in range(rng.randint(3, 8))),
                    nLoop=1, active=rng.randint(2, 4), form=form)
    if kind == "oc":
        return dict(kind=kind, n=int(_log(rng, 2e3, 2e7)), V0=round(rng.uniform(0.08, 0.4), 3))
    ny, nx, nz = _shape(rng, 10, 100)
    c = dict(kind=kind, ny=ny, nx=nx, nz=nz, form=form if kind == "solve" else "fp64")
    if kind == "update":
        c.update(rMin=round(rng.uniform(1.5, 6.0), 3), V0=round(rng.uniform(0.08, 0.4), 3))
    return c


# ------------------------------------------------------------------- inputs
def _params(case):
    return MIXED if case["form"] == "mixed" else {}


def _load(rng):
    d = rng.standard_normal(3)
    return d / np.linalg.norm(d) * rng.uniform(0.5, 2.0)


def _cantilever(ny, nx, nz, force):
    """The built-in cuboid's supports (the face x = 0) and load patch (the lower
    sixth of the opposite face) with the given total force."""
    jy = np.arange(ny + 1)
    fix = (jy[None, :] + (ny + 1) * (nx + 1) * np.arange(nz + 1)[:, None]).reshape(-1)
    top = int(math.floor(nz / 6.0 + 1.0 + 0.5))
    load = (jy[None, :] + (ny + 1) * (nx + (nx + 1) * np.arange(top)[:, None])).reshape(-1)
    return (fix, np.ones((fix.size, 3), np.uint8)), (load, np.tile(force / load.size, (load.size, 1)))


@functools.lru_cache(maxsize=4)
def _irregular(ny, nx, nz):
    return irregular.generate(0, (ny, nx, nz))


def _problem(case, rng):
    ny, nx, nz = case["ny"], case["nx"], case["nz"]
    force = _load(rng)
    if case.get("domain") == "irregular":
        m = _irregular(ny, nx, nz)
        n = len(m["load_nodes"])
        return t3x.Problem(m["voxels"], (m["fix_nodes"], m["fix_state"]),
                           (m["load_nodes"], np.tile(force / n, (n, 1))), **_params(case))
    fix, load = _cantilever(ny, nx, nz, force)
    return t3x.Problem(np.ones((ny, nx, nz), bool), fix, load, **_params(case))


def _density(shape, rng):
    """A design part-way through an optimisation: a smooth field pushed towards
    0 and 1, in the compact cell order (y fastest)."""
    ny, nx, nz = shape
    y, x, z = np.arange(ny)[None, None, :], np.arange(nx)[None, :, None], np.arange(nz)[:, None, None]
    f = np.zeros((nz, nx, ny))
    for _ in range(6):
        k = rng.uniform(0.03, 0.25, 3)
        p = rng.uniform(0, 2 * np.pi, 3)
        f += np.sin(k[0] * y + p[0]) * np.sin(k[1] * x + p[1]) * np.sin(k[2] * z + p[2])
    return np.clip(0.35 + 0.45 * f, 0.05, 1.0).reshape(-1)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "run":
        return dict(kind=kind, p=_problem(case, rng),
                    args=(case["mode"], case["V0"], case["nLoop"], R_MIN, case["rHat"]))
    if kind == "serve":
        reqs = []
        for tag, s in enumerate(int(v) for v in case["sizes"].split(",")):
            f = _load(rng)
            glob = rng.random() < 0.7
            reqs.append(dict(tag=tag, nely=s, nelx=2 * s, nelz=s, mode="GLOBAL" if glob else "LOCAL",
                             V0=float(rng.uniform(0.08, 0.3) if glob else rng.uniform(0.4, 0.6)), nLoop=case["nLoop"],
                             rMin=R_MIN, rHat=0.0 if glob else float(rng.integers(4, 9)),
                             load_dir=tuple(f / np.linalg.norm(f)), load_mag=float(np.linalg.norm(f))))
        return dict(kind=kind, reqs=reqs,
                    server=t3x.Server(max_active=case["active"], mem_budget=8 << 30, **_params(case)))
    if kind == "oc":
        g = torch.Generator(device="cuda").manual_seed(int(seed))
        n = case["n"]
        x = torch.rand(n, generator=g, device="cuda", dtype=torch.float64) * 0.9 * case["V0"] + 0.05
        dc = -(0.01 + torch.rand(n, generator=g, device="cuda", dtype=torch.float64)) * 3 * x * x
        return dict(kind=kind, n=n, V0=case["V0"], x0=x, x=x.clone(), xPhys=x.clone(), dc=dc)
    p = _problem(case, rng)
    x = _density((case["ny"], case["nx"], case["nz"]), rng)
    if kind == "update":
        p.filter_setup(0, case["rMin"])
        dc = -np.exp(rng.normal(-2.0, 1.0, x.size)) * 3 * x * x
        return dict(kind=kind, p=p, x=x, xdc=x * dc, V0=case["V0"])
    E = EMIN + x ** PENAL * (E0 - EMIN)
    if kind == "solve":
        return dict(kind=kind, p=p, E=E, F=p.load_vector())
    p.set_modulus(E)
    return dict(kind=kind, p=p, u=rng.standard_normal(3 * p.nN))


def run(s):
    kind = s["kind"]
    if kind == "run":
        r = s["p"].run(*s["args"])
        # (without the wall-clock times; consHist is volHist - V0 in GLOBAL mode: at a met bound only its rounding)
        return {k: r[k] for k in ("xPhys", "cHist", "volHist", "sharpHist", "lssIts", "cSolid")}
    if kind == "solve":
        p = s["p"]
        p.set_modulus(s["E"])
        p.assemble()
        u, its, _ = p.pcg(s["F"])
        return {"u": u, "its": its, "ce": p.compliance(u)}
    if kind == "matvec":
        return s["p"].apply_K(s["u"])
    if kind == "update":
        dc, its = s["p"].filter(0, s["xdc"])
        x, change, nbis = s["p"].oc(s["x"], s["x"], dc / np.maximum(1e-3, s["x"]), s["V0"])
        return {"dc": dc, "its": its, "x": x, "change": change, "bisections": nbis}
    if kind == "oc":
        s["x"].copy_(s["x0"])
        change, nbis = t3x.oc_noalloc(s["n"], s["x"].data_ptr(), s["xPhys"].data_ptr(), s["dc"].data_ptr(), 0, s["V0"])
        return {"x": s["x"], "change": change, "bisections": nbis}
    for r in s["reqs"]:
        s["server"].submit(**r)
    done = {}
    while len(done) < len(s["reqs"]):
        for c in s["server"].poll(wait_ms=1000):
            done[c["tag"]] = c
    return {str(t): {k: done[t][k] for k in ("status", "loops", "pcgIts", "cSolid", "cHist", "xPhys")}
            for t in sorted(done)}


# --------------------------------------------------------------------- work
def _solve_work(ny, nx, nz, its):
    """Bytes and flops of `its` iterations of the preconditioned CG: the
    operator, the residual and direction updates and one V-cycle's fine level,
    each vector and modulus read or written once."""
    nn, ne = (ny + 1.0) * (nx + 1) * (nz + 1), float(ny) * nx * nz
    return its * (nn * (48 + 72 + 120 + 48) + 8 * ne), its * (196 * ne + 60 * nn)


def work(case):
    kind = case["kind"]
    if kind == "serve":
        b = f = 0.0
        for s in (int(v) for v in case["sizes"].split(",")):
            w = _solve_work(s, 2 * s, s, 25 * (case["nLoop"] + 1))
            b, f = b + w[0], f + w[1]
        return dict(bytes=b, flops=f)
    if kind == "oc":  # xPhys once, x and dc once per four of about 50 bisections, x written
        return dict(bytes=case["n"] * (8.0 + 16 * 13 + 8), flops=case["n"] * 250.0)
    ny, nx, nz = case["ny"], case["nx"], case["nz"]
    nn, ne = (ny + 1.0) * (nx + 1) * (nz + 1), float(ny) * nx * nz
    fill = 0.35 if case.get("domain") == "irregular" else 1.0
    if kind == "run":
        b, f = _solve_work(ny, nx, nz, 25 * (case["nLoop"] + 1))
        return dict(bytes=fill * b, flops=fill * f)
    if kind == "solve":
        b, f = _solve_work(ny, nx, nz, 25)
        return dict(bytes=b + 8 * (6 * nn + 2 * ne), flops=f)
    if kind == "matvec":
        return dict(bytes=48 * nn + 8 * ne, flops=196 * ne + 21 * nn)
    return dict(bytes=48 * ne + 8 * 80 * nn + 16 * 13 * ne, flops=8 * 150 * nn + 250 * ne)


# -------------------------------------------------------------------- exact
_LOC = [(1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 0), (1, 0, 1), (1, 1, 1), (0, 1, 1), (0, 0, 1)]  # dy, dx, dz
_NAT = [(1 if dx else -1, -1 if dy else 1, 1 if dz else -1) for dy, dx, dz in _LOC]


def _gauss():
    g = 1 / math.sqrt(3.0)
    for q in range(8):
        xi = [g if q >> k & 1 else -g for k in range(3)]
        N = np.array([0.125 * np.prod([1 + s[k] * xi[k] for k in range(3)]) for s in _NAT])
        dN = np.array([[0.125 * s[k] * np.prod([1 + s[m] * xi[m] for m in range(3) if m != k]) for k in range(3)]
                       for s in _NAT])
        yield N, dN


def _element_stiffness():
    lam, mu = NU / ((1 + NU) * (1 - 2 * NU)), 0.5 / (1 + NU)
    D = np.zeros((6, 6))
    D[:3, :3] = lam
    D[range(6), range(6)] += [2 * mu] * 3 + [mu] * 3
    K = np.zeros((24, 24))
    for _, dN in _gauss():
        B = np.zeros((6, 24))
        for a in range(8):
            bx, by, bz = 2 * dN[a]
            B[:, 3 * a:3 * a + 3] = [[bx, 0, 0], [0, by, 0], [0, 0, bz], [0, bz, by], [bz, 0, bx], [by, bx, 0]]
        K += 0.125 * B.T @ D @ B
    return K


def _dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def _corners(U):
    """(nz, nx, ny, 8, ...) nodal values of every cell from the (NZ, NX, NY, ...) grid."""
    NZ, NX, NY = U.shape[:3]
    return torch.stack([U[dz:NZ - 1 + dz, dx:NX - 1 + dx, dy:NY - 1 + dy] for dy, dx, dz in _LOC], dim=3)


def _scatter(V, shape):
    out = torch.zeros(shape, dtype=torch.float64, device=V.device)
    NZ, NX, NY = shape[:3]
    for a, (dy, dx, dz) in enumerate(_LOC):
        out[dz:NZ - 1 + dz, dx:NX - 1 + dx, dy:NY - 1 + dy] += V[:, :, :, a]
    return out


def _elastic(E, ny, nx, nz):
    """u -> K u with the face x = 0 fixed, and the operator's diagonal."""
    Ke = _dev(_element_stiffness())
    Eg = _dev(E).reshape(nz, nx, ny, 1, 1)
    shape = (nz + 1, nx + 1, ny + 1, 3)

    def apply(u):
        v = u.reshape(shape).clone()
        v[:, 0] = 0
        w = _corners(v).reshape(-1, 24) @ Ke
        y = _scatter(w.reshape(nz, nx, ny, 8, 3) * Eg, shape)
        y[:, 0] = u.reshape(shape)[:, 0]
        return y.reshape(-1)
    d = _scatter(Ke.diagonal().reshape(1, 1, 1, 8, 3) * Eg, shape)
    d[:, 0] = 1
    return apply, d.reshape(-1), Ke


def _cg(apply, diag, b, tol, most):
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz, end = z.clone(), r @ z, tol * float(b.norm())
    for k in range(most):
        q = apply(p)
        a = rz / (p @ q)
        x += a * p
        r -= a * q
        if k % 16 == 15 and float(r.norm()) < end:
            return x
        z = r / diag
        rz, old = r @ z, rz
        p = z + (rz / old) * p
    return None


def _oc(x, xPhys, dc, V0):
    l1, l2, n = 0.0, 1e9, 0
    fval = float(xPhys.mean()) - V0
    lo, hi, t = (x - 0.2).clamp(min=0.0), (x + 0.2).clamp(max=1.0), x * (-dc).sqrt()
    while (l2 - l1) / (l1 + l2) > 1e-6:
        lm = 0.5 * (l1 + l2)
        xn = torch.maximum(lo, torch.minimum(hi, t / math.sqrt(lm)))
        if fval + float((xn - x).sum()) > 0:
            l1 = lm
        else:
            l2 = lm
        n += 1
    return xn, float((xn - x).abs().max()), n


def exact(case, seed):
    kind = case["kind"]
    if kind in ("run", "serve"):
        return None
    if kind == "oc":
        s = prepare(case, seed)
        x, change, n = _oc(s["x0"], s["xPhys"], s["dc"], s["V0"])
        return {"x": x, "change": change, "bisections": n}
    ny, nx, nz = case["ny"], case["nx"], case["nz"]
    rng = np.random.default_rng(seed)
    force = _load(rng)
    x = _density((ny, nx, nz), rng)
    if kind == "update":
        dc = -np.exp(rng.normal(-2.0, 1.0, x.size)) * 3 * x * x
        ir2 = (case["rMin"] / 2 / math.sqrt(3.0)) ** 2
        K = sum(ir2 * (dN @ dN.T) + np.outer(N, N) / 8 for N, dN in _gauss())
        Kd, shape = _dev(K), (nz + 1, nx + 1, ny + 1)

        def apply(u):
            return _scatter(_corners(u.reshape(shape)) @ Kd, shape).reshape(-1)
        ones = torch.ones((nz, nx, ny, 8), dtype=torch.float64, device="cuda")
        b = _scatter(_dev(x * dc).reshape(nz, nx, ny, 1) * ones / 8, shape).reshape(-1)
        u = _cg(apply, _scatter(ones * Kd.diagonal(), shape).reshape(-1), b, 1e-14, 400)
        if u is None:
            return None
        f = _corners(u.reshape(shape)).mean(dim=3).reshape(-1)
        xd = _dev(x)
        xn, change, n = _oc(xd, xd, f / xd.clamp(min=1e-3), case["V0"])
        return {"dc": f, "its": None, "x": xn, "change": change, "bisections": n}
    E = EMIN + x ** PENAL * (E0 - EMIN)
    apply, diag, Ke = _elastic(E, ny, nx, nz)
    if kind == "matvec":
        return apply(_dev(rng.standard_normal(3 * (ny + 1) * (nx + 1) * (nz + 1))))
    if (ny + 1) * (nx + 1) * (nz + 1) > 200_000:
        return None
    _, (nodes, vec) = _cantilever(ny, nx, nz, force)
    b = np.zeros(((ny + 1) * (nx + 1) * (nz + 1), 3))
    b[nodes] = vec
    u = _cg(apply, diag, _dev(b).reshape(-1), 1e-11, 12000)
    if u is None:
        return None
    ue = _corners(u.reshape(nz + 1, nx + 1, ny + 1, 3)).reshape(-1, 24)
    return {"u": u, "its": None, "ce": ((ue @ Ke) * ue).sum(dim=1)}
