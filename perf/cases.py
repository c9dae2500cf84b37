"""Performance cases of the library, called as a user's program calls it: the
C ABI of include/spdk.h through spd_k_amd.lib() and spd_k_amd.Context on device
tensors, and the whole driver spd_k_amd.run().

listed() names the cases, draw() gives further ones of the same ranges,
prepare() makes inputs and handles, run() is one pass, work() the bytes and
operations a pass cannot do without, exact() the same results from plain
float64 torch. Steps start from the prepared state on every pass (the state is
copied back first, as a program that may reject a step does).
"""
import ctypes
import math
import os
import shutil
import tempfile

import numpy as np
import torch

import spd_k_amd as sk

HERE = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GAMMA, CFL, NAD_TOL = 1.4, 0.8, 1e-5
BC = {"periodic": 0, "gradfree": 1, "reflective": 2}


def listed():
    return [
        # a small 2-D run inside a serving loop: launches and the dt read-back
        {"name": "step2d_32", "kind": "step", "dim": 2, "p": 3, "nx": 32, "ny": 32, "nz": 1, "flow": "sine",
         "bc": "periodic", "integ": "ader", "form": "noalloc"},
        # the plain FP64 update at an ordinary 3-D size
        {"name": "step3d_64", "kind": "step", "dim": 3, "p": 3, "nx": 64, "ny": 64, "nz": 64, "flow": "kh",
         "bc": "periodic", "integ": "ader", "form": "fp64"},
        # the mixed-precision update at the largest configured mesh
        {"name": "mixed3d_96", "kind": "step", "dim": 3, "p": 3, "nx": 96, "ny": 96, "nz": 96, "flow": "kh",
         "bc": "periodic", "integ": "ader", "form": "mixed"},
        # 2-D p = 4 Kelvin-Helmholtz with residual-driven Picard
        {"name": "residual2d_512_p4", "kind": "step", "dim": 2, "p": 4, "nx": 512, "ny": 512, "nz": 1, "flow": "kh",
         "bc": "periodic", "integ": "ader", "form": "residual"},
        # a 2-D blast with trouble detection and the fallback, walls all round
        {"name": "blast2d_256", "kind": "fallback", "dim": 2, "p": 3, "nx": 256, "ny": 256, "nz": 1, "flow": "blast",
         "bc": "reflective", "form": "fp64"},
        # 3-D Kelvin-Helmholtz with the fallback in FP64, a ragged mesh
        {"name": "fallback3d_62", "kind": "fallback", "dim": 3, "p": 3, "nx": 62, "ny": 66, "nz": 61, "flow": "kh",
         "bc": "periodic", "form": "fp64"},
        # the configured production step: 96^3, fallback, learned Picard guess
        {"name": "learned3d_96", "kind": "fallback", "dim": 3, "p": 3, "nx": 96, "ny": 96, "nz": 96, "flow": "kh",
         "bc": "periodic", "form": "learned"},
        # the 2-D field loop at its configured size
        {"name": "induction2d_1024", "kind": "induction", "dim": 2, "p": 3, "nx": 1024, "ny": 1024, "nz": 1,
         "bc": "periodic", "form": "fp64"},
        # the 3-D induction solver in mixed precision, a ragged mesh
        {"name": "induction3d_40", "kind": "induction", "dim": 3, "p": 3, "nx": 40, "ny": 37, "nz": 43,
         "bc": "periodic", "form": "mixed"},
        # degree 7 runs the stage kernels one by one (128 cells per axis)
        {"name": "stages3d_p7", "kind": "stages", "dim": 3, "p": 7, "nx": 16, "ny": 16, "nz": 16, "flow": "sine",
         "bc": "periodic", "integ": "rk3"},
        # a whole run from the command line: set-up, 40 steps with the
        # fallback, the final output
        {"name": "run_kh2d_64", "kind": "driver", "p": 3, "nx": 64, "ny": 64, "steps": 40},
        # training the Picard guess: 8 Adam steps, the weights fetched
        {"name": "train_guess", "kind": "train", "din": 326, "hidden": 256, "dout": 1280, "batch": 4096, "steps": 8},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh(rng, dim, lo, hi):
    n = _size(rng, lo, hi)
    around = [max(lo, min(hi, n + rng.randint(-max(1, n // 8), max(1, n // 8)))) for _ in range(dim)]
    return around + [1] * (3 - dim)


def draw(rng):
    kind = rng.choice(["step", "step", "step", "fallback", "fallback", "induction", "stages", "driver", "train"])
    if kind == "driver":
        nx, ny, _ = _mesh(rng, 2, 16, 96)
        return {"kind": kind, "p": rng.randint(2, 4), "nx": nx, "ny": ny, "steps": rng.randint(5, 40)}
    if kind == "train":
        return {"kind": kind, "din": rng.randint(100, 400), "hidden": rng.choice([128, 192, 256]),
                "dout": rng.randint(300, 1300), "batch": rng.randint(500, 4096), "steps": rng.randint(2, 8)}
    if kind == "stages":
        nx, ny, nz = _mesh(rng, 3, 4, 14)
        return {"kind": kind, "dim": 3, "p": rng.randint(5, 7), "nx": nx, "ny": ny, "nz": nz, "flow": "sine",
                "bc": rng.choice(["periodic", "gradfree"]), "integ": rng.choice(["rk2", "rk3"])}
    dim = rng.choice([2, 3])
    p = rng.randint(1, 4 if dim == 2 else 3)
    top = {2: 500, 3: 60}[dim]
    if kind == "induction":
        nx, ny, nz = _mesh(rng, dim, 8, top if dim == 2 else 40)
        return {"kind": kind, "dim": dim, "p": p, "nx": nx, "ny": ny, "nz": nz,
                "bc": rng.choice(["periodic", "gradfree"]), "form": rng.choice(["fp64", "mixed"])}
    bc = rng.choice(["periodic", "periodic", "gradfree", "reflective"])
    if kind == "fallback":
        nx, ny, nz = _mesh(rng, dim, 8, top if dim == 2 else 48)
        flow = rng.choice(["kh", "blast"]) if bc != "periodic" else "kh"
        form = "fp64" if flow == "blast" else rng.choice(["fp64", "mixed", "residual"])
        return {"kind": kind, "dim": dim, "p": max(p, 2), "nx": nx, "ny": ny, "nz": nz, "flow": flow, "bc": bc,
                "form": form}
    nx, ny, nz = _mesh(rng, dim, 8, top)
    form = rng.choice(["fp64", "fp64", "mixed", "residual"])
    integ = rng.choice(["ader", "rk2", "rk3"]) if form == "fp64" else "ader"
    return {"kind": kind, "dim": dim, "p": p, "nx": nx, "ny": ny, "nz": nz, "flow": rng.choice(["sine", "kh"]),
            "bc": bc, "integ": integ, "form": form}


# ---- basis, operators and geometry: what a calling program holds -----------------
def _lagrange(xa, xb, deriv=False):
    """Values (or derivatives) at xb of the Lagrange polynomials on xa."""
    n = len(xa)
    out = np.zeros((len(xb), n))
    for j, y in enumerate(xb):
        for i in range(n):
            o = [k for k in range(n) if k != i]
            if deriv:
                out[j, i] = sum(np.prod([(y - xa[m]) / (xa[i] - xa[m]) for m in o if m != k]) / (xa[i] - xa[k])
                                for k in o)
            else:
                out[j, i] = np.prod([(y - xa[m]) / (xa[i] - xa[m]) for m in o])
    return out


def _gauss(n):
    x, w = np.polynomial.legendre.leggauss(n)
    return 0.5 * (x + 1), 0.5 * w


def _basis(p, ader):
    x_sp = 0.5 * (1 - np.cos((2 * np.arange(p + 1) + 1) / (2.0 * (p + 1)) * np.pi))
    x_fp = np.concatenate([[0.0], _gauss(p)[0], [1.0]])
    q, w = _gauss(p + 1)

    def averages(src):  # cell averages between the flux points of the basis on src
        return np.stack([_lagrange(src, x_fp[k] + q * (x_fp[k + 1] - x_fp[k])).T @ w for k in range(p + 1)])

    xt, wt = (q, w) if ader else (np.zeros(1), np.ones(1))
    end = _lagrange(xt, [1.0])[0]
    D = np.outer(end, end) - _lagrange(xt, xt, True).T * wt[None, :]
    b = {"x_sp": x_sp, "x_fp": x_fp, "wt": wt, "sp_to_fp": _lagrange(x_sp, x_fp), "fp_to_sp": _lagrange(x_fp, x_sp),
         "dfp_to_sp": _lagrange(x_fp, x_sp, True), "sp_to_cv": averages(x_sp), "fp_to_cv": averages(x_fp),
         "invader": np.linalg.inv(D) if ader else np.zeros((1, 1))}
    b["cv_to_sp"] = np.linalg.inv(b["sp_to_cv"])
    return b


class _Mesh:
    """Element mesh of a case: counts with ghosts, widths, the FV sub-grid."""

    def __init__(self, c, ader=True):
        self.c, self.p, self.n = c, c["p"], c["p"] + 1
        self.dim = c.get("dim", 2)
        self.N = [c["nx"], c["ny"], c.get("nz", 1)]
        self.act = [d < self.dim for d in range(3)]
        self.Nt = [self.N[d] + 2 if self.act[d] else 1 for d in range(3)]
        self.q = [self.n if a else 1 for a in self.act]
        self.h = [1.0 / self.N[d] if self.act[d] else 1.0 for d in range(3)]
        self.b = _basis(self.p, ader)
        self.T = len(self.b["wt"])
        self.bc = [BC[c.get("bc", "periodic")]] * 3
        self.nc = [self.N[d] * self.n + 4 if self.act[d] else 1 for d in range(3)]
        self.faces, self.centers = [], []
        for d in range(3):
            if not self.act[d]:
                self.faces.append(np.array([-1.0, 0.0]))
                self.centers.append(np.array([-1.0]))
                continue
            f = (np.arange(-1, self.N[d] + 1)[:, None] + self.b["x_fp"][None, :-1]).reshape(-1) * self.h[d]
            f = np.append(f, (self.N[d] + 1) * self.h[d])
            lo = self.n - 2
            self.centers.append(0.5 * (f[1:] + f[:-1])[lo:lo + self.nc[d]])
            self.faces.append(f[lo:lo + self.nc[d] + 1].copy())
            self.faces[d][-1] = 0.0  # the last ghost face is not set

    def shape(self, nt=1, nv=6, stag=()):
        s = [self.q[d] + 1 if d in stag and self.act[d] else self.q[d] for d in range(3)]
        return (nt, nv, self.Nt[2], self.Nt[1], self.Nt[0], s[2], s[1], s[0])

    def fv_shape(self, nv=6, face=None):
        s = [self.nc[d] + (d == face) for d in range(3)]
        return (nv, s[2], s[1], s[0])

    def points(self):
        return float(np.prod(self.N)) * self.n ** self.dim

    def at(self, d, x):
        """Coordinates of points x of every element along axis d, shaped for broadcasting over (element, point)."""
        if not self.act[d]:
            return torch.full((1,) * 6, 0.5, dtype=torch.float64, device="cuda")
        v = (np.arange(-1, self.N[d] + 1)[:, None] + x[None, :]) * self.h[d]
        s = [1] * 6
        s[2 - d], s[5 - d] = v.shape
        return torch.from_numpy(v).cuda().reshape(s)

    def context(self, **kw):
        ops = {k: self.b[k] for k in sk.Context.MATS}
        ops.update(wt=self.b["wt"], fv_faces=self.faces, fv_centers=self.centers)
        return sk.Context(self.p, self.act, self.bc, self.T, ops, gamma=GAMMA, cfl=CFL, h=self.h, nad_tol=NAD_TOL, **kw)


def _flow(m, seed):
    """Primitive variables at the solution points (ghosts included) and a stable time step."""
    c, g = m.c, torch.Generator(device="cuda")
    g.manual_seed(seed)
    r = np.random.default_rng(seed)
    x, y, z = (m.at(d, m.b["x_sp"]) for d in range(3))
    w = torch.zeros(m.shape()[1:], dtype=torch.float64, device="cuda")
    if c["flow"] == "sine":
        w[0] = 1.0 + 0.125 * torch.sin(2 * math.pi * (x + y + r.uniform()))
        w[1], w[2], w[4] = 1.0, 1.0, 1.0
    elif c["flow"] == "kh":
        inner = torch.sigmoid((0.25 - (y - 0.5).abs()) / 0.01)
        w[0] = 1.0 + inner
        w[1] = -0.5 + inner
        s2 = 2 * 0.05 ** 2 / 2
        layers = torch.exp(-(y - 0.25) ** 2 / s2) + torch.exp(-(y - 0.75) ** 2 / s2)
        noise = torch.randn(m.shape()[2:5] + (1, 1, 1), generator=g, dtype=torch.float64, device="cuda")
        w[2] = layers * (0.01 * noise + 0.05 * torch.sin(4 * math.pi * (x + r.uniform())))
        if m.act[2]:
            w[3] = 0.05 * layers * torch.sin(2 * math.pi * (z + r.uniform()))
        w[4] = 2.5
    else:  # a blast: hot sphere in a cold gas
        cx = 0.5 + 0.1 * r.uniform(-1, 1, 3)
        rr = (x - cx[0]) ** 2 + (y - cx[1]) ** 2 + ((z - cx[2]) ** 2 if m.act[2] else 0.0)
        w[0] = 1.0
        w[4] = 0.1 + (10.0 + r.uniform()) * torch.sigmoid((0.15 - rr.sqrt()) / 0.004)
    cs = (GAMMA * w[4] / w[0]).sqrt()
    speed = sum(w[1 + d].abs() + cs for d in range(m.dim))
    dt = 0.9 * CFL * min(m.h[:m.dim]) / float(speed.max()) / m.n
    u = torch.zeros((1,) + tuple(w.shape), dtype=torch.float64, device="cuda")
    u[0, 0] = w[0]
    for v in (1, 2, 3):
        u[0, v] = w[0] * w[v]
    u[0, 4] = w[4] / (GAMMA - 1) + 0.5 * w[0] * (w[1] ** 2 + w[2] ** 2 + w[3] ** 2)
    return u, dt


def _field(m, seed):
    """Face magnetic field of a loop with a weak z component, and a stable time step."""
    r = np.random.default_rng(seed)
    cx, cy, R = 0.5 + 0.1 * r.uniform(-1, 1), 0.5 + 0.1 * r.uniform(-1, 1), r.uniform(0.2, 0.3)
    out = []
    for d in range(3):
        x, y, z = (m.at(e, m.b["x_fp"] if e == d else m.b["x_sp"]) for e in range(3))
        x, y = x - torch.floor(x) - cx, y - torch.floor(y) - cy
        rr = (x * x + y * y).sqrt()
        loop = 0.001 * torch.sigmoid((R - rr) / 0.01) / (rr + 1e-3)
        b = -loop * y if d == 0 else loop * x if d == 1 else 1e-4 * torch.cos(2 * math.pi * (x + y)) + 0 * z
        out.append((b + torch.zeros(m.shape(1, 1, (d,)), dtype=torch.float64, device="cuda")).contiguous())
    return out, CFL * min(m.h[:m.dim]) / sum(abs(v) for v in VEL[:m.dim]) / m.n


VEL = (1.0, 0.5, 0.25)


# ---- the C ABI through ctypes -----------------------------------------------------
class _Picard(ctypes.Structure):
    _fields_ = [("residual", ctypes.c_int), ("guess", ctypes.c_int), ("tol", ctypes.c_double),
                ("max_sweeps", ctypes.c_int), ("guess_keep", ctypes.c_int)]


class _PicardStats(ctypes.Structure):
    _fields_ = [("steps", ctypes.c_longlong), ("fallbacks", ctypes.c_longlong), ("sweeps", ctypes.c_double),
                ("last_residual", ctypes.c_double)]


def _p(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _d(v):
    return ctypes.c_double(v)


def _zeros(shape, dtype=torch.float64):
    return torch.zeros(shape, dtype=dtype, device="cuda")


def _workspace(fn, ctx, m):
    fn.restype = ctypes.c_size_t
    nb = fn(ctx, (ctypes.c_int * 3)(*m.Nt))
    if nb == 0:
        raise RuntimeError(sk.last_error())
    return _zeros(nb, torch.uint8)


class _Net:
    """A network handle, freed with its state."""

    def __init__(self, dims, batch, params):
        self.L, self.net, self.dims = sk.lib(), ctypes.c_void_p(), dims
        sk.check(self.L.spdk_mlp_create((ctypes.c_int * 4)(*dims), batch,
                                        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream),
                                        ctypes.byref(self.net)), "mlp_create")
        assert self.L.spdk_mlp_param_count(self.net) == len(params)
        sk.check(self.L.spdk_mlp_set_params(self.net, params.ctypes.data), "mlp_set_params")

    def __del__(self):
        self.L.spdk_mlp_destroy(self.net)


def _weights(path):
    """A weights file: magic, four dimensions, degree, dimensionality, count, parameters."""
    with open(path, "rb") as f:
        head = f.read(40)
        dims = np.frombuffer(head, np.int32, 4, 8)
        return [int(v) for v in dims], np.frombuffer(f.read(), np.float32).copy()


def prepare(case, seed):
    kind = case["kind"]
    if kind == "driver":
        r = np.random.default_rng(seed)
        args = ["-i", os.path.join(HERE, "tests", "inputs", "kelvin_helmholtz.athinput"), "mesh/p=%d" % case["p"],
                "mesh/nx1=%d" % case["nx"], "mesh/nx2=%d" % case["ny"], "time/tlim=10", "output/dt=-1",
                "time/nlim=%d" % case["steps"], "problem/amp=%.17g" % r.uniform(0.05, 0.1),
                "problem/v1=%.17g" % r.uniform(0.4, 0.5), "output/fields=W_cv", "job/final_output=true"]
        return {"kind": kind, "case": case, "args": args, "amp": float(args[8].split("=")[1]),
                "v1": float(args[9].split("=")[1])}
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        s = {"step": _prepare_hydro, "fallback": _prepare_hydro, "stages": _prepare_stages,
             "induction": _prepare_induction, "train": _prepare_train}[kind](case, seed)
    s.update(kind=kind, case=case, stream=stream)
    return s


def run(s):
    if s["kind"] == "driver":
        return _run_driver(s)
    with torch.cuda.stream(s["stream"]):
        return {"step": _run_step, "fallback": _run_fallback, "stages": _run_stages, "induction": _run_induction,
                "train": _run_train}[s["kind"]](s)


def _prepare_hydro(c, seed):
    rk = c.get("integ", "ader")
    m = _Mesh(c, rk == "ader")
    u0, dt = _flow(m, seed)
    ctx = m.context(rk_order=0 if rk == "ader" else int(rk[2]))
    L, form = sk.lib(), c["form"]
    s = {"m": m, "ctx": ctx, "U0": u0, "U": u0.clone(), "dt": dt, "W_cv": torch.zeros_like(u0), "pc": None, "ws": None}
    if form in ("fp64", "mixed", "residual", "learned"):
        s["ws"] = _workspace(L.spdk_fused_workspace_bytes if form == "fp64" else L.spdk_mixed_workspace_bytes, ctx.ctx, m)
    if form not in ("fp64", "noalloc"):
        s["pc"] = _Picard(int(form != "mixed"), 2 if form == "learned" else 0, 1e-6, 1 if form == "learned" else 0, 0)
        s["stats"] = _PicardStats()
    if form == "learned":
        dims, params = _weights(os.path.join(HERE, "spd_k_amd", "weights", "kh3d_p3.mlp"))
        s["net"] = _Net(dims, 65536, params)
        sk.check(L.spdk_mixed_attach_mlp(ctx.ctx, s["net"].net), "attach_mlp")
    if c["kind"] == "fallback":
        for name in ("A", "B", "W_new", "W_old", "troubles"):
            s[name] = _zeros(m.fv_shape())
        s["theta"], s["theta_tmp"] = _zeros(m.fv_shape(1)), _zeros(m.fv_shape(1))
        s["abits"] = _zeros(m.fv_shape(1), torch.int16)
        s["F"] = [[_zeros(m.fv_shape(6, d)) if m.act[d] else None for d in range(3)] for _ in range(m.T)]
        s["Fp"] = (ctypes.c_void_p * (3 * m.T))(*[f.data_ptr() if f is not None else None for t in s["F"] for f in t])
    return s


def _run_step(s):
    L, ctx, U, c = sk.lib(), s["ctx"], s["U"], s["case"]
    U.copy_(s["U0"])
    if c["form"] == "noalloc":
        dt = ctx.hydro_step_fused_noalloc(U, s["dt"], s["W_cv"])
        return {"U": U, "W_cv": s["W_cv"], "dt": dt}
    out = ctypes.c_double()
    if c["form"] == "fp64":
        sk.check(L.spdk_hydro_step_fused(ctx.ctx, _p(U), sk.SDShape.of(U.shape), _p(s["ws"]), _d(s["dt"]),
                                         _p(s["W_cv"]), None, ctypes.byref(out)), "hydro_step_fused")
    else:
        sk.check(L.spdk_hydro_step_mixed(ctx.ctx, _p(U), sk.SDShape.of(U.shape), _p(s["ws"]), _d(s["dt"]),
                                         _p(s["W_cv"]), None, ctypes.byref(s["pc"]), ctypes.byref(s["stats"]),
                                         ctypes.byref(out)), "hydro_step_mixed")
    return {"U": U, "W_cv": s["W_cv"], "dt": out.value}


def _run_fallback(s):
    """One ADER step with the FV update, trouble detection and the MUSCL-HLLC fallback."""
    L, x, U, m = sk.lib(), s["ctx"].ctx, s["U"], s["m"]
    sp, fv, th = sk.SDShape.of(U.shape), sk.FVShape.of(m.fv_shape()), sk.FVShape.of(m.fv_shape(1))
    dt = s["dt"]
    U.copy_(s["U0"])
    if s["pc"] is None:
        sk.check(L.spdk_fused_predict_fv_fluxes(x, _p(U), sp, _p(s["ws"]), _d(dt), s["Fp"], fv, None,
                                                sk.SDShape.of(m.shape(m.T))), "fused_predict_fv_fluxes")
    else:
        sk.check(L.spdk_mixed_predict_fv_fluxes(x, _p(U), sp, _p(s["ws"]), _d(dt), ctypes.byref(s["pc"]),
                                                ctypes.byref(s["stats"]), s["Fp"], fv, None, 0),
                 "mixed_predict_fv_fluxes")
    A, B, Wn, Wo, tr, theta = s["A"], s["B"], s["W_new"], s["W_old"], s["troubles"], s["theta"]
    sk.check(L.spdk_fv_state_from_sd(x, _p(U), sp, _p(A), fv), "fv_state_from_sd")
    for t in range(m.T):
        F = [_p(f) for f in s["F"][t]]
        sk.check(L.spdk_fv_state_update_prims(x, _p(B), _p(Wn), _p(Wo), _p(A), *F, fv, t, _d(dt), 0x11), "update_prims")
        sk.check(L.spdk_fill_fv_ghosts(x, _p(Wo), fv), "fill_fv_ghosts")
        sk.check(L.spdk_fill_fv_ghosts(x, _p(Wn), fv), "fill_fv_ghosts")
        sk.check(L.spdk_detect_troubles_bits(x, _p(Wn), _p(Wo), _p(tr), _p(s["abits"]), fv, 1, 0x11), "detect_troubles")
        sk.check(L.spdk_fill_fv_ghosts(x, _p(tr), fv), "fill_fv_ghosts")
        sk.check(L.spdk_blend_theta(x, _p(tr), _p(s["theta_tmp"]), _p(theta), fv), "blend_theta")
        sk.check(L.spdk_fill_fv_ghosts(x, _p(theta), th), "fill_fv_ghosts")
        sk.check(L.spdk_muscl_hllc_blend(x, _p(Wo), _p(theta), *F, fv, _d(m.b["wt"][t] * dt)), "muscl_hllc_blend")
        sk.check(L.spdk_fv_state_update_blended(x, _p(B), _p(A), *F, _p(theta), fv, t, _d(dt)), "update_blended")
        A, B = B, A
    out = ctypes.c_double()
    sk.check(L.spdk_fv_state_to_sd(x, _p(A), fv, _p(U), sp, _p(s["W_cv"]), ctypes.byref(out)), "fv_state_to_sd")
    return {"U": U, "W_cv": s["W_cv"], "dt": out.value}


def _prepare_stages(c, seed):
    m = _Mesh(c, False)
    u0, dt = _flow(m, seed)
    s = {"m": m, "ctx": m.context(rk_order=int(c["integ"][2])), "U0": u0, "U": u0.clone(), "dt": dt}
    for name in ("U_ader", "W_sp", "W_cv", "tmp", "Ustart"):
        s[name] = torch.zeros_like(u0)
    s["U_fp"] = [_zeros(m.shape(1, 6, (d,))) for d in range(3)]
    s["F_fp"] = [_zeros(m.shape(1, 6, (d,))) for d in range(3)]
    return s


def _run_stages(s):
    """One SSP-RK step through the kernel-layer functions, as the reference's integrator calls them."""
    x, m, U, Ua, Uf, F = s["ctx"], s["m"], s["U"], s["U_ader"], s["U_fp"], s["F_fp"]
    U.copy_(s["U0"])
    s["Ustart"].copy_(U)
    for a in {"rk2": (0.0, 0.5), "rk3": (0.0, 0.75, 1.0 / 3.0)}[s["case"]["integ"]]:
        x.copy_ader(U, Ua)
        for d in range(3):
            x.transform_a_to_b_1d(Ua, Uf[d], sk.SPDK_M_SP_TO_FP, d)
        for d in range(3):
            x.compute_fluxes(Uf[d], F[d], d)
        for d in range(3):
            x.boundaries(Uf[d], d)
        for d in range(3):
            x.sd_riemann_solver(Uf[d], F[d], d)
        x.update_solution(U, Ua, F[0], F[1], F[2], m.p + 2, s["dt"])
        if a > 0:
            x.combine_solution(U, s["Ustart"], a)
    x.compute_primitives(U, s["W_sp"])
    x.transform_a_to_b(s["W_sp"], s["W_cv"], s["tmp"], sk.SPDK_M_SP_TO_CV)
    return {"U": U, "W_cv": s["W_cv"], "dt": x.compute_dt(s["W_cv"])}


def _prepare_induction(c, seed):
    m = _Mesh(c)
    b0, dt = _field(m, seed)
    ctx, L = m.context(vel=VEL), sk.lib()
    size = L.spdk_induction_fused_workspace_bytes if c["form"] == "fp64" else L.spdk_induction_mixed_workspace_bytes
    return {"m": m, "ctx": ctx, "B0": b0, "B": [b.clone() for b in b0], "dt": dt, "ws": _workspace(size, ctx.ctx, m)}


def _run_induction(s):
    L, B = sk.lib(), s["B"]
    for b, b0 in zip(B, s["B0"]):
        b.copy_(b0)
    step = L.spdk_induction_step_fused if s["case"]["form"] == "fp64" else L.spdk_induction_step_mixed
    args = [v for b in B for v in (_p(b), sk.SDShape.of(b.shape))]
    sk.check(step(s["ctx"].ctx, *args, _p(s["ws"]), _d(s["dt"])), "induction_step")
    return B


def _run_driver(s):
    out = tempfile.mkdtemp(prefix="spdk_run_")
    try:
        r = sk.run(s["args"], out)
        c = s["case"]
        w = np.fromfile(os.path.join(out, "W_cv_N%dp%d_0_0.dat" % (c["nx"], c["p"])))
        return {"W_cv": w, "t": r["t_final"], "steps": r["steps"]}
    finally:
        shutil.rmtree(out)


def _net_params(c, seed):
    dims = [c["din"], c["hidden"], c["hidden"], c["dout"]]
    r, out = np.random.default_rng(seed), []
    for i in range(3):
        out.append(r.standard_normal(dims[i + 1] * dims[i]) * math.sqrt(2.0 / dims[i]) * (0.1 if i == 2 else 1.0))
        out.append(np.zeros(dims[i + 1]))
    return dims, np.concatenate(out).astype(np.float32)


def _train_data(c, seed):
    """Feature and target rows: smooth functions of a few hidden coordinates of each element."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    rows = 2 * c["batch"]
    h = torch.randn(rows, 16, generator=g, device="cuda")
    X = torch.tanh(h @ torch.randn(16, c["din"], generator=g, device="cuda") * 0.3)
    Y = torch.sin(h @ torch.randn(16, c["dout"], generator=g, device="cuda") * 0.3)
    idx = torch.stack([torch.randperm(rows, generator=g, device="cuda")[:c["batch"]] for _ in range(c["steps"])])
    return X.contiguous(), Y.contiguous(), idx.to(torch.int32).contiguous()


LR = 1e-3


def _prepare_train(c, seed):
    dims, params = _net_params(c, seed)
    X, Y, idx = _train_data(c, seed)
    return {"net": _Net(dims, c["batch"], params), "params": params, "X": X, "Y": Y, "idx": idx,
            "Xb": torch.zeros(c["batch"], c["din"], device="cuda"), "Yb": torch.zeros(c["batch"], c["dout"], device="cuda"),
            "out": np.zeros_like(params)}


def _run_train(s):
    """Adam steps on gathered batches from the initial weights, the trained weights back on the host."""
    L, net, c = sk.lib(), s["net"].net, s["case"]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    n, ld = c["batch"], ctypes.c_long
    sk.check(L.spdk_mlp_set_params(net, s["params"].ctypes.data), "mlp_set_params")
    for k in range(c["steps"]):
        i = ctypes.c_void_p(s["idx"][k].data_ptr())
        sk.check(L.spdk_gather_rows(_p(s["X"]), ld(c["din"]), i, n, c["din"], _p(s["Xb"]), st), "gather_rows")
        sk.check(L.spdk_gather_rows(_p(s["Y"]), ld(c["dout"]), i, n, c["dout"], _p(s["Yb"]), st), "gather_rows")
        sk.check(L.spdk_mlp_train_step(net, _p(s["Xb"]), c["din"], _p(s["Yb"]), c["dout"], n, LR, None), "train_step")
    sk.check(L.spdk_mlp_get_params(net, s["out"].ctypes.data), "mlp_get_params")
    return s["out"]


# ---- what a pass cannot do without --------------------------------------------------
def work(case):
    k = case["kind"]
    if k == "train":
        d = [case["din"], case["hidden"], case["hidden"], case["dout"]]
        mac = sum(a * b for a, b in zip(d, d[1:]))
        # forward, weight gradients, input gradients (not of the first layer)
        flops = 2.0 * case["batch"] * case["steps"] * (3 * mac - d[0] * d[1])
        return {"bytes": 4.0 * case["batch"] * case["steps"] * (d[0] + d[3]) + 24.0 * mac * case["steps"], "flops": flops}
    n, dim = case["p"] + 1, case.get("dim", 2)
    pts = float(case["nx"] * case["ny"] * case.get("nz", 1)) * n ** dim
    steps = case.get("steps", 1)
    if k == "induction":
        # face fields in and out; per slice and sweep: interpolation of two fields, derivatives
        return {"bytes": 2 * 8 * 3 * pts, "flops": pts * n * n * 3 * (4 * n + 4 * (n + 1) + 2 * n)}
    T, sweeps = (1, int(case["integ"][2])) if case.get("integ", "ader")[:2] == "rk" else (n, n)
    # per point, slice and sweep: interpolation and divergence of 5 variables, Euler flux, face solves, time contraction
    sweep = dim * (5 * 2 * (n + 1) + 30 * (n + 1) / n + 80 / n + 5 * 2 * (n + 1)) + 10 * T
    flops = pts * T * sweeps * sweep
    moved = 3 * 6 * 8 * pts  # the state in and out, the cell averages out
    if k in ("fallback", "driver"):
        # per node: face integrals, update, detection and the reconstruction of blended cells
        flops += pts * n * (dim * 5 * 2 * n * (dim - 1) + 60 * dim)
    return {"bytes": moved * steps, "flops": flops * steps}


# ---- the same results in plain float64 ------------------------------------------------
def _apply(M, u, axis):
    M = torch.as_tensor(M, dtype=torch.float64, device=u.device)
    v = u.movedim(axis, -1)
    return (v.reshape(-1, v.shape[-1]) @ M.T).reshape(v.shape[:-1] + (M.shape[0],)).movedim(-1, axis)


def _prims(u):
    w = torch.empty_like(u)
    w[0] = u[0]
    w[1:4] = u[1:4] / u[0]
    w[4] = (u[4] - 0.5 * (w[1:4] * u[1:4]).sum(0)) * (GAMMA - 1)
    return w


def _cons(w):
    u = torch.empty_like(w)
    u[0] = w[0]
    u[1:4] = w[0] * w[1:4]
    u[4] = w[4] / (GAMMA - 1) + 0.5 * (w[1:4] * u[1:4]).sum(0)
    return u


def _sound(w):
    return (GAMMA * w[4] / w[0]).clamp(min=1e-14).sqrt()


def _flux(u, d, w=None):
    w = _prims(u) if w is None else w
    f = u * w[1 + d]
    f[1 + d] += w[4]
    f[4] += w[4] * w[1 + d]
    return f


def _llf(a, b, d):
    wa, wb = _prims(a), _prims(b)
    c = torch.maximum(_sound(wa) + wa[1 + d].abs(), _sound(wb) + wb[1 + d].abs())
    return 0.5 * (_flux(b, d, wb) + _flux(a, d, wa)) - 0.5 * c * (b - a)


def _ghost(v, sign, lo_hi, bc):
    """Values (left, right) of the two ghost sides from the interior's (low side, high side)."""
    lo, hi = lo_hi
    return (hi, lo) if bc == 0 else (lo, hi) if bc == 1 else (lo * sign, hi * sign)


def _sign(u, d):
    s = torch.ones((u.shape[0],) + (1,) * (u.dim() - 1), dtype=u.dtype, device=u.device)
    s[1 + d] = -1
    return s


def _face_fluxes(m, u, d):
    """Flux-point fluxes along d of one slice u (5, element, point), face solves included."""
    ea, pa = 3 - d, 6 - d
    v = _apply(m.b["sp_to_fp"], u, pa)
    F = _flux(v, d)
    lo, hi = v.select(pa, 0), v.select(pa, -1)
    N = v.shape[ea]
    left, right = _ghost(v, _sign(lo.select(ea, 0), d), (lo.select(ea, 1).clone(), hi.select(ea, N - 2).clone()), m.bc[d])
    hi.select(ea, 0).copy_(left)
    lo.select(ea, N - 1).copy_(right)
    f = _llf(hi.narrow(ea, 0, N - 1), lo.narrow(ea, 1, N - 1), d)
    F.select(pa, -1).narrow(ea, 0, N - 1).copy_(f)
    F.select(pa, 0).narrow(ea, 1, N - 1).copy_(f)
    return F


def _rate(m, u):
    r = torch.zeros_like(u)
    for d in range(m.dim):
        r += _apply(m.b["dfp_to_sp"], _face_fluxes(m, u, d), 6 - d) / m.h[d]
    return r


def _cv(m, u, name="sp_to_cv"):
    for d in range(m.dim):
        u = _apply(m.b[name], u, 6 - d)
    return u


def _slot(u):
    return torch.cat([u, torch.zeros_like(u[:1])])[None]


def _finish(m, u):
    """U with its slot, the cell averages of the primitives, the next time step."""
    w = _cv(m, _prims(u))
    inner = w
    for d in range(m.dim):
        inner = inner.narrow(3 - d, 1, m.N[d])
    speed = sum(inner[1 + d].abs() + _sound(inner) for d in range(m.dim))
    dt = CFL * min([1.0] + m.h[:m.dim]) / speed.max() / m.n
    return {"U": _slot(u), "W_cv": _slot(w), "dt": float(dt)}


def _predict(m, u, dt):
    """The slices of the ADER predictor after its p Picard sweeps."""
    w, inv = m.b["wt"], m.b["invader"]
    slices = [u] * m.T
    for k in range(m.T - 1):
        r = [_rate(m, s) for s in slices] if k else [_rate(m, u)] * m.T
        slices = [u - dt * sum(inv[t, q] * w[q] * r[q] for q in range(m.T)) for t in range(m.T)]
        del r
    return slices


def _exact_step(m, u, dt, integ):
    if integ == "ader":
        du = torch.zeros_like(u)
        for t, s in enumerate(_predict(m, u, dt)):
            du += m.b["wt"][t] * dt * _rate(m, s)
        return u - du
    u0 = u
    for a in {"rk2": (0.0, 0.5), "rk3": (0.0, 0.75, 1.0 / 3.0)}[integ]:
        v = u - dt * _rate(m, u)
        u = a * u0 + (1 - a) * v
    return u


def _cells(m, u):
    """Cell values (5, element, point) of the interior on the FV grid without ghosts."""
    for d in range(m.dim):
        u = u.narrow(3 - d, 1, m.N[d])
    v, c, b, a, r, q, p = u.shape
    return u.permute(0, 1, 4, 2, 5, 3, 6).reshape(v, c * r, b * q, a * p)


def _fill(m, a, vector=True):
    """a (variables, z, y, x) without ghosts -> with two ghost layers per active axis."""
    for d in range(m.dim):
        ax, n = 3 - d, a.shape[3 - d]
        first, last = a.narrow(ax, 0, 2), a.narrow(ax, n - 2, 2)
        if m.bc[d] == 2:
            sign = _sign(a, d) if vector else 1.0
            a = torch.cat([first.flip(ax) * sign, a, last.flip(ax) * sign], ax)
        elif m.bc[d] == 1:
            a = torch.cat([first, a, last], ax)
        else:
            a = torch.cat([last, a, first], ax)
    return a


def _shift(a, off, grow):
    """a (.., z, y, x) shifted by off (per axis x, y, z), trimmed by grow per axis."""
    for d in range(3):
        if grow[d]:
            ax = a.dim() - 1 - d
            a = a.narrow(ax, grow[d] + off[d], a.shape[ax] - 2 * grow[d])
    return a


def _box(m):
    r = [(-1, 0, 1) if m.act[d] else (0,) for d in range(3)]
    return [(i, j, k) for k in r[2] for j in r[1] for i in r[0]]


def _along(v, d):
    s = [1, 1, 1]
    s[2 - d] = -1
    return torch.as_tensor(v, dtype=torch.float64, device="cuda").reshape(s)


def _theta(m, old, new):
    """Blending weights, with two ghost layers, from the primitives before and after the update (with ghosts)."""
    g1 = [1 if a else 0 for a in m.act]
    tr = torch.zeros_like(old[0])
    core = _shift(tr, (0, 0, 0), g1)
    for v in (0, 4):
        near = [_shift(old[v], o, g1) for o in _box(m)]
        hi, lo = near[0], near[0]
        for x in near[1:]:
            hi, lo = torch.maximum(hi, x), torch.minimum(lo, x)
        del near
        w = _shift(new[v], (0, 0, 0), g1)
        bad = (w > hi + hi.abs() * NAD_TOL) | (w < lo - lo.abs() * NAD_TOL)
        if m.p > 1:
            alpha = None
            for d in range(m.dim):
                ax, c, f, x = 2 - d, m.centers[d], m.faces[d], new[v]
                n = x.shape[ax]
                u = [x.narrow(ax, 2 + o, n - 4) for o in (-2, -1, 0, 1, 2)]
                span = _along(c[3:-1] - c[1:-3], d)
                du = (u[3] - u[1]) / span
                dup = (u[4] - u[2]) / _along(c[4:] - c[2:-2], d)
                dum = (u[2] - u[0]) / _along(c[2:-2] - c[:-4], d)
                dv = 0.5 * (dup - dum) / span * _along(f[3:-2] - f[2:-3], d)
                side = []
                for e in (du - dum, dup - du):
                    s = torch.where(dv < 0, e.clamp(max=0), e.clamp(min=0)) / dv
                    side.append(torch.where(dv == 0, torch.ones_like(s), s.clamp(max=1)))
                al = torch.zeros_like(x)  # cells without a stencil keep 0
                keep = [slice(2, -2) if a else slice(None) for a in m.act][::-1]
                inside = torch.minimum(*side)
                cut = [slice(None) if (2 - k) == d or not m.act[2 - k] else slice(2, -2) for k in range(3)]
                al[tuple(keep)] = inside[tuple(cut)]
                for o in (-1, 0, 1):
                    off = [0, 0, 0]
                    off[d] = o
                    s = _shift(al, off, g1)
                    alpha = s if alpha is None else torch.minimum(alpha, s)
            bad &= alpha < 1
        core.copy_(torch.maximum(core, bad.double()))
    for v in (0, 4):
        w = _shift(new[v], (0, 0, 0), g1)
        core[(w < 1e-10) | (w > 1e10)] = 1
    tr = _fill(m, _shift(tr, (0, 0, 0), [2 if a else 0 for a in m.act])[None], False)[0]
    weight = (1.0, 0.75, 0.5, 0.375)
    raw = torch.zeros_like(tr)
    core = _shift(raw, (0, 0, 0), g1)
    for o in _box(m):
        core.copy_(torch.maximum(core, weight[sum(map(abs, o))] * _shift(tr, o, g1)))
    out = torch.zeros_like(raw)
    core = _shift(out, (0, 0, 0), g1)
    core.copy_(_shift(raw, (0, 0, 0), g1))
    for o in _box(m):
        core.copy_(torch.maximum(core, 0.25 * (_shift(raw, o, g1) > 0).double()))
    return _fill(m, _shift(out, (0, 0, 0), [2 if a else 0 for a in m.act])[None], False)[0]


def _hllc(a, b, d):
    wa, wb = _prims(a), _prims(b)
    c = torch.maximum(_sound(wa) + wa[1 + d].abs(), _sound(wb) + wb[1 + d].abs())
    va, vb = wa[1 + d], wb[1 + d]
    sa, sb = torch.minimum(va, vb) - c, torch.maximum(va, vb) + c
    ra, rb = wa[0] * (va - sa), wb[0] * (sb - vb)
    vs = (rb * vb + ra * va + (wa[4] - wb[4])) / (rb + ra)
    ps = (rb * wa[4] + ra * wb[4] + ra * rb * (va - vb)) / (rb + ra)

    def star(w, u, v, s):
        return w[0] * (s - v) / (s - vs), ((s - v) * u[4] - w[4] * v + ps * vs) / (s - vs)

    (r1, e1), (r2, e2) = star(wa, a, va, sa), star(wb, b, vb, sb)

    def pick(w1, w2, w3, w4):
        return torch.where(sa > 0, w1, torch.where(vs > 0, w2, torch.where(sb > 0, w3, w4)))

    r, v = pick(wa[0], r1, r2, wb[0]), pick(va, vs, vs, vb)
    p, e = pick(wa[4], ps, ps, wb[4]), pick(a[4], e1, e2, b[4])
    f = torch.empty_like(a)
    f[0] = r * v
    for k in (1, 2, 3):
        f[k] = r * v * v + p if k == 1 + d else r * v * torch.where(vs > 0, wa[k], wb[k])
    f[4] = v * (e + p)
    return f


def _muscl(m, w, d, dt):
    """HLLC fluxes along d at the interior faces from primitives w with ghosts."""
    g1 = [1 if a else 0 for a in m.act]
    c0 = _shift(w, (0, 0, 0), g1)
    slope = []
    for e in range(3):
        if not m.act[e]:
            slope.append(torch.zeros_like(c0))
            continue
        off = [0, 0, 0]
        off[e] = 1
        c, f = m.centers[e], m.faces[e]
        up = (_shift(w, off, g1) - c0) / _along(c[2:] - c[1:-1], e)
        off[e] = -1
        dn = (c0 - _shift(w, off, g1)) / _along(c[1:-1] - c[:-2], e)
        ratio = (dn / up).clamp(max=1)
        ratio = torch.where(ratio > 0, ratio, torch.zeros_like(ratio))  # 0 / 0 gives no slope
        s = torch.where(up == 0, torch.zeros_like(up), ratio * up)
        slope.append(0.5 * s * _along(f[2:-1] - f[1:-2], e))
    v, dwt = c0[1:4], torch.zeros_like(c0)
    for e in range(3):
        q = slope[e]
        dwt[0] -= v[e] * q[0] + c0[0] * q[1 + e]
        dwt[4] -= v[e] * q[4] + GAMMA * c0[4] * q[1 + e]
        for k in range(3):
            dwt[1 + k] -= v[e] * q[1 + k]
        dwt[1 + e] -= q[4] / c0[0]
    hann = dwt * dt / _along(m.faces[d][2:-1] - m.faces[d][1:-2], d)
    wl, wr = c0 + slope[d] + hann, c0 - slope[d] + hann
    ax = 3 - d
    cut = [1 if m.act[e] and e != d else 0 for e in range(3)]
    wl, wr = _shift(wl, (0, 0, 0), cut), _shift(wr, (0, 0, 0), cut)
    n = wl.shape[ax] - 1
    return _hllc(_cons(wl.narrow(ax, 0, n)), _cons(wr.narrow(ax, 1, n)), d)


def _exact_fallback(m, u, dt):
    slices, start = _predict(m, u, dt), u
    A = _cells(m, _cv(m, u))
    g2 = [2 if a else 0 for a in m.act]
    for t in range(m.T):
        F = []
        for d in range(m.dim):
            f = _face_fluxes(m, slices[t], d)
            for e in range(m.dim):
                if e != d:
                    f = _apply(m.b["sp_to_cv"], f, 6 - e)
            body = f.narrow(6 - d, 0, m.n)
            last = f.narrow(6 - d, 0, 1).narrow(3 - d, m.N[d] + 1, 1)
            pad = [last] * m.n  # one more element that holds the last face in its first cell
            body = torch.cat([body.narrow(3 - d, 0, m.N[d] + 1), torch.cat(pad, 6 - d)], 3 - d)
            mm = list(m.N)
            for e in range(m.dim):
                body = body.narrow(3 - e, 1, mm[e] + (e == d))
            v, c, b, a, r, q, p = body.shape
            F.append(body.permute(0, 1, 4, 2, 5, 3, 6).reshape(v, c * r, b * q, a * p).narrow(3 - d, 0, m.N[d] * m.n + 1))
        slices[t] = None

        def update(F):
            r = torch.zeros_like(A)
            for d in range(m.dim):
                n = F[d].shape[3 - d] - 1
                r += (F[d].narrow(3 - d, 1, n) - F[d].narrow(3 - d, 0, n)) / _along(np.diff(m.faces[d][2:-2]), d)
            return A - m.b["wt"][t] * dt * r

        old = _fill(m, _prims(A))
        theta = _theta(m, old, _fill(m, _prims(update(F))))
        for d in range(m.dim):
            th = _shift(theta, (0, 0, 0), [0 if e == d else g2[e] for e in range(3)])
            ax = 2 - d
            n = m.N[d] * m.n + 1
            th = torch.maximum(th.narrow(ax, 1, n), th.narrow(ax, 2, n))
            f = _muscl(m, old, d, m.b["wt"][t] * dt)
            F[d] = torch.where(th > 0, F[d] + th * (f - F[d]), F[d])
        A = update(F)
    out = _cv(m, _cv(m, start), "cv_to_sp")
    back = A
    v = back.shape[0]
    back = back.reshape(v, m.N[2], m.q[2], m.N[1], m.q[1], m.N[0], m.q[0]).permute(0, 1, 3, 5, 2, 4, 6)
    inner = out
    for d in range(m.dim):
        inner = inner.narrow(3 - d, 1, m.N[d])
    inner.copy_(_cv(m, back, "cv_to_sp"))
    return out


def _exact_induction(m, B, dt):
    """One ADER step of the face fields B[d] (element, point), ghosts included."""
    w, inv = m.b["wt"], m.b["invader"]

    def edge(Bs):
        E = []
        for d in range(3):
            e1, e2 = (d + 1) % 3, (d + 2) % 3
            b1 = _apply(m.b["sp_to_fp"], Bs[e1], 5 - e2) if m.act[e2] else Bs[e1]
            b2 = _apply(m.b["sp_to_fp"], Bs[e2], 5 - e1) if m.act[e1] else Bs[e2]
            E.append(VEL[e1] * b2 - VEL[e2] * b1)
        for d in range(m.dim):
            for e in ((d + 1) % 3, (d + 2) % 3):
                lo, hi, N = E[e].select(5 - d, 0), E[e].select(5 - d, -1), m.Nt[d]
                l, r = _ghost(None, 1.0, (lo.select(2 - d, 1).clone(), hi.select(2 - d, N - 2).clone()), m.bc[d])
                hi.select(2 - d, 0).copy_(l)
                lo.select(2 - d, N - 1).copy_(r)
        for d in range(m.dim):
            for e in ((d + 1) % 3, (d + 2) % 3):
                N = m.Nt[d]
                hi, lo = E[e].select(5 - d, -1).narrow(2 - d, 0, N - 1), E[e].select(5 - d, 0).narrow(2 - d, 1, N - 1)
                up = (hi if VEL[d] > 0 else lo if VEL[d] < 0 else 0.5 * (lo + hi)).clone()
                hi.copy_(up)
                lo.copy_(up)
        return E

    def rate(E, d):
        e1, e2 = (d + 1) % 3, (d + 2) % 3
        r = torch.zeros_like(B[d])
        if m.act[e2]:
            r += _apply(m.b["dfp_to_sp"], E[e1], 5 - e2) / m.h[e2]
        if m.act[e1]:
            r -= _apply(m.b["dfp_to_sp"], E[e2], 5 - e1) / m.h[e1]
        for a in range(m.dim):  # ghost elements keep their values
            r.select(2 - a, 0).zero_()
            r.select(2 - a, m.Nt[a] - 1).zero_()
        return r

    slices = [list(B) for _ in range(m.T)]
    for k in range(m.T):
        E = [edge(s) for s in slices]
        r = [[rate(E[t], d) for d in range(3)] for t in range(m.T)]
        if k < m.T - 1:
            slices = [[B[d] - dt * sum(inv[t, q] * w[q] * r[q][d] for q in range(m.T)) for d in range(3)]
                      for t in range(m.T)]
    return [(B[d] - dt * sum(w[t] * r[t][d] for t in range(m.T)))[None, None] for d in range(3)]


def _exact_train(c, seed):
    dims, params = _net_params(c, seed)
    X, Y, idx = _train_data(c, seed)
    P, o = [], 0
    for i in range(3):
        for shape in ((dims[i + 1], dims[i]), (dims[i + 1],)):
            n = int(np.prod(shape))
            P.append(torch.from_numpy(params[o:o + n].astype(np.float64)).reshape(shape).cuda().requires_grad_())
            o += n
    mo, ve = [torch.zeros_like(q) for q in P], [torch.zeros_like(q) for q in P]
    for k in range(c["steps"]):
        x, y = X[idx[k].long()].double(), Y[idx[k].long()].double()
        for i in range(3):
            x = x @ P[2 * i].T + P[2 * i + 1]
            x = torch.nn.functional.gelu(x) if i < 2 else x
        grads = torch.autograd.grad(((x - y) ** 2).mean(), P)
        with torch.no_grad():
            for q, g, a, b in zip(P, grads, mo, ve):
                a.mul_(0.9).add_(g, alpha=0.1)
                b.mul_(0.999).addcmul_(g, g, value=0.001)
                q -= LR * (a / (1 - 0.9 ** (k + 1))) / ((b / (1 - 0.999 ** (k + 1))).sqrt() + 1e-8)
    return torch.cat([q.detach().reshape(-1) for q in P]).cpu().numpy()


def _kh_run(m, amp, v1):
    """Cell averages of the driver's Kelvin-Helmholtz problem, by Gauss quadrature of each cell."""
    q, w = _gauss(m.n)
    fx = m.b["x_fp"]
    x, y = ((np.arange(-1, m.N[d] + 1)[:, None, None] + fx[None, :-1, None]
             + q[None, None, :] * np.diff(fx)[None, :, None]) * m.h[d] for d in range(2))
    inner = ((y > 0.25) & (y < 0.75)).astype(float) @ w
    s2 = 2 * (0.05 / math.sqrt(2.0)) ** 2
    ys = (np.exp(-(y - 0.25) ** 2 / s2) + np.exp(-(y - 0.75) ** 2 / s2)) @ w
    xs = np.sin(4 * math.pi * x) @ w
    one = np.ones(m.shape()[2:])

    def along_y(v):
        return v[None, :, None, None, :, None] * one

    out = np.zeros(m.shape()[1:])[:5]
    out[0], out[1], out[4] = along_y(1 + inner), along_y(v1 * (2 * inner - 1)), 2.5 * one
    out[2] = amp * along_y(ys) * xs[None, None, :, None, None, :]
    return torch.from_numpy(out).cuda()


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_train(case, seed)
    if kind == "driver":
        s = prepare(case, seed)
        m = _Mesh(case)
        w = _kh_run(m, s["amp"], s["v1"])
        u = _cons(_cv(m, w, "cv_to_sp"))
        cell = w.narrow(2, 1, m.N[1]).narrow(3, 1, m.N[0])
        speed = sum(cell[1 + d].abs() + _sound(cell) for d in range(2))
        dt, t = float(CFL * min(m.h[:2]) / speed.max() / m.n), 0.0
        for _ in range(case["steps"]):
            u = _exact_fallback(m, u, dt)
            t += dt
            out = _finish(m, u)
            dt = out["dt"]
        return {"W_cv": out["W_cv"].reshape(-1).cpu().numpy(), "t": t, "steps": None}
    m = _Mesh(case, case.get("integ", "ader") == "ader")
    if kind == "induction":
        b, dt = _field(m, seed)
        return _exact_induction(m, [v[0, 0] for v in b], dt)
    u, dt = _flow(m, seed)
    u = u[0, :5].contiguous()
    if kind == "fallback":
        return _finish(m, _exact_fallback(m, u, dt))
    return _finish(m, _exact_step(m, u, dt, case["integ"]))
