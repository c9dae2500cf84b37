"""Mixed-precision steps against the FP64 fused step for every tile variant, on
meshes whose element counts leave idle lanes, waves and workgroups: boundary
types, gravity, the residual form with partly converged meshes, and the three
forms of the face integrals against each other.

Tolerance: the state is carried as FP32 deviations of size A inside an element
(A <= 0.2 here); an update chains interpolations, divergences and time
contractions of at most N + 1 terms with operator norms below 64 / (dt/h
included), so 64 (N + 1) 2^-24 A bounds it, times the sweeps' contraction < 2."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import dev, host, sd_shape  # noqa: E402

A = 0.2


class Picard(ctypes.Structure):
    _fields_ = [("residual", ctypes.c_int), ("guess", ctypes.c_int), ("tol", ctypes.c_double),
                ("max_sweeps", ctypes.c_int), ("guess_keep", ctypes.c_int)]


class Stats(ctypes.Structure):
    _fields_ = [("steps", ctypes.c_longlong), ("fallbacks", ctypes.c_longlong), ("sweeps", ctypes.c_double),
                ("last_residual", ctypes.c_double)]


def ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def context(p, act, bc, N, g=(0, 0, 0)):
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"]
    return sk.Context(p, act, bc, p + 1, ops, h=[1.0 / N[d] if act[d] else 1.0 for d in range(3)], g=g)


def state(N, n, act, rng, flat=0.0):
    """Conserved variables with deviations of at most A / 2 about a uniform state; the
    first `flat` of the elements along x hold the uniform state alone."""
    s = sd_shape(1, 6, N, n, act)
    U = np.empty(s)
    for v, (b, a) in enumerate([(1.0, A / 2), (0.3, A / 2), (-0.2, A / 2), (0.1, A / 2), (3.0, A / 2), (0.0, 0.0)]):
        U[0, v] = b + a * rng.uniform(-1, 1, s[2:])
        U[0, v, :, :, : int(flat * s[4])] = b
    return dev(U)


def workspace(c, U):
    N = (ctypes.c_int * 3)(U.shape[4], U.shape[3], U.shape[2])
    return torch.empty(sk.lib().spdk_mixed_workspace_bytes(c.ctx, N), dtype=torch.uint8, device="cuda")


def mixed(c, U, dt, W, pc=None):
    out, st, ws = ctypes.c_double(), Stats(), workspace(c, U)
    sk.check(sk.lib().spdk_hydro_step_mixed(c.ctx, ptr(U), sk.SDShape.of(U.shape), ptr(ws), ctypes.c_double(dt), ptr(W),
                                            None, ctypes.byref(pc) if pc else None, ctypes.byref(st),
                                            ctypes.byref(out)), "hydro_step_mixed")
    return out.value, st


def inner(x, act):
    """The interior elements: no interior element reads a ghost element, whose
    residual is not tested, so in the residual form ghosts may stop early."""
    return x[(slice(None), slice(None)) + tuple(slice(1, -1) if act[d] else slice(None) for d in (2, 1, 0))].contiguous()


MESHES = [((1, 0, 0), N, p) for p, N in [(1, (1, 1, 1)), (1, (190, 1, 1)), (2, (83, 1, 1)), (3, (62, 1, 1)),
                                         (4, (47, 1, 1))]] + \
         [((1, 1, 0), N, p) for p, N in [(1, (7, 5, 1)), (2, (6, 3, 1)), (3, (5, 1, 1)), (4, (7, 2, 1)), (4, (1, 1, 1))]] + \
         [((1, 1, 1), N, p) for p, N in [(1, (3, 2, 4)), (2, (2, 3, 1)), (3, (3, 2, 2)), (3, (1, 1, 1))]]


@pytest.mark.parametrize("act,N,p", MESHES)
@pytest.mark.parametrize("bc,g", [((0, 0, 0), (0, 0, 0)), ((1, 2, 0), (0, 0, 0)), ((2, 1, 2), (0.1, -0.2, 0.3))])
def test_step(act, N, p, bc, g):
    rng = np.random.default_rng(10 * p + sum(act))
    tol = 2 * 64 * (p + 2) * 2.0 ** -24 * A
    dt = 0.02 / max(N) / (p + 1)
    c = context(p, act, bc, N, g)
    U = state(N, p + 1, act, rng)
    a, b, r = U.clone(), U.clone(), U.clone()
    Wa, Wb = torch.zeros_like(U), torch.zeros_like(U)
    dta = c.hydro_step_fused(a, dt, Wa)
    dtb, _ = mixed(c, b, dt, Wb)
    assert float((a - U).abs().max()) > 100 * tol  # the step moves the state by far more
    assert float((a - b).abs().max()) < tol
    assert float((Wa - Wb).abs().max()) < 20 * tol  # velocities and pressure of the new state
    assert abs(dta - dtb) < 20 * tol * dta
    # never converged: the fixed count, sweep by sweep
    mixed(c, r, dt, None, Picard(1, 0, 1e-30, 0, 0))
    assert np.array_equal(host(inner(b, act)), host(inner(r, act)))
    c.close()


@pytest.mark.parametrize("act,N,p", [((1, 0, 0), (90, 1, 1), 4), ((1, 1, 0), (9, 7, 1), 4), ((1, 1, 1), (9, 2, 3), 3),
                                     ((1, 1, 1), (7, 3, 2), 2)])
def test_partly_converged(act, N, p):
    rng = np.random.default_rng(p)
    tol = 2 * 64 * (p + 2) * 2.0 ** -24 * A
    dt = 0.02 / max(N) / (p + 1)
    c = context(p, act, (0, 0, 0), N)
    U = state(N, p + 1, act, rng, flat=0.6)
    a, b = U.clone(), U.clone()
    c.hydro_step_fused(a, dt, None)
    _, st = mixed(c, b, dt, None, Picard(1, 0, 1e-12, 0, 0))
    assert 2.0 < st.sweeps < p + 1  # the uniform elements stopped early
    assert float(inner(a - b, act).abs().max()) < tol
    c.close()


@pytest.mark.parametrize("N", [(1, 1, 1), (3, 2, 2), (6, 1, 3)])
@pytest.mark.parametrize("bc", [(0, 0, 0), (1, 2, 0), (2, 1, 2)])
def test_face_integrals(N, bc):
    """3-D p = 3: the staged form, the unstaged one (with the x flux points) and the
    vector one write the same faces."""
    p, act = 3, (1, 1, 1)
    n = p + 1
    c = context(p, act, bc, N)
    U = state(N, n, act, np.random.default_rng(7))
    cells = [n * N[d] + 4 for d in range(3)]
    fv = sk.FVShape.of((6, cells[2], cells[1], cells[0]))
    E = U.shape[2] * U.shape[3] * U.shape[4]
    got = []
    for fx, valu in [(False, 0), (True, 0), (False, 1)]:
        F = [torch.full((6, cells[2] + (d == 2), cells[1] + (d == 1), cells[0] + (d == 0)), 7e7, dtype=torch.float64,
                        device="cuda") for t in range(n) for d in range(3)]
        Fx = torch.zeros(n * 6 * E * n * n * (n + 1), dtype=torch.float64, device="cuda") if fx else None
        P = (ctypes.c_void_p * len(F))(*[f.data_ptr() for f in F])
        st, ws, pc = Stats(), workspace(c, U), Picard(0, 0, 0.0, 0, 0)
        sk.check(sk.lib().spdk_mixed_predict_fv_fluxes(c.ctx, ptr(U), sk.SDShape.of(U.shape), ptr(ws),
                                                       ctypes.c_double(1e-4), ctypes.byref(pc), ctypes.byref(st), P, fv,
                                                       ptr(Fx), valu), "mixed_predict_fv_fluxes")
        got.append([host(f) for f in F])
    for f, g, h in zip(*got):
        assert np.array_equal(f == 7e7, g == 7e7) and np.array_equal(f == 7e7, h == 7e7)
        assert (f[:5] != 7e7).sum() > 0
        assert np.array_equal(f, g)
        # 16-term FP32 contractions of deviations below 64 A
        assert np.abs(f - h).max() < 64 * A * 17 * 2.0 ** -24
    c.close()
