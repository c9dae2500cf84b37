"""Whole fused FP64 steps against the stage entries they fuse, bit for bit: ADER
and SSP-RK 1 to 3, every boundary type, gravity, meshes from one element per
axis to ragged last workgroups, and states with constants, exact zeros of both
signs and momenta near the smallest normal numbers (where the divisions by the
element width are redone)."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import dev, host, sd_shape, state  # noqa: E402


def stages(c, U, p, T, act, shapes, dt, rk):
    z = lambda s: torch.zeros(s, dtype=torch.float64, device="cuda")
    Ua, U0, W, Wc, tmp = z((T,) + tuple(U.shape[1:])), U.clone(), z(U.shape), z(U.shape), z(U.shape)
    Uf, F = [z(s) if a else None for s, a in zip(shapes, act)], [z(s) if a else None for s, a in zip(shapes, act)]
    dims = [d for d in range(3) if act[d]]

    def fluxes():
        for d in dims:
            c.transform_a_to_b_1d(Ua, Uf[d], sk.SPDK_M_SP_TO_FP, d)
            c.compute_fluxes(Uf[d], F[d], d)
            c.boundaries(Uf[d], d)
            c.sd_riemann_solver(Uf[d], F[d], d)

    if rk == 0:
        c.copy_ader(U, Ua)
        for k in range(T):
            fluxes()
            if k < T - 1:
                c.update_prediction(U, Ua, F[0], F[1], F[2], p + 2, dt)
        c.update_solution(U, Ua, F[0], F[1], F[2], p + 2, dt)
    for a in {0: (), 1: (0.0,), 2: (0.0, 0.5), 3: (0.0, 0.75, 1.0 / 3.0)}[rk]:
        c.copy_ader(U, Ua)
        fluxes()
        c.update_solution(U, Ua, F[0], F[1], F[2], p + 2, dt)
        if a > 0:
            c.combine_solution(U, U0, a)
    c.compute_primitives(U, W)
    c.transform_a_to_b(W, Wc, tmp, sk.SPDK_M_SP_TO_CV)
    return Wc, c.compute_dt(Wc)


MESHES = [((1, 0, 0), (1, 1, 1), 4), ((1, 0, 0), (23, 1, 1), 3), ((1, 0, 0), (40, 1, 1), 1), ((1, 1, 0), (1, 2, 1), 3),
          ((1, 1, 0), (7, 5, 1), 1), ((1, 1, 0), (6, 7, 1), 2), ((1, 1, 0), (5, 3, 1), 4), ((1, 1, 1), (1, 1, 1), 3),
          ((1, 1, 1), (3, 2, 4), 1), ((1, 1, 1), (2, 3, 2), 2), ((1, 1, 1), (3, 1, 2), 3)]


@pytest.mark.parametrize("act,N,p", MESHES)
@pytest.mark.parametrize("rk", [0, 1, 2, 3])
@pytest.mark.parametrize("bc,g", [((0, 0, 0), (0, 0, 0)), ((1, 2, 0), (0, 0, 0)), ((2, 1, 2), (0.1, -0.2, 0.3))])
def test_step(act, N, p, rk, bc, g):
    rng = np.random.default_rng(100 * p + 10 * rk + sum(act))
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"] if rk == 0 else np.ones(1)
    if rk:
        ops["invader"] = np.ones((1, 1))
    T = p + 1 if rk == 0 else 1
    h = [1.7 / (N[d] + 2) if act[d] else 1.0 for d in range(3)]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = sk.Context(p, act, bc, T, ops, h=h, g=g, rk_order=rk)
        U = state(sd_shape(1, 6, N, p + 1, act), rng)
        U[0, 3] *= 10.0 ** rng.uniform(-309, -285, size=U[0, 3].shape)
        U[0, 2, ..., 0] = 0.0
        U[0, 1, ..., -1] = -0.0
        U[0, :, :, :, : U.shape[4] // 2] = U[0, :, :1, :1, :1, :1, :1, :1]  # constant elements
        a, b = dev(U), dev(U)
        Wb = torch.full(U.shape, float("nan"), dtype=torch.float64, device="cuda")
        shapes = [sd_shape(T, 6, N, p + 1, act, stag=d) for d in range(3)]
        Wa, dta = stages(c, a, p, T, act, shapes, 1e-3, rk)
        dtb = c.hydro_step_fused(b, 1e-3, Wb)
        x, y = host(a), host(b)
        assert np.isfinite(x).all()
        assert np.array_equal(x, y), f"U: {int((x != y).sum())} of {x.size} differ"
        assert np.array_equal(host(Wa), host(Wb))
        assert dta == dtb
        c.close()


@pytest.mark.parametrize("act,N,p", [((1, 0, 0), (23, 1, 1), 3), ((1, 1, 0), (6, 7, 1), 2), ((1, 1, 1), (3, 2, 2), 3)])
@pytest.mark.parametrize("rk", [0, 1])
def test_step_subnormal_on_wide_elements(act, N, p, rk):
    """A momentum of a few units of 2^-1074 on elements wider than 1, and a state that is constant elsewhere: sums that
    are zero, with and without terms whose quotients are inexact."""
    rng = np.random.default_rng(70 + p + sum(act))
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"] if rk == 0 else np.ones(1)
    if rk:
        ops["invader"] = np.ones((1, 1))
    T = p + 1 if rk == 0 else 1
    c = sk.Context(p, act, (0, 0, 0), T, ops, h=[1.9, 1.3, 1.7], rk_order=rk)
    U = np.zeros(sd_shape(1, 6, N, p + 1, act))
    U[0, 0], U[0, 4], U[0, 1] = 1.0, 2.5, 1.0
    U[0, 3] = rng.integers(-8, 9, size=U[0, 3].shape) * 5e-324
    U[0, 2, ..., : U.shape[4] // 2, :, :, :] = 0.25  # and velocity along y in half of the elements along x
    a, b = dev(U), dev(U)
    Wb = torch.full(U.shape, float("nan"), dtype=torch.float64, device="cuda")
    shapes = [sd_shape(T, 6, N, p + 1, act, stag=d) for d in range(3)]
    Wa, dta = stages(c, a, p, T, act, shapes, 1.0, rk)
    dtb = c.hydro_step_fused(b, 1.0, Wb)
    x, y = host(a), host(b)
    assert np.isfinite(x).all() and (x[0, 3] != U[0, 3]).any()
    assert np.array_equal(x, y), f"U: {int((x != y).sum())} of {x.size} differ"
    assert np.array_equal(host(Wa), host(Wb))
    assert dta == dtb
    c.close()


@pytest.mark.parametrize("T", [2, 3, 5, 8, 10])
def test_other_slice_counts_are_refused(T):
    """The kernels are compiled for p+1 slices or one: every fused entry of a
    context with another count returns its error before any launch."""
    p, act, N = 3, (1, 1, 1), (2, 3, 2)
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"], ops["invader"] = np.ones(T), np.ones((T, T))
    c = sk.Context(p, act, (0, 0, 0), T, ops, h=[0.5, 0.5, 0.5])
    L, E_CONFIG = sk.lib(), -5
    s, sa = sd_shape(1, 6, N, p + 1, act), sd_shape(T, 6, N, p + 1, act)
    Ne = (ctypes.c_int * 3)(s[4], s[3], s[2])
    assert L.spdk_fused_workspace_bytes(c.ctx, Ne) == 0
    assert L.spdk_fused_fluxes_workspace_bytes(c.ctx, Ne) == 0
    U = torch.ones(s, dtype=torch.float64, device="cuda")
    b = torch.zeros(64, dtype=torch.float64, device="cuda")  # any non-null address: nothing may touch it
    u, q, ss, ssa, dt = ctypes.c_void_p(U.data_ptr()), ctypes.c_void_p(b.data_ptr()), sk.SDShape.of(s), sk.SDShape.of(sa), \
        ctypes.c_double(1e-3)
    fv = sk.FVShape.of((6,) + tuple(N[d] * (p + 1) + 4 for d in (2, 1, 0)))
    faces = (ctypes.c_void_p * (3 * T))(*[b.data_ptr()] * (3 * T))
    assert L.spdk_hydro_step_fused(c.ctx, u, ss, q, dt, None, None, None) == E_CONFIG
    assert L.spdk_hydro_step_fused_noalloc(c.ctx, u, ss, dt, None, None, None) == E_CONFIG
    assert L.spdk_fused_predict(c.ctx, u, ss, q, dt, q, ssa) == E_CONFIG
    assert L.spdk_fused_predict_fluxes(c.ctx, u, ss, q, dt, q, q, q, ssa) == E_CONFIG
    assert L.spdk_fused_predict_fv_fluxes(c.ctx, u, ss, q, dt, faces, fv, None, ssa) == E_CONFIG
    assert L.spdk_fused_fluxes(c.ctx, q, ssa, q, q, q, q) == E_CONFIG
    assert (host(U) == 1).all() and (host(b) == 0).all()
    c.close()
