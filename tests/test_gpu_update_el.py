"""update_prediction and update_solution on whole elements against the oracle,
bit for bit: every degree and dimensionality of the element form and the axis
orders it leaves to the per-point kernels, ragged last workgroups, gravity
(whose source reads the variables written before), SSP-RK's single slice, and
fluxes with exact zeros, magnitudes near the smallest normal number,
infinities and NaN, where a division by the element width is redone."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402,F401
from test_gpu_stages import ctx_for, dev, host, sd_shape, state  # noqa: E402

CASES = [((1, 0, 0), (37, 1, 1), p) for p in (1, 4, 8)] + [((1, 1, 0), (5, 3, 1), p) for p in (1, 2, 3, 6, 8)] + \
        [((1, 1, 1), (3, 2, 2), p) for p in (1, 2, 3, 4, 5)] + [((1, 1, 1), (2, 1, 1), p) for p in (6, 7, 8)] + \
        [((1, 0, 1), (3, 1, 4), 3)]


@pytest.mark.parametrize("act,N,p", CASES)
@pytest.mark.parametrize("g", [(0.0, 0.0, 0.0), (0.1, -0.7, 0.3)])
@pytest.mark.parametrize("values", ["ordinary", "tiny", "nonfinite"])
def test_update(act, N, p, g, values):
    rng = np.random.default_rng(p + 10 * sum(act))
    c, m, _, _ = ctx_for(p, act, N=N, g=g)
    n, T = p + 1, p + 1
    s_a, s_u = sd_shape(T, 6, N, n, act), sd_shape(1, 6, N, n, act)
    U, Ua = state(s_u, rng), state(s_a, rng)
    F = [np.ascontiguousarray(rng.normal(size=sd_shape(T, 6, N, n, act, stag=d))) if act[d]
         else np.zeros(s_a) for d in range(3)]
    if values == "tiny":  # one variable tiny throughout, one zero, one mixed
        U[:, 2] = Ua[:, 2] = 0.0
        for f in F:
            f[:, 2] *= 10.0 ** rng.uniform(-309, -285, size=f[:, 2].shape)
            f[:, 3] = 0.0
            f[:, 1] *= 10.0 ** rng.uniform(-320, 3, size=f[:, 1].shape)
    if values == "nonfinite":
        for f in F:
            for x in (np.inf, -np.inf, np.nan):
                f.flat[int(rng.integers(0, f.size))] = x
    h = np.array([1.0 / N[d] if act[d] else 1.0 for d in range(3)])
    cfg = op.OrcCfg.make(act=act, g=g)
    shapes, dt = [op.ip(f.shape) for f in F], 0.0123
    Fg = [dev(f) if act[d] else None for d, f in enumerate(F)]
    with np.errstate(all="ignore"):
        Ua_o = Ua.copy()
        op.orc().orc_predict(ctypes.byref(cfg), op.dp(U), op.ip(s_u), op.dp(Ua_o), op.ip(s_a), op.dp(F[0]), shapes[0],
                             op.dp(F[1]), shapes[1], op.dp(F[2]), shapes[2], op.dp(m["dfp_to_sp"]), n, n + 1,
                             op.dp(m["invader"]), op.dp(m["wt"]), op.dp(h), ctypes.c_double(dt))
        Ua_g = dev(Ua)
        c.update_prediction(dev(U), Ua_g, Fg[0], Fg[1], Fg[2], p + 2, dt)
        assert np.array_equal(host(Ua_g), Ua_o, equal_nan=True)
        U_o = U.copy()
        op.orc().orc_correct(ctypes.byref(cfg), op.dp(U_o), op.ip(s_u), op.dp(Ua), op.ip(s_a), op.dp(F[0]), shapes[0],
                             op.dp(F[1]), shapes[1], op.dp(F[2]), shapes[2], op.dp(m["dfp_to_sp"]), n, n + 1,
                             op.dp(m["wt"]), op.dp(h), ctypes.c_double(dt))
        U_g = dev(U)
        c.update_solution(U_g, dev(Ua), Fg[0], Fg[1], Fg[2], p + 2, dt)
        assert np.array_equal(host(U_g), U_o, equal_nan=True)
    c.close()


@pytest.mark.parametrize("act,N,p", [((1, 0, 0), (37, 1, 1), 3), ((1, 1, 0), (5, 3, 1), 3), ((1, 1, 1), (3, 2, 2), 3),
                                     ((1, 1, 1), (2, 1, 1), 7)])
def test_update_subnormal_on_wide_elements(act, N, p):
    """Fluxes of a few units of 2^-1074 on elements wider than 1, where a quotient
    formed without division can be zero though its numerator is not."""
    rng = np.random.default_rng(40 + p + sum(act))
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"]
    h = np.array([1.9, 1.3, 1.7])
    c = sk.Context(p, act, (0, 0, 0), p + 1, ops, h=h)
    n, T = p + 1, p + 1
    s_a, s_u = sd_shape(T, 6, N, n, act), sd_shape(1, 6, N, n, act)
    U, Ua = np.zeros(s_u), np.zeros(s_a)
    F = [np.zeros(sd_shape(T, 6, N, n, act, stag=d)) for d in range(3)]
    for d in range(3):
        if act[d]:  # variable v: up to 2^v units
            for v in range(6):
                F[d][:, v] = rng.integers(-2 ** v, 2 ** v + 1, size=F[d][:, v].shape) * 5e-324
    cfg = op.OrcCfg.make(act=act)
    shapes, dt = [op.ip(f.shape) for f in F], 50.0
    Fg = [dev(f) if act[d] else None for d, f in enumerate(F)]
    Ua_o, U_o = Ua.copy(), U.copy()
    op.orc().orc_predict(ctypes.byref(cfg), op.dp(U), op.ip(s_u), op.dp(Ua_o), op.ip(s_a), op.dp(F[0]), shapes[0],
                         op.dp(F[1]), shapes[1], op.dp(F[2]), shapes[2], op.dp(m["dfp_to_sp"]), n, n + 1,
                         op.dp(m["invader"]), op.dp(m["wt"]), op.dp(h), ctypes.c_double(dt))
    op.orc().orc_correct(ctypes.byref(cfg), op.dp(U_o), op.ip(s_u), op.dp(Ua), op.ip(s_a), op.dp(F[0]), shapes[0],
                         op.dp(F[1]), shapes[1], op.dp(F[2]), shapes[2], op.dp(m["dfp_to_sp"]), n, n + 1,
                         op.dp(m["wt"]), op.dp(h), ctypes.c_double(dt))
    assert (U_o != 0).mean() > 0.5
    Ua_g, U_g = dev(Ua), dev(U)
    c.update_prediction(dev(U), Ua_g, Fg[0], Fg[1], Fg[2], p + 2, dt)
    c.update_solution(U_g, dev(Ua), Fg[0], Fg[1], Fg[2], p + 2, dt)
    assert np.array_equal(host(Ua_g), Ua_o)
    assert np.array_equal(host(U_g), U_o)
    c.close()
