"""Trouble detection, theta and the fallback fluxes against the oracle, bit for
bit, at the edges of their tiles (60-cell rows of the theta masks, 8 x 8 x 4
and 16 x 16 fallback tiles, 8-cell columns of the detection) and on values
where a division by a grid width leaves the normal range: exact zeros of both
signs, magnitudes near the smallest normal number, infinities and NaN."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402,F401
from test_gpu_stages import ctx_for, dev, fv_shape, host, state  # noqa: E402

MESHES = [((1, 0, 0), (14, 1, 1)), ((1, 0, 0), (15, 1, 1)), ((1, 0, 0), (31, 1, 1)), ((1, 1, 0), (15, 1, 1)),
          ((1, 1, 0), (16, 9, 1)), ((1, 1, 0), (31, 4, 1)), ((1, 1, 1), (2, 1, 1)), ((1, 1, 1), (15, 2, 3)),
          ((1, 1, 1), (16, 5, 2))]


def setup(act, N, seed, **opts):
    c, _, faces, centers = ctx_for(3, act, N=N, **{k: bool(v) for k, v in opts.items()})
    cfg = op.OrcCfg.make(act=act, p=3, **opts)
    geo = ((ctypes.POINTER(ctypes.c_double) * 3)(*[op.dp(x) for x in centers]),
           (ctypes.POINTER(ctypes.c_double) * 3)(*[op.dp(x) for x in faces]),
           (ctypes.c_int * 3)(*[len(x) for x in centers]))
    return c, cfg, geo, (faces, centers), fv_shape(6, N, 4, act), np.random.default_rng(seed)


def same(a, b):
    return np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("act,N", MESHES)
@pytest.mark.parametrize("density", [0.0, 0.01, 0.4, -1.0])
def test_theta(act, N, density):
    """Troubles 0 or 1 at several densities; density -1: other values among them (the cell-by-cell form)."""
    c, cfg, _, _, s_fv, rng = setup(act, N, 5)
    tr = np.zeros(s_fv)
    tr[5] = rng.uniform(size=s_fv[1:]) < abs(density) * (0.05 if density < 0 else 1)
    if density < 0:
        tr[5].flat[rng.integers(0, tr[5].size, 3)] = [0.5, -2.0, 3.0]
    s_th = (1,) + s_fv[1:]
    tmp_o, th_o = np.zeros(s_th), np.zeros(s_th)
    op.orc().orc_blend(ctypes.byref(cfg), op.dp(tr), op.dp(tmp_o), op.dp(th_o), op.ip(s_fv))
    tmp, th = torch.zeros(s_th, dtype=torch.float64, device="cuda"), torch.zeros(s_th, dtype=torch.float64, device="cuda")
    c.blend_theta(dev(tr), tmp, th)
    assert same(host(th), th_o)
    c.close()


def special(W, rng, nonfinite):
    """Blocks of constants, zero velocities of both signs, and fields near the smallest normal numbers."""
    n = W.shape[-1]
    W[0, ..., : n // 3] = 1.0
    W[4, ..., : n // 3] = 2.5
    W[1, ..., n // 4: n // 2] = 0.0
    W[2, ..., n // 2:] = -0.0
    W[3] *= 10.0 ** rng.uniform(-309, -280, size=W[3].shape)
    W[5] = 0.0
    if nonfinite:
        for v, x in ((1, np.inf), (3, -np.inf), (2, np.nan), (4, np.inf)):
            W[v].flat[int(rng.integers(0, W[v].size))] = x
    return np.ascontiguousarray(W)


@pytest.mark.parametrize("act,N", MESHES)
@pytest.mark.parametrize("opts", [{}, {"nad_delta": 1}, {"nad_moore": 0}])
def test_detection(act, N, opts):
    c, cfg, geo, _keep, s_fv, rng = setup(act, N, 11, **opts)
    Wo = special(state((1,) + s_fv, rng)[0], rng, False)
    Wn = np.ascontiguousarray(Wo * (1 + 1e-3 * rng.normal(size=Wo.shape) * (rng.uniform(size=Wo.shape) < 0.5)))
    mask = 0b11011  # the tiny field and the zeros among the detected ones
    tr_o, al = np.zeros(s_fv), [np.zeros(s_fv) for _ in range(3)]
    op.orc().orc_detect(ctypes.byref(cfg), op.dp(Wn), op.dp(Wo), op.dp(tr_o), *[op.dp(a) for a in al], op.ip(s_fv),
                        *geo, 1, mask)
    z = lambda: torch.zeros(s_fv, dtype=torch.float64, device="cuda")
    tr, ga = z(), [z() for _ in range(3)]
    c.detect_troubles(dev(Wn), dev(Wo), tr, *ga, 1, mask)
    assert same(host(tr), tr_o)
    for d in range(3):
        if act[d]:
            assert same(host(ga[d]), al[d]), d
    tr, bits = z(), torch.zeros(s_fv[1:], dtype=torch.int16, device="cuda")
    c.detect_troubles_bits(dev(Wn), dev(Wo), tr, bits, 1, mask)
    assert same(host(tr), tr_o)
    c.close()


@pytest.mark.parametrize("act,N", MESHES)
@pytest.mark.parametrize("nonfinite", [False, True])
def test_fallback(act, N, nonfinite):
    c, cfg, geo, _keep, s_fv, rng = setup(act, N, 17)
    W = special(state((1,) + s_fv, rng)[0], rng, nonfinite)
    th = np.where(rng.uniform(size=(1,) + s_fv[1:]) < 0.3, rng.choice([0.25, 0.5, 1.0], size=(1,) + s_fv[1:]), 0.0)
    if act[0] and s_fv[3] > 40:
        th[..., 25:38] = 0.0  # tiles without a blended face
    Fs = [np.ascontiguousarray(rng.normal(size=fv_shape(6, N, 4, act, stag=d))) for d in range(3)]
    Fo = [f.copy() for f in Fs]
    op.orc().orc_fallback(ctypes.byref(cfg), op.dp(W), op.dp(th), *[op.dp(f) for f in Fo], op.ip(s_fv), *geo,
                          ctypes.c_double(1e-3))
    Fg = [dev(f) for f in Fs]
    c.fallback_fluxes(dev(W), dev(th), Fg[0], Fg[1] if act[1] else None, Fg[2] if act[2] else None, 1e-3)
    for d in range(3):
        if act[d]:
            got, skip = host(Fg[d]), np.zeros(Fo[d].shape[1:], bool)
            if nonfinite:
                # with theta = 0 the oracle still forms 0 * (F_HLLC - F), which is NaN for a non-finite flux; such
                # faces are left alone here
                t = th[0]
                lo = np.roll(t, 1, axis=2 - d)
                f0 = np.maximum(t, lo) == 0
                pad = [(0, a - b) for a, b in zip(Fo[d].shape[1:], f0.shape)]
                skip = np.pad(f0, pad, constant_values=True)
            ok = (got == Fo[d]) | (np.isnan(got) & np.isnan(Fo[d])) | skip
            assert ok.all(), (d, int((~ok).sum()))
    c.close()


def wide(act, N, seed):
    """As setup, on cells 1.9 wide, with a field that grows by 4 or no units of 2^-1074 from cell to cell."""
    p, faces, centers = 3, [], []
    for d in range(3):
        f = 1.9 * np.arange(4 * N[d] + 5) if act[d] else np.array([-1.0, 0.0])
        faces.append(f)
        centers.append(0.5 * (f[1:] + f[:-1]) if act[d] else np.array([-1.0]))
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"], ops["fv_faces"], ops["fv_centers"] = m["wt"], faces, centers
    c = sk.Context(p, act, (0, 0, 0), p + 1, ops, h=[7.6] * 3)
    geo = ((ctypes.POINTER(ctypes.c_double) * 3)(*[op.dp(x) for x in centers]),
           (ctypes.POINTER(ctypes.c_double) * 3)(*[op.dp(x) for x in faces]),
           (ctypes.c_int * 3)(*[len(x) for x in centers]))
    rng, s_fv = np.random.default_rng(seed), fv_shape(6, N, 4, act)
    W = np.zeros(s_fv)
    W[0], W[4], W[1] = 1.0, 2.5, 1.0
    for d in range(3):
        if act[d]:
            step = 4 * rng.integers(0, 2, size=s_fv[3 - d])
            W[3] += np.cumsum(step).reshape([-1 if a == 2 - d else 1 for a in range(3)]) * 5e-324
    return c, op.OrcCfg.make(act=act, p=p), geo, (faces, centers), s_fv, W, rng


@pytest.mark.parametrize("act,N", MESHES)
def test_detection_subnormal_on_wide_cells(act, N):
    c, cfg, geo, _keep, s_fv, Wn, rng = wide(act, N, 23)
    Wo = Wn.copy()
    Wo[3] = rng.integers(0, 7, size=s_fv[1:]) * 5e-324
    tr_o, al = np.zeros(s_fv), [np.zeros(s_fv) for _ in range(3)]
    op.orc().orc_detect(ctypes.byref(cfg), op.dp(Wn), op.dp(Wo), op.dp(tr_o), *[op.dp(a) for a in al], op.ip(s_fv),
                        *geo, 1, 0b01000)
    z = lambda: torch.zeros(s_fv, dtype=torch.float64, device="cuda")
    tr, ga = z(), [z() for _ in range(3)]
    c.detect_troubles(dev(Wn), dev(Wo), tr, *ga, 1, 0b01000)
    for d in range(3):
        if act[d]:
            assert same(host(ga[d]), al[d]), d
    assert same(host(tr), tr_o)
    tr, bits = z(), torch.zeros(s_fv[1:], dtype=torch.int16, device="cuda")
    c.detect_troubles_bits(dev(Wn), dev(Wo), tr, bits, 1, 0b01000)
    assert same(host(tr), tr_o)
    c.close()


@pytest.mark.parametrize("act,N", MESHES + [((1, 0, 1), (9, 1, 5))])  # the last: one thread per cell
def test_fallback_subnormal_on_wide_cells(act, N):
    c, cfg, geo, _keep, s_fv, W, rng = wide(act, N, 29)
    th = np.ones((1,) + s_fv[1:])
    Fs = [np.zeros(fv_shape(6, N, 4, act, stag=d)) for d in range(3)]
    Fo = [f.copy() for f in Fs]
    op.orc().orc_fallback(ctypes.byref(cfg), op.dp(W), op.dp(th), *[op.dp(f) for f in Fo], op.ip(s_fv), *geo,
                          ctypes.c_double(0.5))
    Fg = [dev(f) for f in Fs]
    c.fallback_fluxes(dev(W), dev(th), Fg[0], Fg[1] if act[1] else None, Fg[2] if act[2] else None, 0.5)
    assert (Fo[0][3] != 0).any()
    for d in range(3):
        if act[d]:
            assert same(host(Fg[d]), Fo[d]), d
    c.close()


@pytest.mark.parametrize("act", [(1, 1, 0), (1, 1, 1)])
def test_axes_without_coordinates_take_those_of_x(act):
    """A context given the FV coordinates of x alone, on a mesh of equal axes, against one given every axis'."""
    N, p, m = [5 if a else 1 for a in act], 3, op.matrices(3)
    xs = [op.fv_geometry(5, p) if a else (np.array([-1.0, 0.0]), np.array([-1.0])) for a in act]
    s_fv, rng = fv_shape(6, N, 4, act), np.random.default_rng(31)
    W = state((1,) + s_fv, rng)[0]
    Wo = np.ascontiguousarray(W * (1 + 1e-2 * rng.normal(size=W.shape)))
    th = rng.choice([0.0, 0.25, 1.0], size=(1,) + s_fv[1:])
    Fs = [rng.normal(size=fv_shape(6, N, 4, act, stag=d)) for d in range(3)]
    out = []
    for own in (True, False):
        ops = {k: m[k] for k in sk.Context.MATS}
        ops["wt"] = m["wt"]
        ops["fv_faces"], ops["fv_centers"] = [[x[q] if own or d == 0 else None for d, x in enumerate(xs)] for q in (0, 1)]
        c = sk.Context(p, act, (0, 0, 0), p + 1, ops, h=[0.2] * 3)
        z = lambda: torch.zeros(s_fv, dtype=torch.float64, device="cuda")
        tr, al, tb = z(), [z() for _ in range(3)], z()
        bits = torch.zeros(s_fv[1:], dtype=torch.int16, device="cuda")
        F = [dev(f) if a else None for a, f in zip(act, Fs)]
        torch.cuda.synchronize()
        c.detect_troubles(dev(W), dev(Wo), tr, *al, 1, 0b10001)
        c.detect_troubles_bits(dev(W), dev(Wo), tb, bits, 1, 0b10001)
        c.fallback_fluxes(dev(W), dev(th), *F, 1e-3)
        out.append([host(x) for x in [tr, tb, bits] + al + [f for f in F if f is not None]])
        c.close()
    assert out[0][0].any()
    for a, b in zip(*out):
        assert same(a, b)
