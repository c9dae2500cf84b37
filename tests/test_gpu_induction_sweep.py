"""The fused induction step against the stage entries it fuses, bit for bit, on
random face fields (all three components, ghosts included): every sign of the
velocity along every axis, zero among them (the face solve then takes the mean
of both sides), periodic and gradfree boundaries, meshes from one element per
axis to a ragged last tile, and widths that are not powers of two."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import dev, host  # noqa: E402


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def stage_step(c, p, B, shapes, E, sE, dt, h, act):
    """copy_ader, p+1 times Solve_E with p predictor updates, update_B_solution (src/induction_ader.hpp:343-359)."""
    L, T = sk.lib(), p + 1
    d8 = ctypes.c_double
    sa = [(T,) + s[1:] for s in shapes]
    Ba = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in sa]
    S = sk.SDShape.of
    for d in range(3):
        c.copy_ader(B[d], Ba[d])
    for k in range(T):
        for e in (2, 1, 0):
            a1, a2 = (e + 1) % 3, (e + 2) % 3
            sk.check(L.spdk_induction_E(c.ctx, ptr(E[e]), S(sE[e]), ptr(Ba[a1]), S(sa[a1]), ptr(Ba[a2]), S(sa[a2]), e))
        for d in range(3):
            for e in sorted({0, 1, 2} - {d}):
                if act[d]:
                    sk.check(L.spdk_fill_sd_traces(c.ctx, ptr(E[e]), S(sE[e]), d))
        for d in range(3):
            if act[d]:
                sk.check(L.spdk_E_riemann(c.ctx, ptr(E[(d + 1) % 3]), S(sE[(d + 1) % 3]), d, 4))
                sk.check(L.spdk_E_riemann(c.ctx, ptr(E[(d + 2) % 3]), S(sE[(d + 2) % 3]), d, 3))
        for d in range(3):
            a1, a2 = (d + 1) % 3, (d + 2) % 3
            args = [ptr(E[a1]), S(sE[a1]), ptr(E[a2]), S(sE[a2]), d8(h[a1]), d8(h[a2]), d8(dt), d]
            if k < T - 1:
                sk.check(L.spdk_B_predict(c.ctx, ptr(B[d]), ptr(Ba[d]), S(sa[d]), *args))
            else:
                sk.check(L.spdk_B_correct(c.ctx, ptr(B[d]), S(shapes[d]), *args))
    torch.cuda.synchronize()


CASES = [(dim, p, N, v, bc)
         for dim, p, N in [(2, 1, (1, 1, 1)), (2, 3, (11, 3, 1)), (2, 4, (8, 5, 1)), (2, 2, (17, 2, 1)),
                           (3, 1, (2, 1, 3)), (3, 2, (6, 2, 2)), (3, 3, (4, 3, 2))]
         for v, bc in [((1.0, 0.5, 0.25), (0, 0, 0)), ((-1.0, 0.0, 0.5), (0, 1, 0)), ((0.0, -0.3, -0.7), (1, 0, 1)),
                       ((0.0, 0.0, 0.0), (1, 1, 1)), ((0.4, -0.6, 0.0), (1, 1, 0))]]


@pytest.mark.parametrize("dim,p,N,v,bc", CASES)
def test_fused_step_equals_the_stages(dim, p, N, v, bc, wide=False):
    act = [d < dim for d in range(3)]
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"]
    h = [1.9, 1.3, 1.7] if wide else [1.3 / (N[d] + 2) if act[d] else 1.0 for d in range(3)]
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        c = sk.Context(p, act, bc, p + 1, ops, h=h, vel=v)
        n = [p + 1 if a else 1 for a in act]
        Ne = [N[d] + 2 if act[d] else 1 for d in range(3)]

        def shape(nt, nv, stag):
            q = [n[d] + 1 if d in stag and act[d] else n[d] for d in range(3)]
            return (nt, nv, Ne[2], Ne[1], Ne[0], q[2], q[1], q[0])

        sB = [shape(1, 1, (d,)) for d in range(3)]
        sE = [shape(p + 1, 8, {0, 1, 2} - {d}) for d in range(3)]
        rng = np.random.default_rng(100 * p + dim)
        B0 = [rng.standard_normal(s) for s in sB]
        B0[0][..., 0] = 0.0  # exact zeros of either sign, and values near the smallest normal ones
        B0[1][..., 0] = -0.0
        B0[2][...] *= 1e-290
        if wide:
            B0 = [rng.integers(-2 ** (d + 1), 2 ** (d + 1) + 1, size=s) * 5e-324 for d, s in enumerate(sB)]
        a, b = [dev(x) for x in B0], [dev(x) for x in B0]
        E = [torch.zeros(s, dtype=torch.float64, device="cuda") for s in sE]
        dt = 8.0 if wide else 0.01
        stage_step(c, p, a, sB, E, sE, dt, h, act)
        L = sk.lib()
        cnt = (ctypes.c_int * 3)(*Ne)
        L.spdk_induction_fused_workspace_bytes.restype = ctypes.c_size_t
        nb = L.spdk_induction_fused_workspace_bytes(c.ctx, cnt)
        assert nb > 0, sk.last_error()
        ws = torch.full((nb,), 255, dtype=torch.uint8, device="cuda")  # NaN: nothing stale may be read
        args = [x for d in range(3) for x in (ptr(b[d]), sk.SDShape.of(sB[d]))]
        sk.check(L.spdk_induction_step_fused(c.ctx, *args, ptr(ws), ctypes.c_double(dt)))
        for d in range(3):
            x, y = host(a[d]), host(b[d])
            assert np.isfinite(x).all()
            assert np.array_equal(x, y), f"B{'xyz'[d]}: {int((x != y).sum())} of {x.size} differ"
        c.close()


@pytest.mark.parametrize("dim,p,N", [(2, 3, (11, 3, 1)), (3, 3, (4, 3, 2))])
@pytest.mark.parametrize("v", [(1.0, 0.5, 0.25), (0.0, -0.7, -1.0)])
def test_subnormal_on_wide_elements(dim, p, N, v):
    """A field of a few units of 2^-1074 on elements wider than 1: sums that are zero though their terms are not."""
    test_fused_step_equals_the_stages(dim, p, N, v, (0, 0, 0), wide=True)
