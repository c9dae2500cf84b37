"""The face fluxes of the FP64 sweep (spdk_fused_predict_fv_fluxes) against the
flux-point fluxes of spdk_fused_predict_fluxes through spdk_fv_face_integral,
bit for bit, with and without the x flux points, on meshes that leave idle
elements in the last workgroup."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import ctx_for, dev, host, sd_shape, state  # noqa: E402


def ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("act,N,p", [((1, 0, 0), (7, 1, 1), 3), ((1, 1, 0), (6, 5, 1), 3), ((1, 1, 0), (3, 4, 1), 4),
                                     ((1, 1, 1), (1, 1, 1), 3), ((1, 1, 1), (3, 2, 4), 3), ((1, 1, 1), (6, 1, 2), 3),
                                     ((1, 1, 1), (2, 3, 2), 2), ((1, 1, 1), (3, 2, 1), 1)])
@pytest.mark.parametrize("bc", [(0, 0, 0), (2, 1, 0)])
def test_faces(act, N, p, bc):
    n, L, dt = p + 1, sk.lib(), ctypes.c_double(1e-3)
    c = ctx_for(p, act, bc, N=N)[0]
    U = dev(state(sd_shape(1, 6, N, n, act), np.random.default_rng(p)))
    sp = sk.SDShape.of(U.shape)
    nb = L.spdk_fused_workspace_bytes(c.ctx, (ctypes.c_int * 3)(U.shape[4], U.shape[3], U.shape[2]))
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
    s_ader = sk.SDShape.of(sd_shape(n, 6, N, n, act))
    z = lambda s, x=0.0: torch.full(s, x, dtype=torch.float64, device="cuda")
    fp = [z(sd_shape(n, 6, N, n, act, stag=d)) if act[d] else None for d in range(3)]
    sk.check(L.spdk_fused_predict_fluxes(c.ctx, ptr(U), sp, ptr(ws), dt, *[ptr(x) for x in fp], s_ader), "predict_fluxes")
    cells = [n * N[d] + 4 if act[d] else 1 for d in range(3)]
    fv = sk.FVShape.of((6, cells[2], cells[1], cells[0]))
    shape = lambda d: (6, cells[2] + (d == 2 and act[2]), cells[1] + (d == 1 and act[1]), cells[0] + (d == 0))
    for fx in (None, torch.zeros_like(fp[0])):
        F = [z(shape(d), 7e7) if act[d] else None for _ in range(n) for d in range(3)]
        P = (ctypes.c_void_p * len(F))(*[f.data_ptr() if f is not None else 0 for f in F])
        sk.check(L.spdk_fused_predict_fv_fluxes(c.ctx, ptr(U), sp, ptr(ws), dt, P, fv, ptr(fx), s_ader), "predict_fv_fluxes")
        if fx is not None:
            assert np.array_equal(host(fx)[:, :5], host(fp[0])[:, :5])
        for t in range(n):
            for d in range(3):
                if not act[d]:
                    continue
                W = z(shape(d), 7e7)
                c.face_integral(fp[d], W, z((1,) + tuple(fp[d].shape[1:])), t, d)
                # the faces of the active cells (the stage entry also fills some beyond them)
                box = (slice(0, 5),) + tuple((slice(2, cells[x] - 1) if x == d else slice(2, -2)) if act[x] else slice(None)
                                             for x in (2, 1, 0))
                assert np.array_equal(host(F[3 * t + d])[box], host(W)[box]), (t, d, fx is not None)
    c.close()
