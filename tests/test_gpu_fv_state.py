"""The step's state between the solution points and the FV cells
(spdk_fv_state_from_sd, spdk_fv_state_to_sd) against the stage transforms, bit
for bit, on rows with and without ghost elements and partial last groups; and
the ghost fill of arrays of 1 to 8 variables against a copy by index."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import ctx_for, dev, host, sd_shape  # noqa: E402


def ptr(t):
    return ctypes.c_void_p(t.data_ptr())


MESHES = [((1, 0, 0), (1, 1, 1), 3), ((1, 0, 0), (300, 1, 1), 1), ((1, 0, 0), (131, 1, 1), 5), ((1, 1, 0), (1, 1, 1), 2),
          ((1, 1, 0), (67, 3, 1), 3), ((1, 1, 0), (40, 2, 1), 4), ((1, 1, 0), (3, 5, 1), 1), ((1, 1, 1), (1, 1, 1), 3),
          ((1, 1, 1), (19, 2, 3), 3), ((1, 1, 1), (70, 2, 1), 1), ((1, 1, 1), (3, 2, 2), 5), ((1, 1, 1), (21, 1, 2), 2)]


@pytest.mark.parametrize("act,N,p", MESHES)
def test_state_round(act, N, p):
    n = p + 1
    rng = np.random.default_rng(p)
    c = ctx_for(p, act, N=N)[0]
    s = sd_shape(1, 6, N, n, act)
    u = rng.uniform(-0.3, 0.3, s)
    u[:, 0] += 1.0
    u[:, 4] += 3.0
    u[:, 5] = 0.0
    U = dev(u)
    cells = [n * N[d] + 4 if act[d] else 1 for d in range(3)]
    fv = sk.FVShape.of((6, cells[2], cells[1], cells[0]))
    A = torch.full((6, cells[2], cells[1], cells[0]), 7e7, dtype=torch.float64, device="cuda")
    sk.check(sk.lib().spdk_fv_state_from_sd(c.ctx, ptr(U), sk.SDShape.of(U.shape), ptr(A), fv), "from_sd")
    C, tmp = torch.zeros_like(U), torch.zeros_like(U)
    c.transform_a_to_b(U, C, tmp, sk.SPDK_M_SP_TO_CV)

    def rows(x):  # active elements of an SD array as FV rows (v, z, y, x)
        x = host(x)[0][(slice(None),) + tuple(slice(1, -1) if act[d] else slice(None) for d in (2, 1, 0))]
        return x.transpose(0, 1, 4, 2, 5, 3, 6).reshape(6, *(n * N[d] if act[d] else 1 for d in (2, 1, 0)))

    inner = (slice(None),) + tuple(slice(2, -2) if act[d] else slice(None) for d in (2, 1, 0))
    a = host(A)
    assert np.array_equal(a[inner][:5], rows(C)[:5])
    # to_sd: other cell values in the active elements, the ghosts' own round trip
    new = a.copy()
    new[inner] *= 1.0 + 1e-3 * rng.uniform(-1, 1, new[inner].shape)
    Cn = host(C).copy()
    act_el = tuple(slice(1, -1) if act[d] else slice(None) for d in (2, 1, 0))
    e = [N[d] if act[d] else 1 for d in range(3)]
    q = [n if act[d] else 1 for d in range(3)]
    Cn[0][(slice(None),) + act_el] = new[inner].reshape(6, e[2], q[2], e[1], q[1], e[0], q[0]).transpose(0, 1, 3, 5, 2, 4, 6)
    Cn[0, 5] = 0.0
    V, W, Wc = torch.zeros_like(U), torch.zeros_like(U), torch.zeros_like(U)
    c.transform_a_to_b(dev(Cn), V, tmp, sk.SPDK_M_CV_TO_SP)
    c.compute_primitives(V, W)
    c.transform_a_to_b(W, Wc, tmp, sk.SPDK_M_SP_TO_CV)
    got, Wg, dt = U.clone(), torch.zeros_like(U), ctypes.c_double()
    sk.check(sk.lib().spdk_fv_state_to_sd(c.ctx, ptr(dev(new)), fv, ptr(got), sk.SDShape.of(U.shape), ptr(Wg),
                                          ctypes.byref(dt)), "to_sd")
    assert np.array_equal(host(got)[0, :5], host(V)[0, :5])
    assert np.array_equal(host(Wg)[0, :5], host(Wc)[0, :5])
    assert dt.value == c.compute_dt(Wc)
    c.close()


def source(l, n, bc):
    if 2 <= l < n - 2:
        return l, 1.0
    lo = l < 2
    if bc == 0:
        return (n - 4 + l, 1.0) if lo else (l - (n - 4), 1.0)
    if bc == 1:
        return (2 + l, 1.0) if lo else (l - 2, 1.0)
    return (3 - l, -1.0) if lo else (2 * (n - 2) - 1 - l, -1.0)


@pytest.mark.parametrize("nv", [1, 5, 6, 8])
@pytest.mark.parametrize("act,bc", [((1, 0, 0), (2, 0, 0)), ((1, 1, 0), (0, 2, 0)), ((1, 1, 0), (1, 0, 0)),
                                    ((1, 1, 1), (2, 1, 0)), ((1, 1, 1), (0, 2, 2))])
def test_ghost_fill(act, bc, nv):
    N = [9 if act[0] else 1, 8 if act[1] else 1, 11 if act[2] else 1]
    c = ctx_for(1, act, bc)[0]
    x = np.random.default_rng(nv).uniform(0.5, 1, (nv, N[2], N[1], N[0]))
    X = dev(x)
    sk.check(sk.lib().spdk_fill_fv_ghosts(c.ctx, ptr(X), sk.FVShape.of(X.shape)), "fill_fv_ghosts")
    src = [[source(l, N[d], bc[d]) if act[d] else (0, 1.0) for l in range(N[d])] for d in range(3)]
    want = x[:, [q for q, _ in src[2]]][:, :, [q for q, _ in src[1]]][:, :, :, [q for q, _ in src[0]]]
    for d in range(3):
        if 1 + d < nv:
            want[1 + d] *= np.array([f for _, f in src[d]]).reshape([-1 if 2 - a == d else 1 for a in range(3)])
    assert np.array_equal(host(X), want)
    c.close()
