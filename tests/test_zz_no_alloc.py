"""The allocation-free whole-step entry (spdk_hydro_step_fused_noalloc,
workspace in a static per-GPU array) against the allocating one
(spdk_hydro_step_fused) through the C ABI: two calls in a row, the second
on a smaller mesh, every output bit for bit; a mesh whose workspace exceeds
the array is rejected before any launch."""
import ctypes

import numpy as np
import pytest

import oracle_py as op

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
import spd_k_amd as sk  # noqa: E402
from test_gpu_stages import ctx_for, dev, host, sd_shape, state  # noqa: E402


def _one(p, act, N, seed, dt):
    c, _, _, _ = ctx_for(p, act, N=N)
    n = p + 1
    s_u = sd_shape(1, 6, N, n, act)
    U0 = state(s_u, np.random.default_rng(seed))
    Ua, Ub = dev(U0), dev(U0)
    Wa = torch.zeros(s_u, dtype=torch.float64, device="cuda")
    Wb = torch.full(s_u, float("nan"), dtype=torch.float64, device="cuda")
    dta = c.hydro_step_fused(Ua, dt, Wa)
    dtb = c.hydro_step_fused_noalloc(Ub, dt, Wb)
    a, b = host(Ua), host(Ub)
    assert np.array_equal(a, b), f"U_sp: {int((a != b).sum())} of {a.size} differ"
    wa, wb = host(Wa), host(Wb)
    assert np.array_equal(wa, wb), f"W_cv: {int((wa != wb).sum())} of {wa.size} differ"
    assert dta == dtb and np.isfinite(dta) and dta > 0
    assert not np.array_equal(a, U0)  # the step changed the state
    c.close()


def test_noalloc_step_equals_allocating_step():
    cap = sk.lib().spdk_fused_noalloc_max_bytes()
    assert cap == 64 << 20
    # 3-D p=3 on 8^3 elements (10^3 with ghosts: 43.5 MB of workspace), then
    # a smaller 2-D p=2 mesh: the array keeps the first call's contents
    _one(3, (1, 1, 1), (8, 8, 8), 11, 1e-3)
    _one(2, (1, 1, 0), (6, 5, 1), 12, 2e-3)


def test_largest_meshes_of_the_array():
    """The two largest 2-D p=3 meshes (8064 and 8065 elements with ghosts) fit
    and step as the allocating entry does, and more elements are refused."""
    L = sk.lib()
    c, _, _, _ = ctx_for(3, (1, 1, 0), N=(82, 94, 1))
    size = lambda *N: L.spdk_fused_workspace_bytes(c.ctx, (ctypes.c_int * 3)(*N))
    assert size(84, 96, 1) <= size(5, 1613, 1) <= (64 << 20) < size(84, 97, 1)
    c.close()
    _one(3, (1, 1, 0), (82, 94, 1), 13, 1e-5)
    _one(3, (1, 1, 0), (3, 1611, 1), 14, 1e-5)


@pytest.mark.parametrize("p,act", [(p, a) for p in (1, 2, 3, 4) for a in ((1, 0, 0), (1, 1, 0), (1, 1, 1))
                                   if p < 4 or not a[2]])
@pytest.mark.parametrize("rk", [0, 3])
def test_workspace_is_state_traces_and_the_step_start(p, act, rk):
    """Nothing beside the predictor slices, two trace buffers and the stage start
    state: a mesh that fits the array does not depend on the launch shapes."""
    dim, n, T = sum(act), p + 1, 1 if rk else p + 1
    m = op.matrices(p)
    ops = {k: m[k] for k in sk.Context.MATS}
    ops["wt"] = m["wt"][:T]
    if rk:
        ops["invader"] = np.ones((1, 1))
    c = sk.Context(p, act, (0, 0, 0), T, ops, rk_order=rk)
    for Ne in ((3, 3, 3), (7, 5, 4), (40, 33, 21)):
        N = [Ne[d] if act[d] else 1 for d in range(3)]
        E = int(np.prod(N))
        doubles = 5 * E * (T * n ** dim + 2 * dim * T * 2 * n ** (dim - 1) + n ** dim)
        assert sk.lib().spdk_fused_workspace_bytes(c.ctx, (ctypes.c_int * 3)(*N)) == 8 * doubles
    c.close()


def test_noalloc_rejects_meshes_beyond_the_array():
    c, _, _, _ = ctx_for(3, (1, 1, 1), N=(12, 12, 12))
    s = sd_shape(1, 6, (12, 12, 12), 4, (1, 1, 1))
    N = (ctypes.c_int * 3)(s[4], s[3], s[2])
    assert sk.lib().spdk_fused_workspace_bytes(c.ctx, N) > (64 << 20)
    U = torch.zeros(s, dtype=torch.float64, device="cuda")
    with pytest.raises(RuntimeError, match="static scratch"):
        c.hydro_step_fused_noalloc(U, 1e-3)
    c.close()
