"""The MLP kernels (BF16 MFMA, FP32 accumulation) against the CPU oracle in
its BF16 mode: forward outputs and all parameter gradients, on dimensions
and a batch that are not multiples of the 64-wide tiles; and GPU training
(forward, backward and Adam on the device) fitting a teacher network."""
import ctypes

import numpy as np
import pytest
import torch

import oracle_py as op
import spd_k_amd

pytestmark = pytest.mark.gpu


def make_net(dims, cap, params):
    L = spd_k_amd.lib()
    net = ctypes.c_void_p()
    spd_k_amd.check(L.spdk_mlp_create((ctypes.c_int * 4)(*dims), cap, None, ctypes.byref(net)), "spdk_mlp_create")
    spd_k_amd.check(L.spdk_mlp_set_params(net, params.ctypes.data_as(ctypes.c_void_p)), "set_params")
    return net


def dev(a):
    return torch.tensor(np.ascontiguousarray(a, dtype=np.float32), device="cuda:0")


DIMS = [70, 128, 64, 90]


def test_forward_matches_oracle():
    rng = np.random.default_rng(5)
    B = 100
    p = op.mlp_init(DIMS, seed=6)
    X = rng.standard_normal((B, DIMS[0]))
    net = make_net(DIMS, 128, p)
    L = spd_k_amd.lib()
    Xd, Yd = dev(X), torch.zeros((B, DIMS[3]), device="cuda:0")
    spd_k_amd.check(L.spdk_mlp_forward(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(DIMS[0]), B,
                                       ctypes.c_void_p(Yd.data_ptr()), ctypes.c_long(DIMS[3])), "forward")
    torch.cuda.synchronize()
    Y = Yd.cpu().double().numpy()
    ref = op.orc_mlp_forward(DIMS, p, X, bf16=True)
    exact = op.orc_mlp_forward(DIMS, p, X, bf16=False)
    # BF16 rounding of the hidden activations can differ by one unit where the
    # FP32 and FP64 pre-activations straddle a rounding boundary
    assert np.abs(Y - ref).max() <= 1e-2 * np.abs(ref).max()
    assert np.linalg.norm(Y - ref) <= 2e-3 * np.linalg.norm(ref)
    # and the BF16 forward is close to the exact one
    assert np.linalg.norm(Y - exact) <= 3e-2 * np.linalg.norm(exact)
    L.spdk_mlp_destroy(net)


def test_gradients_match_oracle():
    rng = np.random.default_rng(7)
    B = 100
    p = op.mlp_init(DIMS, seed=8)
    X = rng.standard_normal((B, DIMS[0]))
    T = rng.standard_normal((B, DIMS[3]))
    net = make_net(DIMS, 128, p)
    L = spd_k_amd.lib()
    n = op.mlp_param_count(DIMS)
    g = np.zeros(n, dtype=np.float32)
    loss = ctypes.c_float()
    Xd, Td = dev(X), dev(T)
    spd_k_amd.check(L.spdk_mlp_gradients(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(DIMS[0]),
                                         ctypes.c_void_p(Td.data_ptr()), ctypes.c_long(DIMS[3]), B,
                                         g.ctypes.data_as(ctypes.c_void_p), ctypes.byref(loss)), "gradients")
    ref, ref_loss = op.orc_mlp_grad(DIMS, p, X, T, bf16=True)
    assert abs(loss.value - ref_loss) <= 1e-3 * ref_loss
    o = 0
    for l in range(3):
        for size in (DIMS[l + 1] * DIMS[l], DIMS[l + 1]):
            a, b = g[o:o + size].astype(np.float64), ref[o:o + size]
            assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b), (l, size, np.linalg.norm(a - b) / np.linalg.norm(b))
            o += size
    L.spdk_mlp_destroy(net)


def test_training_fits_a_teacher():
    """Adam on the device drives the loss on a teacher network's outputs down
    by more than 20x from a different random initialisation."""
    rng = np.random.default_rng(9)
    dims = [32, 128, 128, 48]
    B = 512
    teacher = op.mlp_init(dims, seed=10, scale=0.5)
    X = rng.standard_normal((B, dims[0]))
    T = op.orc_mlp_forward(dims, teacher, X, bf16=False)
    net = make_net(dims, B, op.mlp_init(dims, seed=11, scale=0.5))
    L = spd_k_amd.lib()
    Xd, Td = dev(X), dev(T)
    loss = ctypes.c_float()
    losses = []
    for it in range(600):
        spd_k_amd.check(L.spdk_mlp_train_step(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(dims[0]),
                                              ctypes.c_void_p(Td.data_ptr()), ctypes.c_long(dims[3]), B,
                                              ctypes.c_float(2e-3), ctypes.byref(loss) if it % 50 == 0 else None),
                        "train_step")
        if it % 50 == 0:
            losses.append(loss.value)
    print(losses)
    assert losses[-1] < losses[0] / 20, losses
    L.spdk_mlp_destroy(net)


# batches at the edges of the 64-row tiles and of the weight gradient's row
# steps; the last two fill the chip with 128-wide tiles (layer 3: 19 column
# tiles of 64, 10 of 128), one of them with a ragged last row tile
@pytest.mark.parametrize("B", [1, 63, 64, 65, 257, 6656, 6701])
def test_tiles_match_oracle(B):
    dims = [70, 64, 128, 1210]
    rng = np.random.default_rng(B)
    p = op.mlp_init(dims, seed=9)
    X, T = rng.standard_normal((B, dims[0])), rng.standard_normal((B, dims[3]))
    net = make_net(dims, 6701, p)
    L = spd_k_amd.lib()
    ldy = dims[3] + 3  # rows longer than the outputs: the tail is left alone
    Xd, Td, Yd = dev(X), dev(T), torch.full((B, ldy), 7.0, device="cuda:0")
    spd_k_amd.check(L.spdk_mlp_forward(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(dims[0]), B,
                                       ctypes.c_void_p(Yd.data_ptr()), ctypes.c_long(ldy)), "forward")
    torch.cuda.synchronize()
    Y = Yd.cpu().double().numpy()
    ref = op.orc_mlp_forward(dims, p, X, bf16=True)
    # the bounds of test_forward_matches_oracle (BF16 rounding of the hidden layers)
    assert np.abs(Y[:, :dims[3]] - ref).max() <= 1e-2 * np.abs(ref).max()
    assert np.linalg.norm(Y[:, :dims[3]] - ref) <= 2e-3 * np.linalg.norm(ref)
    assert np.all(Y[:, dims[3]:] == 7.0)
    g = np.zeros(op.mlp_param_count(dims), dtype=np.float32)
    loss = ctypes.c_float()
    spd_k_amd.check(L.spdk_mlp_gradients(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(dims[0]),
                                         ctypes.c_void_p(Td.data_ptr()), ctypes.c_long(dims[3]), B,
                                         g.ctypes.data_as(ctypes.c_void_p), ctypes.byref(loss)), "gradients")
    ref, ref_loss = op.orc_mlp_grad(dims, p, X, T, bf16=True)
    o = 0
    assert abs(loss.value - ref_loss) <= 1e-3 * ref_loss
    for l in range(3):  # every weight matrix and bias by itself
        for n in (dims[l + 1] * dims[l], dims[l + 1]):
            a, b = g[o:o + n].astype(np.float64), ref[o:o + n]
            assert np.linalg.norm(a - b) <= 2e-2 * np.linalg.norm(b), (l, n)
            o += n
    assert L.spdk_mlp_forward(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(dims[0]), B, None,
                              ctypes.c_long(ldy)) != 0
    assert L.spdk_mlp_forward(net, ctypes.c_void_p(Xd.data_ptr()), ctypes.c_long(dims[0]), B,
                              ctypes.c_void_p(Yd.data_ptr()), ctypes.c_long(dims[3] - 1)) != 0
    L.spdk_mlp_destroy(net)
