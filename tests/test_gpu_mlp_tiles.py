"""Gradient and loss of batches that end inside a tile of 32 samples, have more
tiles than blocks, or only the scratch of one partial gradient per 64 samples,
against the float64 oracle. Bound: a gradient entry is a sum over the batch of
products of FP32 values some tens of roundings (2^-24 each) deep; 2e-5 of the
largest entry is 330 of them."""
import ctypes as C

import numpy as np
import pytest

from oracle import mlp_oracle as M
from stardust_amd import _lib as L

pytestmark = pytest.mark.gpu
NP = 9987


@pytest.mark.parametrize("batch,small", [(1, False), (31, False), (32, False), (33, False), (65, True), (2000, True),
                                         (8192, False), (17000, False), (33001, True)])
def test_gradient_of_a_batch(batch, small):
    print("[gpu-case] training batch", batch, small, flush=True)
    L.require_gpu()
    rng = np.random.default_rng(batch)
    X = rng.normal(0, 1, (batch, 22)).astype(np.float32)
    T = rng.normal(0, 1, (batch, 3))
    T = (T / np.linalg.norm(T, axis=1, keepdims=True)).astype(np.float32)
    w = rng.normal(0, 0.15, NP).astype(np.float32)
    idx = rng.permutation(batch).astype(np.int32)
    nb = C.c_size_t()
    L.call("sd_mlp_train_scratch_bytes", batch, C.byref(nb))
    least = -(-batch // 64) * (NP + 1) * 4 + 256
    assert nb.value >= least
    size = least if small else nb.value
    Xd, Td, wd, id_ = (L.DeviceBuffer.from_array(a) for a in (X, T, w, idx))
    g, loss = L.DeviceBuffer(4 * NP), L.DeviceBuffer(4)
    scr = L.DeviceBuffer.from_array(np.full(size // 4, np.nan, np.float32))
    run = lambda bytes_: L.load().sd_mlp_forward_backward(Xd.ptr, Td.ptr, id_.ptr, batch, wd.ptr, g.ptr, loss.ptr,
                                                          scr.ptr, bytes_, None)
    assert run(least - 1) == L.SD_ERR_ARG
    assert run(size) == L.SD_OK
    L.synchronize()
    got, l1 = g.download(np.float32, NP), g.download(np.float32, NP)
    lv = float(loss.download(np.float32, 1)[0])
    Lr, gr = M.loss_and_grad(w, X[idx], T[idx])
    assert abs(lv - Lr) < 1e-5
    assert np.abs(got - gr).max() < 2e-5 * np.abs(gr).max() + 1e-7, np.abs(got - gr).max() / np.abs(gr).max()
    assert run(size) == L.SD_OK  # the same bits again
    L.synchronize()
    assert np.array_equal(g.download(np.float32, NP), l1)
