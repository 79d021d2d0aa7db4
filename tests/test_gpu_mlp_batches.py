"""The network's products at batches around the 32-row tiles and the rounds of the K loop (384 rows of a
weight gradient a round): forward outputs, loss and gradients against the numpy oracle with the same
BF16 rounding, at the bars of the network's parity test (BF16 operands; sums in FP32).
"""
import ctypes as C

import numpy as np
import pytest

from gsstructuralanalysis_amd import _lib as L
from oracle import mlp
from test_gpu_mlp import _f, _net

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [15, 32, 33, 384, 385, 1031])
def test_products_at_batch_edges(batch, ksh):
    lib = L.load()
    print(f"[case] network batch {batch}", flush=True)
    h, n = _net()
    try:
        rng = np.random.default_rng(1000 + batch)
        p = np.zeros(n, dtype=np.float32)
        L.check(lib.ksh_mlp_get_params(h, _f(p)))
        x = rng.standard_normal((batch, 264)).astype(np.float32)
        t = rng.standard_normal((batch, 65)).astype(np.float32)
        y = np.zeros((batch, 65), dtype=np.float32)
        L.check(lib.ksh_mlp_forward(h, _f(x), batch, _f(y)))
        yr = mlp.forward(p, x, bf=True)[0][-1]
        assert np.abs(y - yr).max() <= 2e-3 * np.abs(yr).max()
        y1 = np.zeros((1, 65), dtype=np.float32)
        L.check(lib.ksh_mlp_forward(h, _f(np.ascontiguousarray(x[-1:])), 1, _f(y1)))
        assert np.array_equal(y1[0], y[-1])  # a row's result does not depend on the batch
        g = np.zeros(n, dtype=np.float32)
        loss = C.c_double()
        L.check(lib.ksh_mlp_gradients(h, _f(x), _f(t), batch, _f(g), C.byref(loss)))
        lr, gr = mlp.loss_and_grad(p, x, t, bf=True)
        assert abs(loss.value - lr) <= 1e-3 * lr
        assert np.linalg.norm(g - gr) <= 1e-2 * np.linalg.norm(gr)
    finally:
        lib.ksh_mlp_destroy(h)
