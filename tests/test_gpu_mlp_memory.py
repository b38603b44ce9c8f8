"""The predictor's batch buffers after an allocation that failed: the call reports it, and later calls allocate again."""
import ctypes as C

import numpy as np
import pytest

import mlp_oracle as mo
from ikarus_amd import _capi as capi
from ikarus_amd import learned
from test_gpu_mlp import _data, _rel, _slices

pytestmark = pytest.mark.gpu

TOO_MANY = 1 << 40  # rows: 60 TB of inputs alone, refused by the first allocation; nothing of x or t is read


def test_training_after_a_failed_allocation():
    print("case: mlp training after a failed allocation", flush=True)
    L, m = capi.lib(), learned.MLP(seed=5)
    p = m.params()
    x, t = _data(100, 3)
    loss = C.c_double()
    g = np.zeros_like(p)
    xp, tp = capi.ptr(x), capi.ptr(t)
    assert L.ik_mlp_loss_grad(m.h, xp, tp, TOO_MANY, C.byref(loss), capi.ptr(g), capi.HOST) == capi.IK_EHIP
    assert L.ik_mlp_train_step(m.h, xp, tp, TOO_MANY, C.c_float(1e-3), C.byref(loss), capi.HOST) == capi.IK_EHIP
    assert np.array_equal(m.params(), p)
    l, g = m.loss_grad(x, t)
    lo, go = mo.loss_grad(p, x, t, bf16=True)
    assert abs(l - lo) <= 1e-3 * lo
    for name, sl in _slices():
        assert _rel(g[sl], go[sl]) < 1e-2, name
    m.close()


def test_forward_after_a_failed_allocation():
    print("case: mlp forward after a failed allocation", flush=True)
    L, m = capi.lib(), learned.MLP(seed=6)
    x, _ = _data(100, 4)
    y = np.zeros((100, 3), np.float32)
    assert L.ik_mlp_forward(m.h, capi.ptr(x), TOO_MANY, capi.ptr(y), capi.HOST) == capi.IK_EHIP
    assert _rel(m.forward(x), mo.forward(m.params(), x, bf16=True)[0]) < 2e-3
    m.close()
