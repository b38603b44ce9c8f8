"""The predictor's batched kernels (forward, forward + backward, weight gradients, Adam) at batch sizes on and beside
their tiles: rows per wavefront (16) and workgroup (64), the batch slices of the weight gradients (256 rows, load
steps of 128), more rows than one sweep of the grid covers (16,384 in training, 32,768 in the forward)."""
import numpy as np
import pytest

import mlp_oracle as mo
from ikarus_amd import _capi as capi
from ikarus_amd import learned
from test_gpu_mlp import _data, _rel, _slices
from test_zz_no_alloc import _Hip

pytestmark = pytest.mark.gpu


# the oracle rounds the same operands to BF16; a different FP32 summation order flips the rounding of a few operands by
# one part in 2^8, which stays below 2e-3 of an output vector and 1e-2 of a gradient block (as in test_gpu_mlp)
@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 255, 511, 513, 16385])
def test_gradient_at_tile_edges(n):
    print(f"case: mlp batch gradient n={n}", flush=True)
    m = learned.MLP(seed=5)
    p = m.params()
    x, t = _data(n, 10 + n)
    loss, g = m.loss_grad(x, t)
    lo, go = mo.loss_grad(p, x, t, bf16=True)
    assert abs(loss - lo) <= 1e-3 * lo
    for name, sl in _slices():
        assert _rel(g[sl], go[sl]) < 1e-2, name
    # a training step folds the same gradient into Adam's first step, -lr sign(g) up to eps
    assert m.train_step(x, t, 1e-3) == loss
    step = m.params() - p
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    assert np.allclose(step[big], -1e-3 * np.sign(g[big]), rtol=0.0, atol=1e-3 * 1e-8 / np.abs(g[big]).min() + 2e-7)


@pytest.mark.parametrize("n", [15, 65, 32769])
def test_forward_at_tile_edges(n):
    print(f"case: mlp batch forward n={n}", flush=True)
    m = learned.MLP(seed=6)
    x, _ = _data(n, 20 + n)
    assert _rel(m.forward(x), mo.forward(m.params(), x, bf16=True)[0]) < 2e-3


def test_noalloc_output_may_overlap_its_input():
    print("case: mlp forward noalloc in place", flush=True)
    hip = _Hip()
    m = learned.MLP(seed=7)
    x, _ = _data(1000, 3)
    ref = m.forward(x)
    buf = hip.malloc(x.nbytes)
    try:
        hip.h2d(buf, x)
        m._check(capi.lib().ik_mlp_forward_noalloc(m.h, buf, x.shape[0], buf))
        y = np.zeros_like(ref)
        hip.d2h(y, buf)
        assert np.array_equal(y, ref)
    finally:
        hip.lib.hipFree(buf)
        m.close()
