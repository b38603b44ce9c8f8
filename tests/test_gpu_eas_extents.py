"""EAS tangent of very small and very large elements: the entries of D scale with h^-13, so products of two of them leave
the range of a double long before D does."""
import numpy as np
import pytest

import ikarus_amd as ia
import pyoracle as po
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_eas import _oracle_for, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("material", [capi.NEOHOOKE, capi.SVK])
@pytest.mark.parametrize("h", [1e-17, 1e-12, 1.0, 1e6, 1e18])  # mu h^-13: 1e232, 1e167, 1e11, 1e-67, 1e-223
def test_eas_extents(h, material):
    print(f"case: eas extents h={h} material={material}", flush=True)
    nel = (3, 2, 2)
    p = pb.hex_block(nel, L=tuple(h * n for n in nel), material=material, E=2.1e11, jitter=0.08, seed=23, eas=21)
    p.fixed = pb.clamp_flags(p.X, 2, 0.0, tol=1e-3 * h)
    dev, o = ia.Device(p), _oracle_for(p)
    rng = np.random.default_rng(11)
    u = 0.01 * h * rng.standard_normal(p.ndof) * (1 - p.fixed)
    du = 1e-3 * h * rng.standard_normal(p.ndof) * (1 - p.fixed)
    dev.set_requirement(u, 0.8)
    R = dev.assemble(capi.DBC_FULL, capi.FP64)
    # the FULL treatment puts ones beside entries of mu h: compare the free rows and columns
    K, Ko = dev.csc()[2], o.matrix(u, 0.8, po.FULL)
    one = Ko == 1.0
    assert np.array_equal(K == 1.0, one)
    # FP64 sums of up to 48 products and the condensation (D's condition up to 1e4) in another order: 1e-10
    assert _rel(np.where(one, 0.0, K) / np.abs(Ko[~one]).max(), np.where(one, 0.0, Ko) / np.abs(Ko[~one]).max()) < 1e-10
    assert _rel(R / np.abs(R).max(), o.vector(u, 0.8, po.FULL) / np.abs(R).max()) < 1e-10
    dev.update_state(du)
    o.update_state(u, 0.8, du)
    a, b = dev.alpha(), o.alpha()
    assert _rel(a / np.abs(b).max(), b / np.abs(b).max()) < 1e-9
    dev.close()
