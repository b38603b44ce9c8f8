"""The EAS kernels at element counts beside what a wavefront takes (1, 2 or 4 elements in the tangent by the size of the
mesh, 3 in the internal-variable update), with faces' loads, both materials, at alpha != 0."""
import numpy as np
import pytest

import ikarus_amd as ia
import pyoracle as po
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_eas import _oracle_for, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("material", [capi.NEOHOOKE, capi.SVK])
@pytest.mark.parametrize("nel", [(1, 1, 1), (1, 2, 1), (3, 1, 1), (2, 2, 1), (5, 1, 1), (13, 1, 1), (2048, 1, 1),
                                 (683, 3, 1), (16, 32, 32), (17, 31, 32)])
def test_eas_element_counts(nel, material):
    print(f"case: eas counts nel={nel} material={material}", flush=True)
    p = pb.hex_block(nel, L=nel, material=material, jitter=0.08, seed=23, eas=21)  # unit cubes
    dev, o = ia.Device(p), _oracle_for(p)
    rng = np.random.default_rng(11)
    u = 0.01 * rng.standard_normal(p.ndof) * (1 - p.fixed)
    alpha = 1e-3 * rng.standard_normal((p.ne, 21))
    du = 1e-3 * rng.standard_normal(p.ndof) * (1 - p.fixed)
    for a in (dev, o):
        a.set_alpha(alpha)
    dev.set_requirement(u, 0.8)
    R = dev.assemble(capi.DBC_FULL, capi.FP64)
    # FP64 sums of up to 48 products and the condensation (D's condition up to 1e4) in another order: 1e-10
    assert _rel(dev.csc()[2], o.matrix(u, 0.8, po.FULL)) < 1e-10
    assert _rel(R, o.vector(u, 0.8, po.FULL)) < 1e-10
    dev.update_state(du)
    o.update_state(u, 0.8, du)
    assert _rel(dev.alpha() - alpha, o.alpha() - alpha) < 1e-9
    # the residual alone: the same bits, and the same update from its cache
    updated = dev.alpha()
    dev.set_alpha(alpha)
    dev.set_requirement(u, 0.8)
    assert np.array_equal(dev.vector(capi.DBC_FULL), R)
    dev.update_state(du)
    assert np.array_equal(dev.alpha(), updated)
    dev.close()
