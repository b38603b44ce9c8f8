"""Saint Venant-Kirchhoff tangents on both sides of the size of K at which complete blocks are stored past the caches."""
import numpy as np
import pytest

import ikarus_amd as ia
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_parity import _relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [((50, 50, 50), capi.FP64), ((56, 56, 56), capi.FP64),
                                         ((66, 66, 66), capi.FP32)])
def test_svk_tangent_is_the_residuals_derivative(n, precision):
    """K x = b solved with the assembled tangent, and the central difference of the residual along x gives b again. Step
    1e-5 / |x|_max on elements of size 1/56: truncation and rounding of the difference each below 1e-6 relative, the
    solve 1e-9; an FP32 tangent is rounded to 6e-8, and |K| |x| is below 1e4 |b| for the smooth x: 6e-4."""
    print(f"case: svk tangent stores n={n} precision={precision}", flush=True)
    p = pb.hex_block(n, material=capi.SVK, jitter=0.05, seed=3)
    free = 1 - p.fixed
    u = 0.02 * np.sin(2.0 * p.X).ravel() * free
    dev = ia.Device(p)
    dev.set_requirement(u, 0.5)
    dev.matrix(capi.DBC_FULL, precision)
    b = np.cos(3.0 * p.X).ravel() * free  # smooth: x is a smooth displacement
    kind = capi.PCG_JACOBI_FP64 if precision == capi.FP64 else capi.PCG_TWOLEVEL_FP32_IR
    x, info = dev.solve(b, ia.solver_opts(kind=kind, rtol=1e-9, inner_rtol=1e-3))
    assert info.converged == 1
    h = 1e-5 / np.abs(x).max()
    R = []
    for s in (h, -h):
        dev.set_requirement(u + s * x, 0.5)
        R.append(dev.vector(capi.DBC_FULL))
    assert _relerr((R[0] - R[1]) / (2 * h), b) < (1e-5 if precision == capi.FP64 else 2e-3)
    # the tangent with the residual in the same pass: the same matrix and the residual kernel's bits
    dev.set_requirement(u, 0.5)
    again = dev.assemble(capi.DBC_FULL, precision)
    assert np.array_equal(dev.vector(capi.DBC_FULL), again)
    dev.close()
