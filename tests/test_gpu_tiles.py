"""The tiled tangent kernel where its tiles are not full boxes of a grid: element counts beside the tile size (16), and
fans of n hexahedra around one edge, whose K blocks get up to n element blocks (one accumulator for one or two blocks,
one per block above that, several tiles for n > 16)."""
import numpy as np
import pytest

import ikarus_amd as ia
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_parity import _oracle_for, _relerr

pytestmark = pytest.mark.gpu


def _fan(n, layers, material):
    """n hexahedra around the z axis (corners: axis, rim node i, rim node i + 1 and the point outside them)."""
    a = 2 * np.pi * np.arange(n) / n
    rim, out = np.c_[np.cos(a), np.sin(a)], 1.6 * np.c_[np.cos(a + np.pi / n), np.sin(a + np.pi / n)]
    plane = np.concatenate([[[0.0, 0.0]], rim, out])
    m = len(plane)
    X = np.concatenate([np.c_[plane, np.full(m, 0.5 * z)] for z in range(layers + 1)])
    quad = np.array([[0, 1 + i, 1 + (i + 1) % n, 1 + n + i] for i in range(n)])
    conn = np.concatenate([np.c_[quad + z * m, quad + (z + 1) * m] for z in range(layers)]).astype(np.int32)
    # Dune corner order: (axis, rim i, rim i + 1, outer) is (0,0), (1,0), (0,1), (1,1)
    lam, mu = pb.lame(1000.0, 0.3)
    p = pb.Problem(X, conn, material, lam, mu, name=f"fan{n}")
    p.fixed = pb.clamp_flags(X, 2, 0.0)
    return p


def _check(p, u):
    o = _oracle_for(p)
    dev = ia.Device(p)
    dev.set_requirement(u, 0.5)
    Ro, Ko = o.vector(u, 0.5, capi.DBC_FULL), o.matrix(u, 0.5, capi.DBC_FULL)
    for precision, tol in ((capi.FP64, 1e-12), (capi.FP32, 1e-6)):  # FP32: one rounding per group sum and per block
        R = dev.assemble(capi.DBC_FULL, precision)
        assert _relerr(R, Ro) < 1e-12
        outer, inner, vals = dev.csc(capi.DBC_FULL)
        assert _relerr(vals, Ko) < tol
        again = dev.assemble(capi.DBC_FULL, precision)
        assert np.array_equal(again, R) and np.array_equal(dev.csc(capi.DBC_FULL)[2], vals)  # fixed summation order
    assert np.array_equal(dev.vector(capi.DBC_FULL), R)  # the residual kernel gives the same bits


@pytest.mark.parametrize("material", [capi.NEOHOOKE, capi.SVK])
@pytest.mark.parametrize("n,layers", [(3, 1), (8, 2), (16, 1), (17, 1), (11, 5)])
def test_fan_of_elements_around_an_edge(n, layers, material):
    print(f"case: fan n={n} layers={layers} material={material}", flush=True)
    p = _fan(n, layers, material)
    u = 0.01 * np.random.default_rng(n).standard_normal(p.ndof) * (1 - p.fixed)
    _check(p, u)


@pytest.mark.parametrize("nel", [(1, 1, 1), (3, 5, 1), (4, 2, 2), (17, 1, 1), (5, 5, 5)])
def test_element_counts_beside_the_tile_size(nel):
    print(f"case: tiles nel={nel}", flush=True)
    p = pb.hex_block(nel, jitter=0.05, seed=3)
    u = 0.01 * np.random.default_rng(7).standard_normal(p.ndof) * (1 - p.fixed)
    _check(p, u)


@pytest.mark.parametrize("n,precision", [((50, 50, 50), capi.FP64), ((56, 56, 56), capi.FP64),
                                         ((70, 68, 68), capi.FP64), ((66, 66, 66), capi.FP32)])
def test_large_mesh_tangent_is_the_residuals_derivative(n, precision):
    """K below 256 MB, to 600 MB and above (complete K blocks stored through the caches, past them, through them):
    K x = b solved with the assembled tangent, and the central difference of the residual along x gives b again. Step
    1e-5 / |x|_max on elements of size 1/70: truncation and rounding of the difference each below 1e-6 relative, the
    solve 1e-9; an FP32 tangent is rounded to 6e-8, and |K| |x| is below 1e4 |b| for the smooth x: 6e-4."""
    print(f"case: large mesh tangent n={n} precision={precision}", flush=True)
    p = pb.hex_block(n, jitter=0.05, seed=3)
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
    dev.close()
