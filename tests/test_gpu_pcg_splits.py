"""The PCG kernels on both sides of the node counts where the SpMV's row split and the direction inside the SpMV end, and
with iteration limits at and beside the chunks in which iterations are enqueued."""
import numpy as np
import pytest
import scipy.sparse as sp

import ikarus_amd as ia
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_parity import _oracle_for

pytestmark = pytest.mark.gpu


def _setup(n, shuffle=False):
    p = pb.hex_block(n, jitter=0.05, seed=3)
    if shuffle:  # nodes and elements in random order
        g = np.random.default_rng(5)
        new = g.permutation(len(p.X))
        X, fixed = np.empty_like(p.X), np.empty_like(p.fixed.reshape(-1, 3))
        X[new], fixed[new] = p.X, p.fixed.reshape(-1, 3)
        q = pb.Problem(X, new[p.conn][g.permutation(len(p.conn))].astype(np.int32), p.material, p.lam, p.mu, name="s")
        q.fixed = fixed.ravel()
        p = q
    free = 1 - p.fixed
    u = 0.02 * np.sin(2.0 * p.X).ravel() * free  # smooth: the tangent stays positive definite
    b = np.random.default_rng(8).standard_normal(p.ndof) * free
    return p, u, b


def _true_residual(dev, p, b, x):
    outer, inner, vals = dev.csc(capi.DBC_FULL)
    return np.linalg.norm(b - sp.csc_matrix((vals, inner, outer), shape=(p.ndof, p.ndof)) @ x) / np.linalg.norm(b)


@pytest.mark.parametrize("n", [(1, 1, 1), (5, 4, 3), (24, 24, 24)])
@pytest.mark.parametrize("max_iter", [1, 2, 16, 17, 32, 33, 50])
def test_iteration_limits(n, max_iter):
    """A solve that ends at its limit reports as many iterations, and the residual of the recurrence is that of the
    iterate (to 1e-10: rounding of at most 50 updates at condition below 1e4; an iterate and a residual of different
    iterations differ by far more). One that converges before takes the oracle's iterations within 1."""
    print(f"case: pcg limit n={n} max_iter={max_iter}", flush=True)
    p, u, b = _setup(n)
    dev = ia.Device(p)
    dev.set_requirement(u, 0.5)
    dev.matrix(capi.DBC_FULL, capi.FP64)
    x, info = dev.solve(b, ia.solver_opts(rtol=1e-10, max_iter=max_iter))
    assert abs(info.rel_residual - _true_residual(dev, p, b, x)) < 1e-10
    if info.rel_residual > 1e-10:
        assert info.iterations == max_iter
    else:
        assert abs(info.iterations - _oracle_for(p).cg(u, 0.5, b, tol=1e-10, max_iter=max_iter)[1]) <= 1
    dev.close()


@pytest.mark.parametrize("kind,n,shuffle", [
    (capi.PCG_JACOBI_FP64, (2, 2, 1), False),
    (capi.PCG_JACOBI_FP64, (24, 24, 23), False),       # 15,000 nodes
    (capi.PCG_JACOBI_FP64, (24, 24, 23), True),
    (capi.PCG_JACOBI_FP64, (24, 24, 24), True),
    (capi.PCG_BJACOBI_FP32_IR, (2, 2, 1), False),
    (capi.PCG_BJACOBI_FP32_IR, (24, 49, 39), False),   # 50,000 nodes
    (capi.PCG_BJACOBI_FP32_IR, (24, 49, 39), True),
    (capi.PCG_BJACOBI_FP32_IR, (36, 36, 36), True),
    (capi.PCG_BJACOBI_FP32_IR, (48, 48, 49), False),   # 120,050 nodes
])
def test_residual_at_the_splits(kind, n, shuffle):
    """b - K x with the assembled matrix, in host FP64: within the tolerance of the solve, plus 1e-11 ||b|| for rounding
    (condition below 1e4, a few hundred iterations)."""
    print(f"case: pcg split kind={kind} n={n} shuffle={shuffle}", flush=True)
    p, u, b = _setup(n, shuffle)
    dev = ia.Device(p)
    dev.set_requirement(u, 0.5)
    dev.matrix(capi.DBC_FULL, capi.FP64 if kind == capi.PCG_JACOBI_FP64 else capi.FP32)
    x, info = dev.solve(b, ia.solver_opts(kind=kind, rtol=1e-9, inner_rtol=1e-3))
    assert info.converged == 1
    assert _true_residual(dev, p, b, x) <= 1e-9 + 1e-11
    again, _ = dev.solve(b, ia.solver_opts(kind=kind, rtol=1e-9, inner_rtol=1e-3))
    assert np.array_equal(x, again)  # fixed summation order
    dev.close()


@pytest.mark.parametrize("kind", [capi.PCG_BJACOBI_FP32_IR, capi.PCG_TWOLEVEL_FP32_IR])
@pytest.mark.parametrize("max_iter", [1, 2, 16, 17])
def test_mixed_iterate_at_the_limit(kind, max_iter):
    """After any number of inner iterations of one sweep the iterate is orthogonal to its residual (conjugate gradients
    minimise over the directions, which span it): to 1e-4 in FP32, with 13^3 nodes in several workgroups."""
    print(f"case: mixed limit kind={kind} max_iter={max_iter}", flush=True)
    p, u, b = _setup((12, 12, 12))
    dev = ia.Device(p)
    dev.set_requirement(u, 0.5)
    dev.matrix(capi.DBC_FULL, capi.FP32)
    x, info = dev.solve(b, ia.solver_opts(kind=kind, rtol=1e-12, inner_rtol=1e-9, max_iter=max_iter, max_refine=1))
    outer, inner, vals = dev.csc(capi.DBC_FULL)
    r = b - sp.csc_matrix((vals, inner, outer), shape=(p.ndof, p.ndof)) @ x
    assert np.linalg.norm(r) / np.linalg.norm(b) == pytest.approx(info.rel_residual, rel=1e-9)
    assert abs(x @ r) < 1e-4 * np.linalg.norm(x) * np.linalg.norm(r)
    dev.close()
