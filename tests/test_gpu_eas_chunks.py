"""The EAS tangent where a wavefront takes four elements and the last one fewer, and where a mesh is staged in chunks
that take different numbers of elements per wavefront (4, 2 or 1 by the size of the launch): each element's values must
not depend on it, since a Newton solve mixes R of the R+K pass over chunks with R of the residual-only pass over the
mesh."""
import numpy as np
import pytest

import ikarus_amd as ia
import pyoracle as po
from ikarus_amd import _capi as capi
from ikarus_amd import problems as pb
from test_gpu_eas import _oracle_for, _rel

pytestmark = pytest.mark.gpu


def _state(nel, material):
    p = pb.hex_block(nel, L=nel, material=material, jitter=0.08, seed=23, eas=21)  # unit cubes
    rng = np.random.default_rng(11)
    u = 0.01 * rng.standard_normal(p.ndof) * (1 - p.fixed)
    alpha = 1e-3 * rng.standard_normal((p.ne, 21))
    du = 1e-3 * rng.standard_normal(p.ndof) * (1 - p.fixed)
    return p, u, alpha, du


def _run(p, u, alpha, du, precision=capi.FP64):
    """K, R of the R+K pass and the update from its cache; R of the residual-only pass and the update from its own."""
    dev = ia.Device(p)
    dev.set_alpha(alpha)
    dev.set_requirement(u, 0.8)
    R = dev.assemble(capi.DBC_FULL, precision)
    K = dev.csc()[2]
    dev.update_state(du)
    after = dev.alpha()
    dev.set_alpha(alpha)
    dev.set_requirement(u, 0.8)
    Ronly = dev.vector(capi.DBC_FULL)
    dev.update_state(du)
    afterOnly = dev.alpha()
    dev.close()
    return K, R, after, Ronly, afterOnly


@pytest.mark.parametrize("material", [capi.NEOHOOKE, capi.SVK])
@pytest.mark.parametrize("nel", [(5, 29, 113), (19, 29, 30), (17, 31, 33)])  # 16,385 / 16,530 / 17,391: 1, 2, 3 mod 4
def test_last_wavefront_of_four_is_partial(nel, material):
    print(f"case: eas partial wavefront nel={nel} material={material}", flush=True)
    p, u, alpha, du = _state(nel, material)
    K, R, after, Ronly, afterOnly = _run(p, u, alpha, du)
    o = _oracle_for(p)
    o.set_alpha(alpha)
    # FP64 sums of up to 48 products and the condensation (D's condition up to 1e4) in another order: 1e-10
    assert _rel(K, o.matrix(u, 0.8, po.FULL)) < 1e-10
    assert _rel(R, o.vector(u, 0.8, po.FULL)) < 1e-10
    o.update_state(u, 0.8, du)
    assert _rel(after - alpha, o.alpha() - alpha) < 1e-9
    assert np.array_equal(Ronly, R) and np.array_equal(afterOnly, after)


@pytest.mark.parametrize("material", [capi.NEOHOOKE, capi.SVK])
@pytest.mark.parametrize("nel,chunk", [((17, 31, 33), 17001),   # 17,001 (four each, the last one) and 390 (one each)
                                       ((27, 29, 25), 17000),   # 17,000 (four) and 2,575 (two, the last one)
                                       ((16, 32, 31), 15000),   # 15,000 (two) and 872 (one)
                                       ((33, 35, 31), 16501)])  # 16,501 twice (four) and 2,803 (two)
def test_chunks_of_different_kinds(monkeypatch, nel, chunk, material):
    print(f"case: eas chunks nel={nel} chunk={chunk} material={material}", flush=True)
    p, u, alpha, du = _state(nel, material)
    monkeypatch.delenv("IKARUS_AMD_CHUNK_ELEMENTS", raising=False)
    whole = _run(p, u, alpha, du)
    monkeypatch.setenv("IKARUS_AMD_CHUNK_ELEMENTS", str(chunk))
    cut = _run(p, u, alpha, du)
    for a, b in zip(cut, whole):
        assert np.array_equal(a, b)
    assert np.array_equal(cut[3], cut[1]) and np.array_equal(cut[4], cut[2])


def test_default_chunks():
    """A mesh that is cut into chunks by default (two of 100,949 elements): gathers beside the next chunk's elements, in
    both matrix precisions; R of the R+K pass and of the residual-only pass; the FP32 matrix as the FP64 one rounded."""
    nel = (59, 58, 59)  # 201,898
    print(f"case: eas default chunks nel={nel}", flush=True)
    p, u, alpha, du = _state(nel, capi.NEOHOOKE)
    K, R, after, Ronly, afterOnly = _run(p, u, alpha, du)
    assert np.array_equal(Ronly, R) and np.array_equal(afterOnly, after)
    K32, R32, after32, _, _ = _run(p, u, alpha, du, capi.FP32)
    assert np.array_equal(R32, R) and np.array_equal(after32, after)
    assert np.array_equal(K32, K.astype(np.float32).astype(np.float64))  # staged and summed in FP64, rounded once
