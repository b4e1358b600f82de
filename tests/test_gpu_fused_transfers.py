"""Fine-level launches that carry the grid transfers (restricted residual,
staged coarse correction): every tile shape, whole and partial tiles, chunks of
one to all planes and tiles wider than the grid give the same iterations and
the same C_H, which is the oracle's.  The values a node receives do not depend
on its tile, so only the order of FP64 dot partials differs between shapes."""
import numpy as np
import pytest

from fem_amd import Homogenizer
from fem_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nu", [1, 2])
@pytest.mark.parametrize("shape", [(4, 4, 4), (6, 18, 34), (20, 16, 32), (10, 34, 66)])
def test_tile_and_chunk_shapes_agree(shape, nu):
    E = np.stack([W.binary_modulus(W.binary_cube(shape, s, p=0.6), 1.0, 1e-3) for s in (1, 2)])
    out = []
    for tile in (1, 2, 3):
        for planes in (0, 1, 4, 64):
            h = Homogenizer(shape, nu=0.3, interp="modulus", tol=1e-11, batch=2, nu1=nu, nu2=nu)
            h.set_launch_shapes([(tile << 8) | planes])
            C, st = h.homogenize_many(E, modulus=True)
            h.close()
            out.append((C, [s["iters"] for s in st]))
    C0, it0 = out[0]
    for C, it in out[1:]:
        assert it == it0
        assert np.abs(C - C0).max() <= 1e-12 * np.abs(C0).max()
    for s in range(2):
        ref = O.homogenize(E[s], 0.3, precond="mg", tol=1e-12)
        assert np.linalg.norm(C0[s] - ref["C"]) <= 1e-10 * np.linalg.norm(ref["C"])
        it = O.homogenize(E[s], 0.3, precond="mg", tol=1e-11, nu1=nu, nu2=nu, cheby_ratio=20.0)["iters"]
        assert max(it0[s]) <= 1.5 * max(it) + 2, (it0[s], it)


@pytest.mark.parametrize("nu", [1, 2])
@pytest.mark.parametrize("shape", [(4, 4, 4), (6, 18, 34), (20, 16, 32), (10, 34, 66)])
def test_tile_and_chunk_shapes_agree_in_fp32(shape, nu):
    # (the FP32 variants, in the mixed path's correction sweeps: a coefficient that
    # rounds the other way costs at most one iteration a sweep, and C's error is
    # quadratic in the residual tolerance)
    E = np.stack([W.binary_modulus(W.binary_cube(shape, s, p=0.6), 1.0, 1e-3) for s in (1, 2)])
    ref = [O.homogenize(E[s], 0.3, precond="mg", tol=1e-12)["C"] for s in range(2)]
    it0 = None
    for tile in (1, 2, 3):
        for planes in (0, 1, 4, 64):
            h = Homogenizer(shape, nu=0.3, interp="modulus", precision="mixed", tol=1e-10, batch=2, nu1=nu, nu2=nu)
            h.set_launch_shapes([(tile << 8) | planes])
            C, st = h.homogenize_many(E, modulus=True)
            h.close()
            assert not any(s["fp64_fallback"] for s in st)
            it = np.array([s["iters"] for s in st])
            it0 = it if it0 is None else it0
            assert np.abs(it - it0).max() <= max(max(s["outer"]) for s in st), (tile, planes, it, it0)
            for s in range(2):
                assert np.linalg.norm(C[s] - ref[s]) <= 1e-10 * np.linalg.norm(ref[s])
