"""The multigrid option on a grid with an odd edge: one level only, so the
solve is Jacobi-PCG and equals that preconditioner's result."""
import numpy as np
import pytest

from fem_amd import Homogenizer
from fem_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape", [(9, 7, 5), (8, 8, 7), (3, 3, 3)])
def test_one_level_multigrid_is_jacobi(shape, precision):
    rho = W.simp_density(shape, 3, 1.5, rho_min=0.1)
    ref = O.homogenize(W.simp_modulus(rho), 0.3, precond="jacobi", tol=1e-12)["C"]
    h = Homogenizer(shape, nu=0.3, precision=precision, tol=1e-10)
    C, st = h.homogenize(rho)
    h.close()
    assert st["levels"] == 1
    assert np.linalg.norm(C - ref) <= 1e-10 * np.linalg.norm(ref)
