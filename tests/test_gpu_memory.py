"""Device memory of a context: what its first call adds to what its
constructor took."""
import numpy as np
import pytest
import torch

from fem_amd import Homogenizer
from fem_amd import workloads as W

pytestmark = pytest.mark.gpu


def growth(h, E):
    before = torch.cuda.mem_get_info()[0]
    h.homogenize_many(E, modulus=True, check=False)
    return before - torch.cuda.mem_get_info()[0]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_jacobi_call_adds_no_vector(precision):
    """Moduli, diagonals and their inverses only (7 values a voxel and
    precision); a vector of the four cells takes 510 MB in FP64, 255 in FP32."""
    n, cells = 96, 4
    E = np.stack([W.binary_modulus(W.binary_cube(n, s, p=0.7), 1.0, 0.1) for s in range(cells)])
    kw = dict(max_iter=20) if precision == "fp64" else dict(inner_tol=0.4, max_outer=1)  # (no FP64 fallback)
    h = Homogenizer((n, n, n), nu=0.3, interp="modulus", precond="jacobi", precision=precision, batch=cells, **kw)
    levels = 7 * cells * n ** 3 * (8 if precision == "fp64" else 8 + 4)
    got = growth(h, E)
    h.close()
    assert levels / 2 < got < levels + (64 << 20), (got, levels)


def test_dense_inverse_workspace_is_of_the_cells_at_hand():
    """648 coarsest unknowns, one cell in a context for 16: three FP64 matrices
    (10 MB) of workspace, not 16 times three (161 MB)."""
    n, batch, V = 12, 16, 12 ** 3 + 6 ** 3
    E = W.binary_modulus(W.binary_cube(n, 1, p=0.7), 1.0, 0.1)[None]
    h = Homogenizer((n, n, n), nu=0.3, interp="modulus", levels=2, batch=batch)
    got = growth(h, E)
    h.close()
    vectors = (7 * V + n ** 3) * 18 * batch * 8  # seven per level, the second direction
    operators = ((6 * V + 243 * 6 ** 3 + n ** 3) * batch + 648 ** 2 * batch) * 8
    assert got < vectors + operators + 3 * 648 ** 2 * 8 + (64 << 20), (got, vectors, operators)
