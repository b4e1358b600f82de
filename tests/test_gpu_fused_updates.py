"""PCG updates inside the fine-level launches (vectors beyond 256 MB): r = r -
alpha q in the pre-smoothing, x = x + alpha p in the next A p.  A full batch on
a grid with partial tiles in both directions, whose cells converge after
different (odd and even) numbers of iterations, against one-cell solves, which keep the update in a pass of its own: the arithmetic of
a right-hand side is the same, only the order of FP64 dot partials differs."""
import numpy as np
import pytest

from fem_amd import Homogenizer
from fem_amd import workloads as W

pytestmark = pytest.mark.gpu

SHAPE = (56, 60, 76)  # 16 cells: a vector of 294 MB


def cells():
    E = [W.binary_modulus(W.binary_cube(SHAPE, s, p=0.3 + 0.04 * s), 1.0, 10.0 ** -(1 + s % 4)) for s in range(16)]
    return np.stack(E)


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("planes", [0, 5])
@pytest.mark.parametrize("tile", [1, 2, 3])
def test_batch_equals_single_solves(tile, planes, graph):
    E = cells()
    kw = dict(nu=0.3, interp="modulus", precision="mixed", tol=1e-8, ch_tol=0.0, graph=graph)
    h = Homogenizer(SHAPE, batch=16, **kw)
    h.set_launch_shapes([(tile << 8) | planes])
    C, st = h.homogenize_many(E, modulus=True)
    h.close()
    assert len({sum(s["iters"]) for s in st}) > 4
    h = Homogenizer(SHAPE, batch=1, **kw)
    for s in (0, 3, 6, 15):
        C1, s1 = h.homogenize_many(E[s:s + 1], modulus=True)
        # (a coefficient that rounds the other way costs at most one iteration a sweep)
        assert np.abs(np.array(st[s]["iters"]) - np.array(s1[0]["iters"])).max() <= 2
        # both within tol of the solution, to which C's error is quadratic
        assert np.linalg.norm(C[s] - C1[0]) <= 1e-8 * np.linalg.norm(C1[0])
    h.close()
