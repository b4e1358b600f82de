"""Dense coarsest inverse: grids whose coarsest level has 24 (one LDS matrix),
96, 135 (partial last panel), 375 and 648 (the largest) unknowns, two cells
per call.  C_H equals the oracle's, and the iteration counts stay near those
of the oracle's own multigrid with the same levels and its own exact coarsest
solve (smoothers and lambda_max factors differ, hence the factor 1.5): a wrong
inverse is a poor preconditioner."""
import numpy as np
import pytest

from fem_amd import Homogenizer
from fem_amd import workloads as W
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("shape,levels", [((8, 8, 8), 0), ((4, 4, 16), 2), ((6, 6, 10), 0), ((10, 10, 10), 0),
                                          ((12, 12, 12), 2)])
def test_dense_coarsest_inverse(shape, levels, precision):
    E = np.stack([W.binary_modulus(W.binary_cube(shape, s, p=0.6), 1.0, 1e-3) for s in (1, 2)])
    h = Homogenizer(shape, nu=0.3, interp="modulus", levels=levels, precision=precision, tol=1e-10, batch=2)
    C, st = h.homogenize_many(E, modulus=True)
    h.close()
    for s in range(2):
        ref = O.homogenize(E[s], 0.3, precond="mg", tol=1e-12)
        assert np.linalg.norm(C[s] - ref["C"]) <= 1e-10 * np.linalg.norm(ref["C"])
        if precision == "fp64":
            it = O.homogenize(E[s], 0.3, precond="mg", tol=1e-10, cheby_ratio=20.0, levels=levels or 16)["iters"]
            assert max(st[s]["iters"]) <= 1.5 * max(it) + 2, (st[s]["iters"], it)


@pytest.mark.parametrize("shape,levels", [((8, 8, 8), 0), ((4, 4, 16), 2), ((6, 6, 10), 0), ((10, 10, 10), 0),
                                          ((12, 12, 12), 2)])
def test_fp32_inverse_preconditions_as_the_fp64_one(shape, levels):
    # correction sweeps of 1e-4 each: as many iterations as the same decades take
    # in FP64, and a few at each of the (at most four) restarts; C alone would not
    # show a poor inverse, since more sweeps or the FP64 fallback make up for it
    E = np.stack([W.binary_modulus(W.binary_cube(shape, s, p=0.6), 1.0, 1e-3) for s in (1, 2)])
    st = {}
    for precision in ("fp64", "mixed"):
        h = Homogenizer(shape, nu=0.3, interp="modulus", levels=levels, precision=precision, tol=1e-10, batch=2)
        st[precision] = h.homogenize_many(E, modulus=True)[1]
        h.close()
    for a, b in zip(st["mixed"], st["fp64"]):
        assert a["fp64_fallback"] == 0 and max(a["outer"]) <= 4
        assert max(a["iters"]) <= 2 * max(b["iters"]) + 10, (a["iters"], b["iters"])
