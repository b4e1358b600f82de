"""Solves that outlast 24 iterations with a quarter of their right-hand sides or
fewer left: one hard cell among easy ones, so that the launches are sized anew
for it (FP64, mixed, and mixed with the PCG updates inside the fine launches,
whose vectors are larger than 256 MB).  The sizes set the order of the dot
partials and change after fixed numbers of iterations, so replays, single
launches and any check_every give the same bits; the dense operator and a cell
by itself, whose launches are not sized anew for six right-hand sides, give the
same C_H within the solver's tolerance."""
import numpy as np
import pytest

from fem_amd import Homogenizer
from fem_amd import workloads as W

pytestmark = pytest.mark.gpu

HARD = 2


def cells(shape, n, p):
    E = [W.binary_modulus(W.binary_cube(shape, 9 + s, p=0.7), 1.0, 0.3) for s in range(n)]
    E[HARD] = W.binary_modulus(W.binary_cube(shape, 40 + HARD, p=p), 1.0, 1e-3)
    return np.stack(E)


@pytest.mark.parametrize("shape,n,p,kw", [
    ((24, 20, 28), 6, 0.3, dict(tol=1e-11)),
    ((32, 32, 32), 4, 0.3, dict(tol=1e-11, nu1=1, nu2=1)),
    ((24, 20, 28), 6, 0.3, dict(precision="mixed", inner_tol=1e-5, tol=1e-8)),
    ((56, 60, 76), 16, 0.45, dict(precision="mixed", inner_tol=1e-5, tol=1e-8, nu1=1, nu2=1)),
])
def test_resized_launches(shape, n, p, kw):
    E = cells(shape, n, p)
    kw = dict(kw, nu=0.3, interp="modulus")
    G = np.random.default_rng(0).standard_normal((n, 6, 6))
    out = []
    for graph, every in ((True, 1), (False, 1), (False, 7)):
        h = Homogenizer(shape, batch=n, graph=graph, check_every=every, **kw)
        C, st = h.homogenize_many(E, modulus=True)
        out.append((C, st, h.gradient(G, nb=n)))
        h.close()
    C, st, g = out[0]
    sweep = [np.array(s["iters"]) / np.array(s["outer"]) for s in st]
    assert sweep[HARD].min() > 4 + max(25, max(v.max() for s, v in enumerate(sweep) if s != HARD)), sweep
    for s in st:
        assert s["fp64_fallback"] == 0 and max(s["relres"]) <= kw["tol"]
    for C2, st2, g2 in out[1:]:
        assert np.array_equal(C, C2) and np.array_equal(g, g2)
        for a, b in zip(st, st2):
            assert a["iters"] == b["iters"] and a["relres"] == b["relres"]
    one = dict(apply_kernel="dense") if n < 16 else {}
    h = Homogenizer(shape, batch=1, **one, **kw)
    for s in (HARD, n - 1):
        C1, s1 = h.homogenize_many(E[s:s + 1], modulus=True)
        # C is quadratic in the fields' error
        assert np.linalg.norm(C[s] - C1[0]) <= max(kw["tol"], 1e-10) * np.linalg.norm(C1[0])
        a, b = np.array(st[s]["iters"]), np.array(s1[0]["iters"])
        assert np.abs(a - b).max() <= 2 + 0.1 * b.max(), (s, a, b)
    h.close()
