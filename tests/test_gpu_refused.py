"""A refused cell leaves no hierarchy behind: after a call that raised on its
moduli or its operator, the level calls report that there is none, no launch
shape has been timed on it, and the next good cell is solved as on a fresh
context."""
import ctypes

import numpy as np
import pytest

from fem_amd import FemhError, Homogenizer, lib
from fem_amd import workloads as W
from fem_amd.femh import BAD_ARG, NO_FIELDS, NONFINITE

pytestmark = pytest.mark.gpu

SHAPE = (8, 12, 16)
GOOD = W.binary_modulus(W.binary_cube(SHAPE, 1, p=0.6), 1.0, 1e-3)


def bad(kind):
    E = GOOD.copy()
    if kind == "void":
        E[:] = 0.0
    else:
        E[1, 2, 3] = {"nan": np.nan, "inf": np.inf, "negative": -0.5}[kind]
    return E


def no_hierarchy(h):
    u = np.zeros(3 * int(np.prod(SHAPE)))
    p = u.ctypes.data_as(ctypes.c_void_p)
    assert h.level_dims(0) is None
    assert lib().femh_apply_level(h._h, 0, p, p) == NO_FIELDS


@pytest.mark.parametrize("kind,status", [("nan", NONFINITE), ("inf", NONFINITE), ("negative", BAD_ARG),
                                         ("void", BAD_ARG)])
@pytest.mark.parametrize("precision,precond", [("fp64", "mg"), ("mixed", "mg"), ("fp64", "jacobi")])
def test_refused_moduli(precision, precond, kind, status):
    kw = dict(nu=0.3, interp="modulus", precision=precision, precond=precond)
    h = Homogenizer(SHAPE, **kw)
    h.prepare(GOOD)
    assert h.level_dims(0) == SHAPE
    with pytest.raises(FemhError) as e:
        h.homogenize_modulus(bad(kind))
    assert e.value.status == status
    no_hierarchy(h)
    C, _ = h.homogenize_modulus(GOOD)
    assert h.level_dims(0) == SHAPE
    fresh = Homogenizer(SHAPE, **kw)
    assert np.array_equal(C, fresh.homogenize_modulus(GOOD)[0])
    fresh.close()
    h.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("E", [bad("nan"), bad("void"), -GOOD], ids=["nan", "void", "all negative"])
def test_refused_operator(E, precision):
    h = Homogenizer(SHAPE, nu=0.3, interp="modulus", precision=precision)
    with pytest.raises(FemhError) as e:
        h.prepare(E)
    assert e.value.status == NONFINITE
    no_hierarchy(h)
    h.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_refused_cell_is_not_timed(precision):
    h = Homogenizer(SHAPE, nu=0.3, interp="modulus", precision=precision, autotune=True)
    with pytest.raises(FemhError):
        h.homogenize_modulus(bad("nan"))
    assert h.launch_shapes() == [0]  # as before the first call
    h.homogenize_modulus(GOOD)
    assert len(h.launch_shapes()) == 3
    h.close()
