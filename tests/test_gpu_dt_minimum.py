"""CALCTIMESTEP's minimum over the elements, at element counts around the pieces in which one block reads
the per-element values: the element with the smallest time step, and the one with an error, first and
last, against the oracle."""
import numpy as np
import pytest

import pyoracle as O
from fluxo_amd.mesh import box_mesh
from fluxo_amd.native import Engine, MhdEngine

pytestmark = pytest.mark.gpu

COUNTS = [1, 1023, 1025, 3 * 1024 + 1, 7 * 1024, 8 * 1024 + 1, 15 * 1024 + 1]


@pytest.mark.parametrize("mhd", [False, True])
@pytest.mark.parametrize("count", COUNTS)
def test_minimum_and_error_anywhere(count, mhd):
    m = box_mesh((count, 1, 1), 2, length=(float(count), 1.0, 1.0))
    U = np.zeros((count, 3, 3, 3, 9 if mhd else 5))
    U[..., 0] = 1.0
    U[..., 4] = 2.0 + 0.1 * np.cos(np.arange(count))[:, None, None, None]
    e = MhdEngine(m) if mhd else Engine(m)
    P = O.MhdProblem(m) if mhd else O.Problem(m, volflux=32, riemann=1)
    scales = (0.5, 0.5) if mhd else (0.5,)
    for at in {0, count // 2, count - 1}:
        V = U.copy()
        V[at, ..., 4] = 9.0
        e.upload(V)
        dt, err = e.calc_dt(0.5, 0.5)
        assert err == 0 and dt == pytest.approx(P.calc_dt(V, *scales)[0], rel=1e-12)
        V[at, 0, 0, 0, 0] = np.nan
        e.upload(V)
        assert e.calc_dt(0.5, 0.5)[1] == 1
    e.close()
