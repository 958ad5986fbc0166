"""The node form of the FP64 volume kernel (N >= 3) against the oracle, on meshes whose element count
leaves the last block partly filled (or one element alone), in its three forms (VolInt alone,
right-hand side, LSERK stage), with the Ranocha flux (halved metrics) and one that takes them
whole, and blended with the sub-cell scheme.  Bars: the right-hand-side bar 1e-12 of the repository
(2e-12 at N = 5) and 1e-12 for one step."""
import numpy as np
import pytest

import pyoracle as O
from fluxo_amd.mesh import box_mesh
from fluxo_amd.native import Engine
from fluxo_amd.workloads import density_wave

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("N", [3, 4, 5])
@pytest.mark.parametrize("K", [(1, 1, 1), (3, 1, 1), (2, 2, 2), (3, 3, 1)])
@pytest.mark.parametrize("flux,nfvse", [(32, False), (32, True), (10, False)])
def test_node_form_against_oracle(N, K, flux, nfvse):
    m = box_mesh(K, N, length=(2.0,) * 3, Ngeo=2, warp=True, amp=0.04)
    U = density_wave(m["Elem_xGP"], advvel=(0.7, -0.4, 0.9), amp=0.3)
    kw = dict(nfvse=True, fixed_alpha=0.3) if nfvse else {}
    P = O.Problem(m, volflux=flux, riemann=1, **kw)
    bar = 2e-12 if N == 5 else 1e-12
    e = Engine(m, volume_flux=flux, riemann=1, **kw)
    e.upload(U)
    assert rel(e.volint(), P.volint(U)) <= bar
    assert rel(e.rhs(), P.rhs(U)) <= bar
    dt, _ = P.calc_dt(U, 0.5)
    e.rk_step(0.0, dt)
    V, T = U.copy(), np.zeros_like(U)
    P.lserk_step(V, T, 0.0, dt)
    assert rel(e.download(), V) <= 1e-12
    e.close()
