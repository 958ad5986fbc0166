"""The node forms of the volume kernels (FP64 Euler at N >= 3, GLM-MHD) against the oracle, on meshes whose element count
leaves the last block partly filled (or one element alone), in its three forms (VolInt alone,
right-hand side, LSERK stage), with the Ranocha flux (halved metrics) and one that takes them
whole, and blended with the sub-cell scheme.  Bars: the right-hand-side bar 1e-12 of the repository
(2e-12 at N = 5) and 1e-12 for one step."""
import numpy as np
import pytest

import pyoracle as O
from fluxo_amd.mesh import box_mesh
from fluxo_amd.native import FX_PREC_FP32_SPLIT, FX_PREC_FP64, Engine, MhdEngine
from fluxo_amd.workloads import density_wave, perturbed_orszag_tang

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


# at each degree up to its largest mesh of three threads a node, and the first ones with one
MHD_MESHES = [(N, K) for N in (2, 3, 4, 5) for K in ((1, 1, 1), (2, 2, 2), (3, 5, 1))] + [
    (2, (16, 8, 8)), (2, (41, 5, 5)), (3, (8, 8, 8)), (3, (19, 9, 3)), (4, (8, 8, 4)), (4, (13, 5, 4))]


@pytest.mark.parametrize("N,K", MHD_MESHES)
@pytest.mark.parametrize("resistive", [False, True])
def test_mhd_node_form_against_oracle(N, K, resistive):
    """The GLM-MHD volume kernel in FP64 (bar 1e-12) and FP32-split (2e-5: FP32 rounding of
    magnitude 6e-8 through differences of O(100) operator entries) on partly filled blocks."""
    m = box_mesh(K, N, Ngeo=2, warp=True, length=(1.0,) * 3, amp=0.04)
    U = perturbed_orszag_tang(m["Elem_xGP"], 3, amp=0.05)
    U[..., 8] = 0.02 * np.sin(2.0 * np.pi * m["Elem_xGP"][..., 0])
    res = dict(mu=1e-3, eta=2e-3, Pr=0.72) if resistive else None
    P = O.MhdProblem(m, resistive=res)
    ref = P.rhs(U)
    for precision, bar in ((FX_PREC_FP64, 1e-12), (FX_PREC_FP32_SPLIT, 2e-5)):
        e = MhdEngine(m, resistive=res, precision=precision)
        e.upload(U)
        assert rel(e.rhs(), ref) <= bar
        e.close()
    dt, _ = P.calc_dt(U, 0.5, 0.5)
    e = MhdEngine(m, resistive=res)
    e.upload(U)
    assert e.calc_dt(0.5, 0.5)[0] == pytest.approx(dt, rel=1e-12)
    e.rk_step(0.0, dt)
    V, T = U.copy(), np.zeros_like(U)
    P.lserk_step(V, T, dt)
    assert rel(e.download(), V) <= 1e-12
    e.close()
