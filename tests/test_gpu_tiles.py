"""The process-wide tile choice of the volume kernel and the tiles a context accepts."""
import numpy as np
import pytest

from fluxo_amd.mesh import box_mesh
from fluxo_amd.native import FX_PREC_FP32_SPLIT, FX_PREC_FP64, Engine, FxError, MhdEngine, volume_tile
from fluxo_amd.workloads import perturbed_orszag_tang, taylor_green

pytestmark = pytest.mark.gpu

TGV = dict(x0=(-np.pi,) * 3, length=(2 * np.pi,) * 3)


def test_tuning_without_alternatives_keeps_the_choice():
    """A context whose form has one tile (another flux, GLM-MHD) leaves the choice that a Ranocha
    context has tuned for the same degree, equations and precision."""
    keys = [(N, par, prec) for N in (2, 3, 4, 5) for par in (False, True) for prec in (FX_PREC_FP64, FX_PREC_FP32_SPLIT)]
    meshes = {N: box_mesh(4, N, **TGV) for N in (2, 3, 4, 5)}

    def tune(make, U):
        e = make()
        e.upload(U)
        best, times = e.tune_volume(reps=2)
        e.close()
        return best, times

    tuned = {}
    for N, par, prec in keys:
        m = meshes[N]
        U = taylor_green(m["Elem_xGP"])
        tuned[N, par, prec], times = tune(
            lambda: Engine(m, volume_flux=32, parabolic=par, mu0=1.0 / 1600, precision=prec), U)
        assert len(times) == 3 and volume_tile(N, par, prec) == tuned[N, par, prec]
    for N, par, prec in keys:
        m = meshes[N]
        for flux in (0, 5):
            _, times = tune(lambda: Engine(m, volume_flux=flux, parabolic=par, mu0=1.0 / 1600, precision=prec),
                            taylor_green(m["Elem_xGP"]))
            assert len(times) == 1
        res = dict(mu=1e-3, eta=1e-3, Pr=0.72) if par else None
        _, times = tune(lambda: MhdEngine(m, resistive=res, precision=prec), perturbed_orszag_tang(m["Elem_xGP"], 3))
        assert len(times) == 1
    assert {k: volume_tile(*k) for k in keys} == tuned


ACCEPTED = {(2, FX_PREC_FP64): {7, 14, 3}, (3, FX_PREC_FP64): {1, 4, 2, 8}, (4, FX_PREC_FP64): {5, 2, 3},
            (5, FX_PREC_FP64): {3, 1, 2}, (2, FX_PREC_FP32_SPLIT): {7, 14, 3}, (3, FX_PREC_FP32_SPLIT): {4, 2, 8},
            (4, FX_PREC_FP32_SPLIT): {5, 2, 3}, (5, FX_PREC_FP32_SPLIT): {3, 1, 2}}


@pytest.mark.parametrize("N,precision", list(ACCEPTED))
@pytest.mark.parametrize("parabolic", [False, True])
def test_every_accepted_tile_gives_the_same_steps(N, precision, parabolic):
    """Also a tile that the tuner does not time (8 at N = 3 in FP64); 27 elements leave the last block
    partly filled, or are fewer than two blocks."""
    m = box_mesh(3, N, Ngeo=3, warp=True, **TGV)
    U = taylor_green(m["Elem_xGP"])
    e = Engine(m, volume_flux=32, parabolic=parabolic, mu0=1.0 / 1600, precision=precision)
    results = {}
    for epb in range(17):
        try:
            e.use_volume_tile(epb)
        except FxError:
            continue
        e.upload(U)
        t, dt, err = e.run(3, 0.5, 0.5)
        assert err == 0
        results[epb] = e.download()
    e.close()
    assert set(results) == ACCEPTED[N, precision]
    first = next(iter(results.values()))
    assert all(np.array_equal(V, first) for V in results.values())
