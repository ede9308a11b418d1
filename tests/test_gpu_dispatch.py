"""The sizes at which the device path's launch rules change, against the oracle's FP64 results."""
import numpy as np
import pytest

import golden as G
import oracle as O

pytestmark = pytest.mark.gpu

D = pytest.importorskip("discodj_amd")


def _psi(n, scale, seed, dt):
    return np.random.default_rng(seed).normal(scale=scale, size=(3, n, n, n)).astype(dt)


@pytest.mark.parametrize("res, n, prec", [(16, 7, 32), (64, 33, 32), (96, 50, 32), (128, 40, 32), (192, 64, 32),
                                          (256, 65, 32), (64, 33, 64)])
def test_step_over_the_gather_segment_rule(res, n, prec):
    """One pass, kicked in particle order, on meshes of 8 (tiles shared by workgroups) to 4096 tiles (segments
    of several tiles): Psi and Pi after a step against the oracle's force at the drifted positions.  The
    bounds are the force's (2e-5 FP32, 1e-12 FP64); beta makes the kick the momentum's own size."""
    L = 2.0 * res
    dt = np.float32 if prec == 32 else np.float64
    psi, pi = _psi(n, 3.0, res, dt), _psi(n, 1.0, res + 1, dt)
    dd1, alpha, dd2 = 0.5, 0.75, 0.25
    x = psi.astype(np.float64) + dd1 * pi.astype(np.float64)
    acc = O.pm_acceleration(x.astype(dt).astype(np.float64), O.pm_config(res, n, L, worder=2, grad_order=4), "solver")
    beta = float(1.0 / np.std(acc))
    mom = alpha * pi + beta * acc
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L), precision=prec) as S:
        S.set_state(psi, pi)
        S.step(dd1, alpha, beta, dd2)
        psi1, pi1 = S.get_state()
    tol = 2e-5 if prec == 32 else 1e-12
    assert G.rel(pi1, mom) < tol
    assert G.rel(psi1, x + dd2 * mom) < tol


@pytest.mark.parametrize("N, bins, log", [(16, 1, False), (24, 256, True), (96, 7, True), (128, 256, False)])
def test_spectra_over_runs_and_bins(N, bins, log):
    """Every mode in the oracle's bin and P(k) to 1e-10, for meshes whose x runs end short of N/2 and for one
    bin and the most bins (many of them empty at 24^3)."""
    L = 1.7 * N
    f = np.random.default_rng(N).normal(size=(N, N, N))
    with D.PMSolverHIP(D.PMConfig(res_pm=N, n_part=16, boxsize=L), precision=64) as S:
        k, pk, nm = S.field_power_spectrum(f, bins=bins, logarithmic=log)
    ko, pko, nmo = O.power_spectrum(f, L, bins=bins, logarithmic=log)
    assert np.array_equal(nm, nmo)
    assert np.allclose(k, ko, rtol=1e-12, atol=0)
    ok = nmo > 0
    assert np.max(np.abs(pk[ok] / pko[ok] - 1)) < 1e-10 and np.all(pk[~ok] == 0)
