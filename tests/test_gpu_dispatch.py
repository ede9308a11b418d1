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
