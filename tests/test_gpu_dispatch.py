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
                                          (256, 65, 32), (64, 33, 64), (192, 40, 64)])
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


@pytest.mark.parametrize("prec", [32, 64])
def test_force_on_a_384_mesh(prec):
    """The largest radix (24) and, in FP32, the persistent z pass with four lines to a wave.  FP32 positions in
    cells round to 384 2^-24, the deposit and the gather see that shift once each and the force turns over within
    a cell: 4 times it bounds the relative error."""
    res, n = 384, 96
    L = 2.0 * res
    dt = np.float32 if prec == 32 else np.float64
    psi = _psi(n, 3.0, 5, dt)
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L), precision=prec) as S:
        acc = S.pm_acceleration(psi)
    ref = O.pm_acceleration(psi.astype(np.float64), O.pm_config(res, n, L, worder=2, grad_order=4), "solver")
    assert G.rel(acc, ref) < (4 * res * 2.0**-24 if prec == 32 else 1e-12)


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


def _collapse(n, L, dt):
    """Momenta that carry every particle close to the box centre at time 1, a little apart."""
    q = np.arange(n) * (L / n)
    q3 = np.stack([np.broadcast_to(v, (n, n, n)) for v in (q, q[:, None], q[:, None, None])])
    return (0.97 * (L / 2 - q3)).astype(dt)


@pytest.mark.parametrize("aa, prec, grad", [(0, 32, 2), (1, 32, 4), (1, 64, 2), (0, 64, 0)])
def test_run_resumes_at_a_sort_that_overflows(aa, prec, grad):
    """Particles that pile up in a few tiles between two steps of a run overflow the lists reserved from the
    step before; the run goes back to that step.  The same steps one at a time, each call on a new solver
    (whose first sort counts), give the same state: bit for bit in FP32, whose deposit sums in integers, to
    1e-11 in FP64, whose atomics add in any order."""
    n, res, L, steps = 32, 64, 100.0, 6
    dt = np.float32 if prec == 32 else np.float64
    psi, pi = 0.5 * _psi(n, 1.0, 5, dt), _collapse(n, L, dt)
    cfg = D.PMConfig(res_pm=res, n_part=n, boxsize=L, grad_order=grad, antialias=aa)
    dd1, dd2 = np.full(steps, 0.125), np.full(steps, 0.125)
    alpha, beta = np.full(steps, 0.99), np.full(steps, 1e-3)
    with D.PMSolverHIP(cfg, precision=prec) as S:
        S.set_state(psi, pi)
        S.run(dd1, alpha, beta, dd2)
        got = S.get_state()
        seen = []
        S.set_state(psi, pi)
        S.run(dd1, alpha, beta, dd2, want=[0, 0, 1, 0, 1, 0, 0], callback=lambda k: seen.append((k, S.get_state())))
        again = S.get_state()
    ref, refs = (psi, pi), []
    for s in range(steps):
        with D.PMSolverHIP(cfg, precision=prec) as S:
            S.set_state(*ref)
            S.step(dd1[s], alpha[s], beta[s], dd2[s])
            ref = S.get_state()
            refs.append(ref)
    tol = 0 if prec == 32 else 1e-11
    for a, b in ((got, ref), (again, ref), (seen[0][1], refs[1]), (seen[1][1], refs[3])):
        assert G.rel(a[0], b[0]) <= tol and G.rel(a[1], b[1]) <= tol
    assert [k for k, _ in seen] == [2, 4]


@pytest.mark.parametrize("prec", [32, 64])
def test_calls_after_a_state_that_does_not_fit_the_lists(prec):
    """A force and a step of collapsed particles on a solver whose lists are reserved for uniform ones, against
    a new solver's (bit for bit in FP32, 1e-11 in FP64)."""
    n, res, L = 32, 64, 100.0
    dt = np.float32 if prec == 32 else np.float64
    psi = 0.5 * _psi(n, 1.0, 6, dt)
    piled = (psi + _collapse(n, L, dt)).astype(dt)
    pi = _psi(n, 0.1, 7, dt)
    cfg = D.PMConfig(res_pm=res, n_part=n, boxsize=L)
    with D.PMSolverHIP(cfg, precision=prec) as S:
        S.pm_acceleration(psi)
        acc = S.pm_acceleration(piled)
        back = S.pm_acceleration(psi)
        S.set_state(piled, pi)
        S.step(0.0, 0.9, 0.1, 0.2)
        st = S.get_state()
    with D.PMSolverHIP(cfg, precision=prec) as S:
        acc0 = S.pm_acceleration(piled)
    with D.PMSolverHIP(cfg, precision=prec) as S:
        back0 = S.pm_acceleration(psi)
        S.set_state(piled, pi)
    with D.PMSolverHIP(cfg, precision=prec) as S:
        S.set_state(piled, pi)
        S.step(0.0, 0.9, 0.1, 0.2)
        st0 = S.get_state()
    tol = 0 if prec == 32 else 1e-11
    assert G.rel(acc, acc0) <= tol and G.rel(back, back0) <= tol
    assert G.rel(st[0], st0[0]) <= tol and G.rel(st[1], st0[1]) <= tol


@pytest.mark.parametrize("res, n, prec", [(256, 40, 32), (384, 40, 32), (192, 40, 64)])
def test_sort_over_the_scan_rule(res, n, prec):
    """Meshes on both sides of the one-workgroup scan (4096, 13824 and 1728 tiles): the deposit of two calls,
    the second from reserved lists, against the oracle's in the same precision (an FP64 one would count the
    rounding of the FP32 positions, up to 384 x 2^-23 of a cell)."""
    L = 1.5 * res
    dt = np.float32 if prec == 32 else np.float64
    psi = _psi(n, 2.0, res, dt)
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L), precision=prec) as S:
        S.deposit(psi)
        m = S.deposit(psi)
    ref = O.pm_scatter(O.lagrangian_positions(psi, L), res, L, 2)
    assert G.rel(m, ref) < (2e-5 if prec == 32 else 1e-12)


@pytest.mark.parametrize("W", [2, 3, 4])
@pytest.mark.parametrize("res, n, aa, prec", [(16, 9, 0, 32), (64, 30, 1, 32), (96, 33, 2, 32), (64, 31, 1, 64),
                                              (128, 32, 3, 32)])
def test_spectral_force_over_tiles(W, res, n, aa, prec):
    """The tiled interpolation of the spectral gradient's force meshes: regions as large as the mesh (16^3),
    the compile-time regions of FP32, reaches they do not cover (antialias 3) and FP64, against the oracle."""
    L = 2.0 * res
    dt = np.float32 if prec == 32 else np.float64
    psi = _psi(n, 3.0, res + W, dt)
    acc = D.pm_acceleration(psi, D.PMConfig(res_pm=res, n_part=n, boxsize=L, worder=W, grad_order=0, antialias=aa),
                            precision=prec)
    # the oracle's force in the same precision's positions: FP32 rounds the weights' coordinates (res 2^-24 of a
    # cell each), the meshes and the transforms
    ref = O.pm_acceleration(psi, O.pm_config(res, n, L, worder=W, grad_order=0, antialias=aa), "solver")
    assert G.rel(acc, ref) < (2e-5 if prec == 32 else 1e-12)


@pytest.mark.parametrize("W, n, res, aa, prec", [(2, 7, 16, 1, 64), (2, 128, 128, 0, 32), (2, 129, 128, 1, 32),
                                                 (3, 64, 64, 1, 64), (3, 65, 64, 1, 64), (4, 48, 96, 1, 32),
                                                 (4, 49, 64, 0, 64)])
def test_resampled_spectral_force_over_the_order_rule(W, n, res, aa, prec):
    """The spectral gradient with sheet resampling, interpolated in particle order up to a number of particles and
    from the tiles above it, against the oracle (the bounds of test_resampling_vs_oracle)."""
    L = 2.0 * res
    psi = _psi(n, 2.0, n + W, np.float32 if prec == 32 else np.float64)
    kw = dict(worder=W, grad_order=0, antialias=aa, n_resample=2, resampling="linear")
    acc = D.pm_acceleration(psi, D.PMConfig(res_pm=res, n_part=n, boxsize=L, **kw), precision=prec)
    ref = O.pm_acceleration(psi.astype(np.float64), O.pm_config(res, n, L, **kw), "solver")
    assert G.rel(acc, ref) < (1e-12 if prec == 64 else 5e-5)


@pytest.mark.parametrize("n, order, prec", [(16, 2, 32), (24, 1, 64), (48, 1, 32), (96, 1, 64), (128, 2, 64), (192, 1, 64)])
def test_ics_over_the_transform_sizes(n, order, prec):
    """Displacements and momenta of the ICs at sizes whose line groups differ (1e-12, or FP32's rounding of the
    results), and the reverse pass as their transpose: a central difference along one direction is exact up to
    rounding, the ICs being quadratic in the noise."""
    L, a, eps = 2.0 * n, 0.05, 1e-3
    rng = np.random.default_rng(n)
    white, v = rng.normal(size=(n, n, n)), rng.normal(size=(n, n, n))
    pb, mb = rng.normal(size=(3, n, n, n)), rng.normal(size=(3, n, n, n))
    oc = O.Cosmology(0.2621, 0.049, 0.6766, 0.8102, 0.9665)
    k, pk = O.linear_power_spectrum(oc)
    psi1, psi2 = O.compute_core2(O.white_noise_to_fphi(O.ic_operator(n, L, k, pk), white), L)
    psi_ref, pi_ref = O.nbody_ics_lpt2(oc, psi1, psi2 if order == 2 else np.zeros_like(psi2), a)
    Dg = oc.Dplus(a)
    with D.PMSolverHIP(D.PMConfig(res_pm=max(n, 32), n_part=n, boxsize=L), precision=prec) as S:
        S.ics_lpt(k, pk, Dg, order=order, white=white)
        psi, pi = S.get_state()
        tol = 1e-12 if prec == 64 else 2e-7
        assert G.rel(psi, psi_ref) < tol and G.rel(pi, pi_ref) < tol
        if prec == 32:
            return
        f = []
        for e in (eps, -eps):
            S.ics_lpt(k, pk, Dg, order=order, white=white + e * v)
            p, m = S.get_state()
            f.append(float(np.vdot(pb, p) + np.vdot(mb, m)))
        wb = S.vjp_ics_lpt(k, pk, Dg, pb, mb, order=order, white=white)
    # the sum's own scale: its two dot products' norms times the direction's
    scale = np.linalg.norm(wb) * np.linalg.norm(v)
    assert abs(float(np.vdot(wb, v)) - (f[0] - f[1]) / (2 * eps)) < 1e-9 * scale


def _calls(S):
    """Launch groups of the solver's last calls (profiling on), by name."""
    return {k: v["calls"] for k, v in S.kernel_stats().items()}


def _collapse_run(cfg, n, steps, net=None):
    """A collapse over some steps in one run, its launch counts, and the same steps one at a time, each on a new
    solver, whose first sort counts: both states.  net: (parameters, output scale, scale factors of the forces)."""
    psi, pi = 0.5 * _psi(n, 1.0, 5, np.float32), _collapse(n, cfg.boxsize, np.float32)
    dd1, dd2 = np.full(steps, 0.125), np.full(steps, 0.125)
    alpha, beta = np.full(steps, 0.99), np.full(steps, 1e-3)

    def ready(S, state, a):
        if net:
            S.nn_set_params(net[0])
            S.nn_enable(True, net[1])
            S.nn_set_schedule(a)
        S.set_state(*state)

    with D.PMSolverHIP(cfg, precision=32) as S:
        ready(S, (psi, pi), net and net[2])
        S.set_profiling(True)
        S.run(dd1, alpha, beta, dd2)
        calls, got = _calls(S), S.get_state()
    ref = (psi, pi)
    for s in range(steps):
        with D.PMSolverHIP(cfg, precision=32) as S:
            ready(S, ref, net and net[2][s:s + 1])
            S.run(dd1[s:s + 1], alpha[s:s + 1], beta[s:s + 1], dd2[s:s + 1])
            ref = S.get_state()
    return calls, got, ref


@pytest.mark.parametrize("res, aa", [(256, 0), (384, 1)])
def test_run_of_a_large_mesh_makes_no_force_in_vain(res, aa):
    """A sort that overflows in a run on a large mesh (4096 tiles, and 13824 with the three-launch scan) is repeated
    before its force is made: the exact sort ran again, and there is one deposit per step and pass."""
    n, steps = 32, 6
    cfg = D.PMConfig(res_pm=res, n_part=n, boxsize=100.0, grad_order=4, antialias=aa)
    calls, got, ref = _collapse_run(cfg, n, steps)
    assert calls["bin_recount"] >= 2 and calls["scatter"] == steps * (1 + aa), calls
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])


@pytest.mark.parametrize("net", [False, True])
def test_run_of_a_small_mesh_goes_back_to_a_sort_that_overflows(net):
    """On a small mesh the overflow is seen after the step's force: the run has made forces in vain, and the steps it
    goes back to take their own place in the learned correction's schedule."""
    n, res, steps, L = 32, 64, 6, 100.0
    cfg = D.PMConfig(res_pm=res, n_part=n, boxsize=L, grad_order=4)
    params = (D.learned.init_params(1, out_std=1.0), (L / res) ** 2, np.linspace(0.3, 0.9, steps)) if net else None
    calls, got, ref = _collapse_run(cfg, n, steps, params)
    assert calls["bin_recount"] >= 2 and calls["scatter"] > steps, calls
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])


@pytest.mark.parametrize("W", [2, 4])
@pytest.mark.parametrize("res, n, prec", [(32, 20, 64), (48, 24, 64), (64, 40, 32), (64, 40, 64), (96, 40, 32)])
def test_deposit_over_the_sharing_rule(res, n, prec, W):
    """Tiles shared by 4, 2 and 1 workgroups (32, 108, 64, 256 and 216 tiles), against the oracle's deposit in the same
    precision."""
    L = 1.5 * res
    psi = _psi(n, 2.0, res + W, np.float32 if prec == 32 else np.float64)
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L, worder=W), precision=prec) as S:
        m = S.deposit(psi)
    assert G.rel(m, O.pm_scatter(O.lagrangian_positions(psi, L), res, L, W)) < (2e-5 if prec == 32 else 1e-12)


@pytest.mark.parametrize("n, W", [(76, 2), (77, 2), (77, 4)])
def test_force_on_both_sides_of_the_gather_sharing_rule(n, W):
    """216 tiles, taken by one workgroup each or, from 2048 particles a tile, by two, against the oracle (the bound of
    test_step_over_the_gather_segment_rule)."""
    res, L = 96, 192.0
    psi = _psi(n, 3.0, n, np.float32)
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L, worder=W), precision=32) as S:
        acc = S.pm_acceleration(psi)
    ref = O.pm_acceleration(psi.astype(np.float64), O.pm_config(res, n, L, worder=W, grad_order=4), "solver")
    assert G.rel(acc, ref) < 2e-5


@pytest.mark.parametrize("n", [46, 47])
@pytest.mark.parametrize("res, prec", [(48, 64), (64, 32)])
def test_lists_on_both_sides_of_the_bin_size_rule(res, prec, n):
    """Bins of 4 and 8 particles a side (up to and from 100000 particles): the deposit through an exact sort and through
    one into reserved lists, against the oracle's in the same precision."""
    L = 1.5 * res
    psi = _psi(n, 2.0, n, np.float32 if prec == 32 else np.float64)
    ref = O.pm_scatter(O.lagrangian_positions(psi, L), res, L, 3)
    with D.PMSolverHIP(D.PMConfig(res_pm=res, n_part=n, boxsize=L, worder=3), precision=prec) as S:
        for m in (S.deposit(psi), S.deposit(psi)):
            assert G.rel(m, ref) < (2e-5 if prec == 32 else 1e-12)
