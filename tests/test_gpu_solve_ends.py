"""The ends of the two solves: the step's totals, whichever way a loop ends (at its
minimum, later, at its cap, without an iteration), and the CFL step size from the
velocity bound's block maxima."""
import numpy as np
import pytest

import splishsplash_for_cuda_amd as S
from splishsplash_for_cuda_amd import scene

pytestmark = pytest.mark.gpu
H = 0.001


def _solver(n_side=11, **kw):
    sc = scene.small_dam_break(nx=n_side, ny=13, nz=9)
    p = S.default_params(particle_radius=sc.particle_radius, dt=H, **kw)
    s = S.Solver(p)
    s.upload_boundary(sc.boundary)
    # denser than at rest and moving, so that both solvers have work
    rng = np.random.default_rng(3)
    s.upload_fluid((sc.fluid * np.float32(0.92)).astype(np.float32),
                   rng.normal(scale=0.5, size=sc.fluid.shape).astype(np.float32))
    s.neighbor_search()
    return s


@pytest.mark.parametrize("max_iter, max_error, expect", [(0, 0.0, 0), (1, 0.0, 1), (3, 0.0, 3), (3, 1e9, 3), (9, 0.0, 9),
                                                         (100, 1e9, 3), (100, 0.5, None)])
def test_divergence_totals(max_iter, max_error, expect):
    """No warm start on the first step: the total is the increments' sum times h, once."""
    s = _solver()
    it, err = s.divergence_solve(max_iter, max_error)
    assert it == expect if expect is not None else it >= 3
    inc, tot = s.download(S.FIELD_KAPPAV), s.download(S.FIELD_KAPPAV_TOTAL)
    assert np.array_equal(tot, inc * np.float32(H))
    assert (max_iter == 0) == (not inc.any())
    s.close()


@pytest.mark.parametrize("max_iter, max_error, expect", [(0, 0.0, 0), (1, 0.0, 1), (2, 0.0, 2), (2, 1e9, 2), (7, 0.0, 7),
                                                         (100, 1e9, 2)])
def test_density_totals(max_iter, max_error, expect):
    s = _solver()
    s.compute_density_factor()
    it, err = s.pressure_solve(max_iter, max_error)
    assert it == expect
    inc, tot = s.download(S.FIELD_KAPPA), s.download(S.FIELD_KAPPA_TOTAL)
    assert np.array_equal(tot, inc * (np.float32(H) * np.float32(H)))
    assert inc.any()
    s.close()


@pytest.mark.parametrize("n", [1, 512, 513, 5000])
def test_cfl_over_block_maxima(n):
    """h = 0.4 * 2r / max |v + a h|, the fastest particle in the last block or the first."""
    sc = scene.small_dam_break(nx=20, ny=20, nz=13)
    for fast in (0, n - 1):
        s = S.Solver(S.default_params(particle_radius=sc.particle_radius, dt=H, viscosity=0.0))
        s.upload_boundary(sc.boundary)
        v = np.random.default_rng(n).normal(scale=0.1, size=(n, 3)).astype(np.float32)
        v[fast] = (30.0, 4.0, -3.0)
        s.upload_fluid(sc.fluid[:n], v)
        s.neighbor_search()
        s.compute_density_factor()
        s.external_forces()
        dt = s.cfl(1e-6, 1.0, 1.0)
        w = v.astype(np.float64) + np.array([0.0, -9.81, 0.0]) * H
        want = 0.4 * 2.0 * sc.particle_radius / np.sqrt((w ** 2).sum(1).max())
        assert dt == pytest.approx(want, rel=1e-6)
        assert s.cfl(1e-6, 1.0, 1.0) == dt
        s.close()


@pytest.mark.parametrize("dropped", [0, 1, 500, "all but one"])
def test_counts_between_steps(dropped):
    """Counts the host waits for (removals, loaded fluid) between steps whose state is
    waited for too; loaded particles take the mass of fluid particle 0."""
    s = _solver()
    s.step()
    n = len(s.download(S.FIELD_ID))
    keep = np.ones(n, np.uint8)
    keep[np.random.default_rng(5).permutation(n)[:n - 1 if dropped == "all but one" else dropped]] = 0
    ids = s.download(S.FIELD_ID)
    assert s.remove_particles(keep) == keep.sum()
    assert np.array_equal(s.download(S.FIELD_ID), ids[keep == 1])
    r = 0.025
    cand = np.array([[0.75, 1.0, 0.3], [0.8, 1.0, 0.3], [0.85, 1.0, 0.3]], np.float32)   # above the block
    assert s.load_fluid(np.concatenate([cand, s.download(S.FIELD_POS)[:1]]), 0.5 * r, 1e9) == 3
    m = s.download(S.FIELD_MASS)
    assert len(m) == keep.sum() + 3 and np.array_equal(m[-3:], np.repeat(m[0], 3))
    st = s.step()
    assert st.n_fluid == len(m) and st.iters >= 2
    s.close()
