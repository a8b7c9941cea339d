"""The FP32C Verlet steps' sums on the matrix cores at the edges of their tiling: grids of three columns
(every row staged with its own images), sparse rows as wide as a tile can be, stages just within and
just past their capacity, a tile with more particles than a workgroup beside empty cells, a few
particles; and what the range test and the digits have to get right: pairs exactly at the radius,
particles that leave their cells across the box's edges between rebuilds, omegas far apart in size,
phases that are not finite.  Reference: the oracle's FP64 steps.

Bounds: a phasor is rounded once to FP32 (2^-25) and its sums are exact from there, so the mean over the
neighbours errs by at most sqrt(2) 2^-25 < 2^-24: sigma dt 2^-24 in omega.  The stochastic Runge-Kutta step
adds dt^2 / 2 of the complementary force, whose terms err by three roundings of 2^-24 of (|omega_j| +
|omega_i|) at most.  The positions and the phases do not depend on the sums in a first step: 1e-12."""
import numpy as np
import pytest

import oracle
from oracle.pyoracle import METHOD_LINKED_LIST_VERLET, VERLET_EXACT

pytestmark = pytest.mark.gpu

SIGMA, DT = 1.5, 0.002


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _lattice(k, m=64):
    g = (np.arange(k) / m) % 1.0
    return np.stack(np.meshgrid(g, g), -1).reshape(-1, 2)


def _layout(name):
    rng = np.random.default_rng(len(name))
    if name == "three_columns":
        return rng.random((300, 2)), 0.27
    if name == "three_columns_dense":
        return rng.random((2500, 2)), 0.27
    if name == "sparse":
        return rng.random((1500, 2)), 0.01
    if name == "few":
        return rng.random((17, 2)), 0.05
    if name == "one":
        return rng.random((1, 2)), 0.1
    if name.startswith("stage"):  # cells of that many particles: three rows of staged cells around a tile
        m, rho = int(name[5:]), 0.05
        ncv = int(1.0 / (1.2 * rho))
        cells = np.stack(np.meshgrid(np.arange(ncv), np.arange(ncv)), -1).reshape(-1, 1, 2)
        return ((cells + rng.random((ncv * ncv, m, 2))) / ncv).reshape(-1, 2), rho
    if name == "lone_cell":
        return np.concatenate([0.5 + 0.019 * rng.random((300, 2)), rng.random((40, 2))]), 0.02
    if name == "at_radius":
        return _lattice(64), 3.0 / 64.0
    raise KeyError(name)


def _systems(spss, xy, rho, v0=0.3, seed=5):
    n = len(xy)
    kw = dict(model=4, n=n, v0=v0, xi=2.0, sigma=SIGMA, rho=rho, alpha=0.4, natfreq_local=1,
              verlet_mode=VERLET_EXACT, verlet_skin=0.2 * rho)
    rng = np.random.default_rng(seed)
    st = np.concatenate([xy, 2 * np.pi * rng.random((n, 1)), rng.normal(0, 1, (n, 1))], 1)
    w = rng.normal(0, 1, n)
    g, o = spss.ParticleSystem(precision=spss.PRECISION_FP32C, **kw), oracle.Oracle(**kw)
    g.set_natural_frequencies(w)
    o.set_natural_frequencies(w)
    return g, o, st


def _step(spss, g, o, st, stepper):
    n = len(st)
    so, z = st.reshape(-1).copy(), np.zeros((1 if stepper == "euler" else 2) * n)
    getattr(o, stepper + "_step")(METHOD_LINKED_LIST_VERLET, so, DT, z)
    getattr(g, stepper + "_step")(spss.METHOD_LINKED_LIST_VERLET, DT, spss.NOISE_NONE)
    return g.get_state().reshape(-1, 4), so.reshape(-1, 4)


@pytest.mark.parametrize("stepper", ["euler", "srk"])
@pytest.mark.parametrize("name", ["three_columns", "three_columns_dense", "sparse", "few", "one", "stage8", "stage26",
                                  "stage29", "stage31", "stage40", "lone_cell", "at_radius"])
def test_first_step(spss, name, stepper):
    xy, rho = _layout(name)
    g, o, st = _systems(spss, xy, rho)
    g.set_state(st.reshape(-1))
    got, want = _step(spss, g, o, st, stepper)
    d = np.abs(got - want)
    assert d[:, :2].max() <= 1e-12
    tol = SIGMA * DT * 2.0 ** -24 + 1e-13
    if stepper == "srk":
        most = 2 * np.abs(st[:, 3]).max()
        tol += SIGMA * DT ** 2 / 2 * 3 * 2.0 ** -24 * most
        assert np.abs(g.complementary_force() - o.complementary_force()).max() <= SIGMA * 3 * 2.0 ** -24 * most + 1e-12
    assert d[:, 2].max() <= (1e-12 if stepper == "euler" else DT * tol + 1e-12)
    assert d[:, 3].max() <= tol


def test_steps_across_the_edges(spss):
    """a ring of particles around the box's edges, moving fast: several rebuilds and steps between them"""
    rng = np.random.default_rng(4)
    xy = (0.06 * (rng.random((3000, 2)) - 0.5)) % 1.0
    xy[1000:2000, 0] = rng.random(1000)
    xy[2000:, 1] = rng.random(1000)
    g, o, st = _systems(spss, xy, 0.03, v0=1.0)
    g.set_state(st.reshape(-1))
    so, n = st.reshape(-1).copy(), len(xy)
    for _ in range(12):
        o.srk_step(METHOD_LINKED_LIST_VERLET, so, DT, np.zeros(2 * n))
    for _ in range(12):
        g.srk_step(spss.METHOD_LINKED_LIST_VERLET, DT, spss.NOISE_NONE)
    d = np.abs(g.get_state() - so).reshape(-1, 4)
    # a wrong neighbour is a hundredth of sigma dt; roundings grow by no more than the steps
    assert d[:, 3].max() <= 12 * 4 * SIGMA * DT * 2.0 ** -24 + 1e-12


def test_omegas_far_apart(spss):
    """one omega of 1e5 among ones: the particles without it in range keep their precision"""
    xy = np.random.default_rng(8).random((600, 2))
    rho = 0.1
    g, o, st = _systems(spss, xy, rho, v0=0.0)
    st[7, 3] = 1e5
    g.set_state(st.reshape(-1))
    _step(spss, g, o, st, "srk")
    dx = np.abs(xy[:, None] - xy[None])
    near = (np.minimum(dx, 1 - dx) ** 2).sum(-1) <= rho ** 2
    om = np.abs(st[:, 3])
    most = np.where(near, om[None], 0).max(1) + om
    d = np.abs(g.complementary_force() - o.complementary_force())
    assert np.all(d <= SIGMA * 3 * 2.0 ** -24 * most + 1e-12)


def test_phase_not_finite(spss):
    xy = np.random.default_rng(9).random((4000, 2))
    g, o, st = _systems(spss, xy, 0.03)
    st[11, 2] = np.nan
    g.set_state(st.reshape(-1))
    got, want = _step(spss, g, o, st, "euler")
    assert np.array_equal(np.isnan(got), np.isnan(want))
    fine = ~np.isnan(want)
    assert np.abs(got - want)[fine].max() <= SIGMA * DT * 2.0 ** -24 + 1e-12
