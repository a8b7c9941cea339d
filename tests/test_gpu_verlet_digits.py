"""What the FP32C Verlet steps keep of small phasors and omegas: states synchronised near a phase at which sines or cosines
are small, with and without a particle far off the rest in the same tile; an omega that diverges; and densities at which the stage,
not the workgroup, bounds a tile.  Reference: the oracle's FP64 steps.

Bounds: a phasor's component is rounded once to FP32 (2^-25 of itself), its sum over the neighbours is taken
as closely.  With alpha = 0 the mean over the neighbours of sin(phi_j - phi_i) is c_i <s> - s_i <c>, so it errs
by 2^-25 of (|c_i| max |s_j| + |s_i| max |c_j|), and by as much again for all later roundings.  A component's
maximum is taken over the particles in range alone: nothing that is out of range may matter."""
import numpy as np
import pytest

import oracle
from oracle.pyoracle import METHOD_LINKED_LIST_VERLET, VERLET_EXACT
from tests import test_gpu_verlet_tiles as tiles

pytestmark = pytest.mark.gpu

SIGMA, DT = 1.5, 0.002


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _most(xy, rho, v):
    """max |v_j| over the particles in range of each (itself among them)"""
    out = np.empty(len(xy))
    for a in range(0, len(xy), 500):
        dx = np.abs(xy[a:a + 500, None] - xy[None])
        near = (np.minimum(dx, 1 - dx) ** 2).sum(-1) <= (rho * (1 + 1e-9)) ** 2
        out[a:a + 500] = np.where(near, np.abs(v)[None], 0.0).max(1)
    return out


def _systems(spss, n, rho):
    kw = dict(model=4, n=n, v0=0.0, xi=2.0, sigma=SIGMA, rho=rho, alpha=0.0, verlet_mode=VERLET_EXACT,
              verlet_skin=0.2 * rho)
    return spss.ParticleSystem(precision=spss.PRECISION_FP32C, **kw), oracle.Oracle(**kw)


@pytest.mark.parametrize("stray", [0, 1])
@pytest.mark.parametrize("spread", [1e-2, 1e-4, 1e-6, 1e-9, 1e-14])
@pytest.mark.parametrize("phase", [0.0, np.pi / 2])
def test_synchronised_phases(spss, phase, spread, stray):
    n, rho = 3000, 0.06
    print(f"[gpu] verlet digits phase={phase} spread={spread} stray={stray}", flush=True)
    rng = np.random.default_rng(3)
    xy, phi = rng.random((n, 2)), phase + spread * rng.normal(0.0, 1.0, n)
    if stray:
        phi[5] = phase + 1.0
    st = np.concatenate([xy, phi[:, None], np.zeros((n, 1))], 1).reshape(-1)
    g, o = _systems(spss, n, rho)
    g.set_state(st)
    want = st.copy()
    o.euler_step(METHOD_LINKED_LIST_VERLET, want, DT, np.zeros(n))
    g.euler_step(spss.METHOD_LINKED_LIST_VERLET, DT, spss.NOISE_NONE)
    d = np.abs(g.get_state() - want).reshape(-1, 4)[:, 3]
    g.close()
    s, c = np.sin(phi), np.cos(phi)
    tol = SIGMA * DT * 2.0 ** -24 * (np.abs(c) * _most(xy, rho, s) + np.abs(s) * _most(xy, rho, c))
    # the oracle's own roundings: of the phases' differences, and of the sums
    tol += SIGMA * DT * 2.0 ** -50 * (phase + _most(xy, rho, phi - phase))
    assert np.all(d <= tol), (d.max(), np.max(d / tol))


@pytest.mark.parametrize("size", [1e5, 1e8, 1e12, 1e16, 1e25, 1e35])
def test_an_omega_that_diverges(spss, size):
    """the complementary force's terms err by three roundings of 2^-24 of (|omega_j| + |omega_i|) at most, of those
    in range alone"""
    n, rho = 3000, 0.06
    print(f"[gpu] verlet digits omega={size}", flush=True)
    xy = np.random.default_rng(8).random((n, 2))
    g, o, st = tiles._systems(spss, xy, rho, v0=0.0)
    st[7, 3] = size
    g.set_state(st.reshape(-1))
    tiles._step(spss, g, o, st, "srk")
    om = np.abs(st[:, 3])
    d = np.abs(g.complementary_force() - o.complementary_force())
    tol = SIGMA * 3 * 2.0 ** -24 * (_most(xy, rho, om) + om) + 1e-12
    assert np.all(d <= tol), (d.max(), np.max(d / tol))


@pytest.mark.parametrize("stepper", ["euler", "srk"])
@pytest.mark.parametrize("cell", [51, 85, 112, 113])
def test_tiles_that_the_stage_bounds(spss, cell, stepper):
    """cells of that many particles each: the widest tile that fits the stage has 4, 1 and 1 columns, where 256
    particles would allow 5, 3 and 2; at 113 a single column's stage does not fit"""
    print(f"[gpu] verlet tiles cell={cell} {stepper}", flush=True)
    tiles.test_first_step(spss, f"stage{cell}", stepper)
