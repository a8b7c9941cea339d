"""FP32C Verlet steps of dense systems, whose cells do not fit the LDS stage of a tile: uniform and clustered
particles, open tiles beside staged ones, items of less than a wave.  Against the oracle's first step with the
bounds of tests/test_gpu_verlet_tiles.py (partials of two terms round no more than the phasors do), and in
time against the cell list's step of the same system, which visits about as many candidates (a factor of
five; walking lists there took 4 to 60 times as long)."""
import time

import numpy as np
import pytest

from tests import test_gpu_verlet_tiles as tiles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _positions(kind, n):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return rng.random((n, 2))
    if kind == "blob":
        return (0.5 + 0.05 * rng.normal(size=(n, 2))) % 1.0
    if kind == "corner":  # across the box's edges
        return (0.05 * rng.normal(size=(n, 2))) % 1.0
    if kind == "cell":
        return 0.5 + 0.01 * rng.random((n, 2))
    raise KeyError(kind)


@pytest.mark.parametrize("stepper", ["euler", "srk"])
@pytest.mark.parametrize("kind,n,rho", [("uniform", 3000, 0.2), ("blob", 5000, 0.03), ("corner", 4001, 0.04),
                                        ("cell", 257, 0.03), ("cell", 1985, 0.03)])
def test_first_step(spss, kind, n, rho, stepper):
    print(f"[gpu] verlet dense {kind} n={n} rho={rho} {stepper}", flush=True)
    xy = _positions(kind, n)
    g, o, st = tiles._systems(spss, xy, rho)
    g.set_state(st.reshape(-1))
    got, want = tiles._step(spss, g, o, st, stepper)
    d = np.abs(got - want)
    most = 2 * np.abs(st[:, 3]).max()
    tol = tiles.SIGMA * tiles.DT * 2.0 ** -24 + 1e-13
    if stepper == "srk":
        tol += tiles.SIGMA * tiles.DT ** 2 / 2 * 3 * 2.0 ** -24 * most
        assert np.abs(g.complementary_force() - o.complementary_force()).max() <= tiles.SIGMA * 3 * 2.0 ** -24 * most + 1e-12
    assert d[:, :2].max() <= 1e-12 and d[:, 3].max() <= tol
    g.close()


@pytest.mark.parametrize("stepper", ["euler", "srk"])
@pytest.mark.parametrize("kind,n,rho", [("uniform", 30000, 0.1), ("blob", 10000, 0.03), ("cell", 3000, 0.03)])
def test_time(spss, kind, n, rho, stepper):
    best = {}
    for method in (spss.METHOD_LINKED_LIST, spss.METHOD_LINKED_LIST_VERLET):
        g, _, st = tiles._systems(spss, _positions(kind, n), rho, v0=0.001)
        g.set_state(st.reshape(-1))
        runs = []
        for _ in range(5):
            t0 = time.perf_counter()
            g.run(spss.STEPPER_EULER if stepper == "euler" else spss.STEPPER_SRK, method, 20, 0.001, spss.NOISE_PHILOX)
            g.synchronize()
            runs.append(time.perf_counter() - t0)
        best[method] = min(runs[1:]) / 20
        g.close()
    a, b = best[spss.METHOD_LINKED_LIST], best[spss.METHOD_LINKED_LIST_VERLET]
    print(f"[gpu] verlet dense {kind} n={n} {stepper}: cells {a * 1e6:.0f} us, lists {b * 1e6:.0f}", flush=True)
    assert b <= 5 * a
