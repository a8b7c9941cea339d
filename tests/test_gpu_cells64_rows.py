"""FP64 cell lists of particles that are unevenly spread over the rows of cells, whose chunks go round all
workgroups: all in one row, in one cell, in a blob, in some rows.  Against the oracle, and in time
against as many candidates per particle spread over all rows (a factor of 2.5; with a row's chunks left to
its own workgroups 10 and more)."""
import time

import numpy as np
import pytest

import oracle
from oracle.pyoracle import METHOD_LINKED_LIST

pytestmark = pytest.mark.gpu


def _state(model, kind, n, rho):
    rng = np.random.default_rng(n)
    st = rng.random((n, model))
    if kind == "row":
        st[:, 1] = 0.5 + 0.8 * rho * (st[:, 1] - 0.5)
    elif kind == "cell":
        st[:, :2] = 0.5 + 0.8 * rho * (st[:, :2] - 0.5)
    elif kind == "blob":
        st[:, :2] = (0.5 + 0.05 * rng.normal(size=(n, 2))) % 1.0
    elif kind == "rows":  # every fourth row of cells, the last among them
        nc = int(1.0 / rho)
        r = nc - 1 - 4 * rng.integers(0, nc // 4, n)
        st[:, 1] = (r + st[:, 1]) / nc
    st[:, 4 if model == 6 else 2] *= 6.0
    return st.reshape(-1)


@pytest.mark.parametrize("kind,n,rho", [("row", 3001, 0.03), ("cell", 1500, 0.2), ("blob", 6000, 0.02),
                                        ("rows", 5000, 0.02), ("rows", 45000, 0.006), ("row", 300, 0.3)])
@pytest.mark.parametrize("model", [3, 4, 6])
def test_rhs(model, kind, n, rho):
    import spsslangevinintegration_amd as spss
    print(f"[gpu] cells64 rows {kind} model={model} n={n}", flush=True)
    kw = dict(model=model, n=n, rho=rho, sigma=1.5, xi=0.5, v0=0.01, alpha=0.2)
    g, o = spss.ParticleSystem(**kw), oracle.Oracle(**kw)
    st, z = _state(model, kind, n, rho), np.zeros(model * n)
    for _ in range(2):
        ko, kg = np.zeros(model * n), np.zeros(model * n)
        o.evaluate_rhs(METHOD_LINKED_LIST, st, z, ko, 0.0, 0.01)
        g.evaluate_rhs(spss.METHOD_LINKED_LIST, st, z, kg, 0.0, 0.01)
        assert np.abs(kg - ko).max() <= 1e-12
        st = st + 1e-3 * np.random.default_rng(1).random(st.size)
    g.close()


@pytest.mark.parametrize("kind,rho", [("row", 0.03), ("rows", 0.05)])
def test_time(kind, rho):
    import spsslangevinintegration_amd as spss
    n, best = 30000, {}
    nc = int(1.0 / rho)
    # as many candidates: 3 cells of a row of n, or of a quarter of the rows, against 9 cells of all of them
    rows = 1 if kind == "row" else nc // 4
    even = 1.0 / (np.sqrt(3.0 * nc * rows) + 0.5)
    for name, r in ((kind, rho), ("uniform", even)):
        g = spss.ParticleSystem(model=4, n=n, rho=r, sigma=1.5, xi=0.5, v0=0.001)
        g.set_state(_state(4, name, n, r))
        runs = []
        for _ in range(6):
            t0 = time.perf_counter()
            g.run(spss.STEPPER_EULER, spss.METHOD_LINKED_LIST, 3, 1e-4, spss.NOISE_NONE)
            g.synchronize()
            runs.append(time.perf_counter() - t0)
        best[name] = min(runs[1:]) / 3
        g.close()
    print(f"[gpu] cells64 {kind}: {best[kind] * 1e6:.0f} us, uniform {best['uniform'] * 1e6:.0f}", flush=True)
    assert best[kind] <= 2.5 * best["uniform"]
