"""FP64 cell lists of few particles on many cells: the grid's part of an evaluation, 2 million cells here, is spread
over the chip however few the particles are, so that 200 of them take no longer than 10,000 (a factor of two
for the clock), and the evaluation is the oracle's."""
import time

import numpy as np
import pytest

import oracle
from oracle.pyoracle import METHOD_LINKED_LIST

pytestmark = pytest.mark.gpu

RHO = 0.0007


def _system(n):
    import spsslangevinintegration_amd as spss
    kw = dict(model=4, n=n, rho=RHO, sigma=1.5, xi=0.5, v0=0.01, alpha=0.2)
    st = np.random.default_rng(n).random((n, 4))
    st[: n // 2, :2] = 0.5 + 20 * RHO * (st[: n // 2, :2] - 0.5)
    return spss, spss.ParticleSystem(**kw), oracle.Oracle(**kw), st.reshape(-1)


def test_time():
    best = {}
    for n in (10000, 200):
        spss, g, _, st = _system(n)
        print(f"[gpu] cells64 sparse n={n}", flush=True)
        g.set_state(st)
        runs = []
        for _ in range(6):
            t0 = time.perf_counter()
            g.run(spss.STEPPER_EULER, spss.METHOD_LINKED_LIST, 20, 1e-4, spss.NOISE_NONE)
            g.synchronize()
            runs.append(time.perf_counter() - t0)
        best[n] = min(runs[1:]) / 20
        g.close()
    print(f"  {best[10000] * 1e6:.0f} us a step of 10,000, {best[200] * 1e6:.0f} of 200", flush=True)
    assert best[200] <= 2 * best[10000]


@pytest.mark.parametrize("n", [1, 2, 200, 3001])
def test_rhs(n):
    spss, g, o, st = _system(n)
    ko, kg = np.zeros(4 * n), np.zeros(4 * n)
    for _ in range(2):
        o.evaluate_rhs(METHOD_LINKED_LIST, st, np.zeros(4 * n), ko, 0.0, 0.01)
        g.evaluate_rhs(spss.METHOD_LINKED_LIST, st, np.zeros(4 * n), kg, 0.0, 0.01)
        assert np.abs(kg - ko).max() <= 1e-13
        st[0::4] += 0.3
    g.close()
