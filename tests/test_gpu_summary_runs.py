"""The summary's float sums, taken through maps of runs of terms, against the same additions one after
the other (numpy's add.accumulate in float32): particle counts around the runs' and long runs' edges,
and phases whose partial sums wander through the binades, climb through them, stay at zero, cancel, or
stay tiny.  The phases come from few values, so that the device's and the host's phasors are the same
floats; |Z| and arg Z then differ by the last bit of hypot and atan2 on either side at most: 2 ulps."""
import numpy as np
import pytest

from oracle import observer_oracle as OO

pytestmark = pytest.mark.gpu

SETS = {
    "wander": np.linspace(0.1, 6.2, 23),
    "climb": np.array([-0.3, -0.1, 0.05, 0.2, 0.4]),
    "descend": np.pi + np.array([-0.3, 0.1, 0.25]),
    "zero": np.array([0.0]),
    "cancel": np.array([0.5, -0.5, np.pi - 0.5, np.pi + 0.5]),
    "tiny": np.array([1e-9, -2e-9, 3e-12, 0.0, 5e-6]),
    "halves": np.array([np.pi / 3, 2 * np.pi / 3, np.pi / 6, 7 * np.pi / 6]),
}


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.mark.parametrize("n", [1, 63, 65, 256, 257, 4095, 4097, 70001, 1048579])
@pytest.mark.parametrize("kind", sorted(SETS))
def test_summary_of_runs(spss, kind, n):
    print(f"[gpu] summary runs {kind} n={n}", flush=True)
    rng = np.random.default_rng(n)
    st = np.zeros((n, 3))
    st[:, 2] = rng.choice(SETS[kind], n)
    g = spss.ParticleSystem(model=3, n=n, rho=0.8)
    g.set_state(st.reshape(-1))
    for _ in range(2):
        a, arg = g.summary()
    wa, warg = OO.summary(st.reshape(-1), 3)
    g.close()
    assert abs(a - wa) <= 2 * np.spacing(np.float32(wa)), (a, wa)
    assert abs(arg - warg) <= 2 * np.spacing(np.float32(abs(warg))), (arg, warg)
