"""The summary of phases whose float sums the maps of runs once got wrong, against numpy's sequential float32
additions.  |Z| and arg Z differ by the last bit of hypot and atan2 on either side at most: 2 ulps."""
import numpy as np
import pytest

from oracle import observer_oracle as OO

pytestmark = pytest.mark.gpu

NEAR_TIES = np.concatenate([np.full(140000, np.arccos(0.95)), np.tile([np.arccos(0.95), 1.5786089058042636], 2000)])


TINY = np.tile([5e-18, -1e-18, 1e-30], 4000)  # the sines' sum starts at zero and stays below 2^-45


@pytest.mark.parametrize("phases", [NEAR_TIES, np.full(1000, 1e-18), TINY], ids=["near ties", "1e-18", "tiny"])
def test_summary(phases):
    import spsslangevinintegration_amd as spss
    n = phases.size
    print(f"[gpu] summary sums n={n}", flush=True)
    st = np.zeros((n, 3))
    st[:, 2] = phases
    g = spss.ParticleSystem(model=3, n=n, rho=0.8)
    g.set_state(st.reshape(-1))
    a, arg = g.summary()
    g.close()
    wa, warg = OO.summary(st.reshape(-1), 3)
    assert abs(a - wa) <= 2 * np.spacing(np.float32(wa)), (a, wa)
    assert abs(arg - warg) <= 2 * np.spacing(np.float32(abs(warg))), (arg, warg)


@pytest.mark.parametrize("n", [2, 255, 8191, 16383, 16384, 16385, 20479, 20480, 20481, 69633])
def test_summary_counts(n):
    """sums of one launch (up to 16,384 particles) and of maps of runs (beyond), around their steps"""
    import spsslangevinintegration_amd as spss
    print(f"[gpu] summary counts n={n}", flush=True)
    st = np.zeros((n, 6))
    st[:, 4] = np.random.default_rng(n).choice(np.linspace(-1.2, 4.5, 17), n)
    g = spss.ParticleSystem(model=6, n=n, rho=0.8)
    g.set_state(st.reshape(-1))
    a, arg = g.summary()
    g.close()
    wa, warg = OO.summary(st.reshape(-1), 6)
    assert abs(a - wa) <= 2 * np.spacing(np.float32(wa)), (a, wa)
    assert abs(arg - warg) <= 2 * np.spacing(np.float32(abs(warg))), (arg, warg)
