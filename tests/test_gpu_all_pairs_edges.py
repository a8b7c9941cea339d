"""The FP64 all-pairs sums at the edges of their tiling (groups of particles, segments and tiles of
the j's) and on inputs that leave the cheap distance test: pairs exactly at the radius, positions
outside and far outside the box, phases without a finite phasor.  Reference: the oracle's restatement
of EvaluateInteractionsWithAllPairs (ParticleSystemFirstOrderPtr.cpp:225-316).

Bounds: 1e-12 relative to max(1, |k|) as for every FP64 right-hand side; near synchrony (phases
within 1e-7 of each other) 1e-12 relative to the largest force, since the sums run in the frame of
one particle's phase and every rounding scales with the spread."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _both(spss, st, model, rho, ho, x_size=1.0, config=None):
    import oracle
    n = st.shape[0]
    kw = dict(model=model, n=n, v0=0.3, xi=0.0, sigma=1.3, rho=rho, alpha=0.4, xi_r=0.9, x_size=x_size)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    if ho:
        o.set_higher_order(1)
        g.set_higher_order(1)
    if config is not None:
        g.set_all_pairs_config(config)
    kp = 0.3 * np.sin(np.arange(model * n) * 0.37)
    kp[np.arange(n) * model + 2] = 0.0  # phases and what follows them as given
    ko, kg = np.full(model * n, 7.0), np.full(model * n, 7.0)
    o.evaluate_rhs(2, st.reshape(-1), kp, ko, 0.0, 0.01)
    g.evaluate_rhs(spss.METHOD_ALL_PAIRS, st.reshape(-1), kp, kg, 0.0, 0.01)
    co, cg = (o.complementary_force(), g.complementary_force()) if ho else (None, None)
    g.close()
    return ko, kg, co, cg


def _state(n, model, seed, spread=1.0, width=2.0 * np.pi):
    rng = np.random.default_rng(seed)
    st = rng.random((n, model))
    st[:, :2] = spread * st[:, :2] - 0.5 * (spread - 1.0)
    st[:, 4 if model == 6 else 2] = 11.0 + width * rng.random(n)
    if model != 3:
        st[:, model - 1] = rng.normal(0, 1, n)
    return st


@pytest.mark.parametrize("model,n,ho,spread,x_size,config", [
    (4, 1, 1, 1.0, 1.0, None), (4, 2, 0, 1.0, 1.0, None), (3, 63, 0, 3.0, 1.0, 0), (6, 64, 0, 1.0, 1.0, 2),
    (6, 65, 0, 2.0, 1.0, None), (4, 129, 1, 5.0, 1.0, 1), (3, 257, 0, 1.0, 1.0, None), (4, 1025, 0, 1.0, 0.7, 3),
    (4, 4099, 1, 1.0, 1.0, None), (6, 3000, 0, 1.0, 1.0, 5)])
def test_all_pairs_edges(spss, model, n, ho, spread, x_size, config):
    print(f"[gpu] all-pairs edges model={model} n={n} spread={spread} x_size={x_size}", flush=True)
    st = _state(n, model, n + model, spread)
    if n > 100:
        st[5, :2] = st[4, :2] + [0.125, 0.0]  # with rho = 0.125 exactly at the radius, up to rounding
        st[7, 0] = -1e-17                     # wraps to the box's far edge
        if model != 6:
            st[9, 0] += 1e5                   # far outside the box: the exact test
    ko, kg, co, cg = _both(spss, st, model, 0.125 if n > 100 else 0.6, ho, x_size, config)
    assert np.max(np.abs(kg - ko) / np.maximum(np.abs(ko), 1.0)) <= 1e-12
    if ho:
        assert np.max(np.abs(co - cg) / np.maximum(np.abs(co), 1.0)) <= 1e-12


@pytest.mark.parametrize("model", [3, 4, 6])
def test_all_pairs_near_synchrony(spss, model):
    print(f"[gpu] all-pairs near synchrony model={model}", flush=True)
    st = _state(900, model, 3, width=1e-7)
    import oracle
    kw = dict(model=model, n=900, v0=0.0, xi=0.0, sigma=1.0, rho=0.4, alpha=0.0)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    ko, kg, z = np.zeros(model * 900), np.zeros(model * 900), np.zeros(model * 900)
    o.evaluate_rhs(2, st.reshape(-1), z, ko, 0.0, 0.01)
    g.evaluate_rhs(spss.METHOD_ALL_PAIRS, st.reshape(-1), z, kg, 0.0, 0.01)
    fo, fg = ko[model - 1::model], kg[model - 1::model]
    assert 0.0 < np.max(np.abs(fo)) < 1e-6
    assert np.max(np.abs(fg - fo)) <= 1e-12 * np.max(np.abs(fo))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_all_pairs_bad_phase_stays_with_its_neighbours(spss, bad):
    print(f"[gpu] all-pairs with a phase of {bad}", flush=True)
    for where in (0, 300):  # also the particle whose phase is the frame's reference
        st = _state(700, 4, 8)
        st[where, 2] = bad
        ko, kg, co, cg = _both(spss, st, 4, 0.05, 1)
        assert np.array_equal(np.isnan(ko), np.isnan(kg)) and np.array_equal(np.isnan(co), np.isnan(cg))
        fine = ~np.isnan(ko)
        assert 0 < np.count_nonzero(~fine) < 200
        assert np.max(np.abs(kg - ko)[fine] / np.maximum(np.abs(ko[fine]), 1.0)) <= 1e-12
