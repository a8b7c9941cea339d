"""The FP64 Verlet lists and pair sums at the edges of their split over lanes: fewer particles than
a wave's groups, lists shorter and much longer than a group, empty lists, particle counts on both
sides of the change of lanes per particle; phases far from the origin and without a sine.
Reference: the oracle's restatement of EvaluateInteractionsWith[LinkedListAnd]VerletNeighborList
(ParticleSystemFirstOrderPtr.cpp:470-815): lists equal in content and order, the right-hand side
within 1e-12 relative to max(1, |k|)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.mark.parametrize("model,n,rho,method,dense,phase", [
    (4, 1, 0.1, 5, 0, 0.0), (3, 3, 0.2, 4, 0, 0.0), (4, 65, 0.3, 4, 0, 1e4), (4, 777, 0.02, 5, 0, 0.0),
    (3, 2500, 0.06, 5, 1200, 0.0), (4, 3001, 0.01, 4, 0, 2e9), (4, 16383, 0.04, 5, 0, 0.0), (4, 16400, 0.04, 5, 0, 0.0),
    (3, 20011, 0.12, 5, 0, 300.0)])
def test_verlet_edges(spss, model, n, rho, method, dense, phase):
    import oracle
    print(f"[gpu] verlet edges model={model} n={n} rho={rho} method={method}", flush=True)
    rng = np.random.default_rng(n + method)
    st = rng.random((n, model)) * 1.4 - 0.2
    st[:dense, :2] = 0.4 + 0.01 * rng.random((dense, 2))
    st[:, 2] = phase + 7.0 * rng.random(n)
    kw = dict(model=model, n=n, v0=0.3, xi=0.7, sigma=1.3, rho=rho, alpha=0.4)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    if model == 4:
        o.set_higher_order(1)
        g.set_higher_order(1)
    z = np.zeros(model * n)
    ko, kg = np.full(model * n, 7.0), np.full(model * n, 7.0)
    o.evaluate_rhs(method, st.reshape(-1), z, ko, 0.0, 0.01)
    g.evaluate_rhs(method, st.reshape(-1), z, kg, 0.0, 0.01)
    oi, oj = o.verlet_lists()  # (i, j) of every entry, in list order
    lists = g.verlet_lists()
    assert np.array_equal(np.repeat(np.arange(n), [len(a) for a in lists]), oi)
    assert np.array_equal(np.concatenate(lists), oj)
    assert np.max(np.abs(kg - ko) / np.maximum(np.abs(ko), 1.0)) <= 1e-12
    if model == 4:
        co, cg = o.complementary_force(), g.complementary_force()
        assert np.max(np.abs(co - cg) / np.maximum(np.abs(co), 1.0)) <= 1e-12


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_verlet_bad_phase(spss, bad):
    import oracle
    print(f"[gpu] verlet with a phase of {bad}", flush=True)
    rng = np.random.default_rng(2)
    st = rng.random((900, 4))
    st[11, 2] = bad
    kw = dict(model=4, n=900, v0=0.3, xi=0.7, sigma=1.3, rho=0.05, alpha=0.4)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    z = np.zeros(3600)
    ko, kg = np.full(3600, 7.0), np.full(3600, 7.0)
    o.evaluate_rhs(5, st.reshape(-1), z, ko, 0.0, 0.01)
    g.evaluate_rhs(5, st.reshape(-1), z, kg, 0.0, 0.01)
    assert np.array_equal(np.isnan(ko), np.isnan(kg)) and np.isnan(ko).any()
    assert np.nanmax(np.abs(kg - ko) / np.maximum(np.abs(ko), 1.0)) <= 1e-12


@pytest.mark.parametrize("model,n,rho,method,order", [
    (4, 1, 0.1, 5, 0), (3, 65, 0.3, 4, 0), (4, 255, 0.05, 5, 1), (4, 2500, 0.06, 4, 1), (3, 16383, 0.03, 5, 0),
    (4, 16385, 0.03, 5, 0)])
def test_verlet_rk4_steps(spss, model, n, rho, method, order):
    """Runge-Kutta steps, whose launches go on to the next stage: four steps, lists rebuilt on the way.
    Each derivative is within 1e-12 of the oracle's, so that a step of 0.02 adds less than 1e-13 and the
    state after four stays within 1e-12; the displacement's sum is one of values near 0.02."""
    import oracle
    print(f"[gpu] verlet rk4 model={model} n={n} rho={rho} method={method}", flush=True)
    rng = np.random.default_rng(3 * n + method)
    st = rng.random((n, model)) - 0.5
    st[:, 2] *= 6.0
    kw = dict(model=model, n=n, v0=1.0, xi=0.7, sigma=1.3, rho=rho, alpha=0.4)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    if model == 4:
        o.set_higher_order(order)
        g.set_higher_order(order)
    so = st.reshape(-1).copy()
    g.set_state(so)
    rebuilt = 0
    for _ in range(4):
        o.rk4_step(method, so, 0.02)
        g.rk4_step(method, 0.02)
        flag, acc, uses = g.verlet_status()
        assert uses and flag == o.should_update_lists and abs(acc - o.accumulated_displacement) <= 1e-13
        rebuilt += flag
        assert np.max(np.abs(g.get_state().reshape(-1) - so) / np.maximum(np.abs(so), 1.0)) <= 1e-12
    assert rebuilt
