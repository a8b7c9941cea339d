"""The FP64 linked-list sums at the edges of their tiling: fewer particles than a workgroup, rows of
cells shorter and longer than one, cells denser than the LDS stage, spans wider than its columns, the
smallest grid; and inputs that leave the cheap distance test: pairs exactly at the radius, positions
outside and far outside the box, phases without a finite phasor.  Reference: the oracle's
restatement of EvaluateInteractionsWithLinkedList (ParticleSystemFirstOrderPtr.cpp:318-468).

Bounds: 1e-12 relative to max(1, |k|) as for every FP64 right-hand side; near synchrony (phases
within 1e-7 of each other) 1e-12 relative to the largest force.  A second evaluation runs in the
order the first one left and has to give the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _state(n, model, seed, spread=1.0, width=2.0 * np.pi):
    rng = np.random.default_rng(seed)
    st = rng.random((n, model))
    st[:, :2] = spread * st[:, :2] - 0.5 * (spread - 1.0)
    st[:, 4 if model == 6 else 2] = 11.0 + width * rng.random(n)
    if model != 3:
        st[:, model - 1] = rng.normal(0, 1, n)
    return st


def _compare(spss, st, model, rho, ho=0, alpha=0.4, rel_force=False):
    import oracle
    n = st.shape[0]
    kw = dict(model=model, n=n, v0=0.0 if rel_force else 0.3, xi=0.0, sigma=1.3, rho=rho, alpha=alpha, xi_r=0.9)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    if ho:
        o.set_higher_order(1)
        g.set_higher_order(1)
    z = np.zeros(model * n)
    ko, kg, k2 = np.full(model * n, 7.0), np.full(model * n, 7.0), np.full(model * n, 7.0)
    o.evaluate_rhs(3, st.reshape(-1), z, ko, 0.0, 0.01)
    g.evaluate_rhs(spss.METHOD_LINKED_LIST, st.reshape(-1), z, kg, 0.0, 0.01)
    g.evaluate_rhs(spss.METHOD_LINKED_LIST, st.reshape(-1), z, k2, 0.0, 0.01)
    assert np.array_equal(kg, k2, equal_nan=True)
    assert np.array_equal(np.isnan(ko), np.isnan(kg))
    fine = ~np.isnan(ko)
    if rel_force:
        fo, fg = ko[model - 1::model], kg[model - 1::model]
        assert 0.0 < np.max(np.abs(fo)) < 1e-6
        assert np.max(np.abs(fg - fo)) <= 1e-12 * np.max(np.abs(fo))
        return
    assert np.max(np.abs(kg - ko)[fine] / np.maximum(np.abs(ko[fine]), 1.0)) <= 1e-12
    if ho:
        co, cg = o.complementary_force(), g.complementary_force()
        fine = ~np.isnan(co)
        assert np.array_equal(fine, ~np.isnan(cg))
        assert np.max(np.abs(co - cg)[fine] / np.maximum(np.abs(co[fine]), 1.0)) <= 1e-12
    g.close()


@pytest.mark.parametrize("model,n,rho,ho,spread", [
    (4, 1, 0.1, 1, 1.0), (3, 2, 0.3, 0, 1.0), (6, 63, 0.3, 0, 2.0), (4, 65, 0.26, 1, 3.0), (4, 500, 0.005, 0, 1.0),
    (6, 500, 0.004, 0, 1.0), (4, 3000, 0.012, 1, 7.0), (3, 4097, 0.05, 0, 1.0), (6, 4097, 0.11, 0, 1.0),
    (4, 6000, 0.3333, 0, 1.0), (3, 131072, 0.01, 0, 1.0), (4, 140001, 0.02, 1, 1.0), (6, 131073, 0.006, 0, 1.0)])
def test_cells_edges(spss, model, n, rho, ho, spread):
    print(f"[gpu] cells edges model={model} n={n} rho={rho}", flush=True)
    st = _state(n, model, n + model, spread)
    if n > 100:
        st[5, :2] = st[4, :2] + [rho, 0.0]
        st[7, 0] = -1e-17  # wraps to the box's far edge
    _compare(spss, st, model, rho, ho)


@pytest.mark.parametrize("model,n,dense,rho", [(4, 5000, 3000, 0.1), (6, 2500, 1400, 0.03), (3, 140000, 3000, 0.02)])
def test_cells_dense_cluster(spss, model, n, dense, rho):
    print(f"[gpu] cells cluster model={model} n={n} dense={dense}", flush=True)
    st = _state(n, model, 5)
    st[:dense, :2] = 0.5 + 0.02 * (st[:dense, :2] - 0.5)
    _compare(spss, st, model, rho, int(model == 4))


@pytest.mark.parametrize("model", [3, 4, 6])
def test_cells_lattice_at_the_radius(spss, model):
    """a lattice of spacing rho / 2 = 1/16: every distance test of a neighbour shell is a tie"""
    print(f"[gpu] cells lattice model={model}", flush=True)
    st = _state(256, model, 9)
    st[:, 0], st[:, 1] = np.arange(256) % 16 / 16.0, np.arange(256) // 16 / 16.0
    _compare(spss, st, model, 0.125)


@pytest.mark.parametrize("model", [3, 4, 6])
def test_cells_near_synchrony(spss, model):
    print(f"[gpu] cells near synchrony model={model}", flush=True)
    _compare(spss, _state(3000, model, 3, width=1e-7), model, 0.06, alpha=0.0, rel_force=True)


@pytest.mark.parametrize("what,value", [("phase", np.nan), ("phase", np.inf), ("x", 1e5), ("y", -3e6)])
def test_cells_inputs_past_the_cheap_test(spss, what, value):
    print(f"[gpu] cells with {what} = {value}", flush=True)
    for model in (3, 4, 6):
        st = _state(900, model, 8)
        st[17, {"phase": 4 if model == 6 else 2, "x": 0, "y": 1}[what]] = value
        _compare(spss, st, model, 0.07, int(model == 4))
