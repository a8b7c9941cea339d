"""The FP64 all-pairs derivative of up to 64 particles, one launch of one wave, against the oracle: pairs at the radius,
a box other than one, positions outside the box and far outside (the exact test).

Bounds: 1e-12 relative to max(1, |k|), as for every FP64 right-hand side."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.mark.parametrize("n", [1, 2, 3, 5, 31, 63, 64, 65])
@pytest.mark.parametrize("model,ho", [(3, 0), (4, 0), (4, 1), (6, 0)])
@pytest.mark.parametrize("where", ["inside", "around", "far"])
def test_few(spss, model, ho, where, n):
    print(f"[gpu] all pairs few model={model} ho={ho} {where} n={n}", flush=True)
    rng = np.random.default_rng(n)
    st = rng.random((n, model))
    st[:, 4 if model == 6 else 2] = 11.0 + 2 * np.pi * rng.random(n)
    if n > 1:
        st[1, :2] = st[0, :2] + [0.25, 0.0]
    if where == "around":
        st[:, :2] = 3 * st[:, :2] - 1
    elif where == "far" and model != 6:
        st[n // 2, 0] += 1e5
    kw = dict(model=model, n=n, v0=0.3, xi=0.2, sigma=1.3, rho=0.25, alpha=0.4, xi_r=0.9, x_size=0.8)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    if ho:
        o.set_higher_order(1)
        g.set_higher_order(1)
    kp = 0.3 * np.sin(np.arange(model * n) * 0.37)
    ko, kg = np.full(model * n, 7.0), np.full(model * n, 7.0)
    o.evaluate_rhs(2, st.reshape(-1), kp, ko, 0.5, 0.01)
    g.evaluate_rhs(spss.METHOD_ALL_PAIRS, st.reshape(-1), kp, kg, 0.5, 0.01)
    assert np.max(np.abs(kg - ko) / np.maximum(np.abs(ko), 1.0)) <= 1e-12
    if ho:
        co, cg = o.complementary_force(), g.complementary_force()
        assert np.max(np.abs(co - cg) / np.maximum(np.abs(co), 1.0)) <= 1e-12
    g.close()


@pytest.mark.parametrize("n", [7, 64])
def test_few_steps(spss, n):
    print(f"[gpu] all pairs few steps n={n}", flush=True)
    kw = dict(model=4, n=n, v0=0.3, xi=0.2, sigma=1.3, rho=0.6, alpha=0.4)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw)
    st = np.random.default_rng(n).random(4 * n)
    g.set_state(st)
    g.run(spss.STEPPER_RK4, spss.METHOD_ALL_PAIRS, 3, 0.01)
    for _ in range(3):
        o.rk4_step(2, st, 0.01)
    assert np.max(np.abs(g.get_state() - st) / np.maximum(np.abs(st), 1.0)) <= 1e-12
    g.close()
