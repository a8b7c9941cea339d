"""Phases of long runs and far beyond, of particles whose differences are of order one: as exact as the
differences are, also where particle 0, whose phase is the frame of the sums, has a small one.  Reference: numpy
over all pairs with the differences, which are exact.

Bound: a difference is exact, its sine and the mean over the neighbours err by a few 2^-53: 1e-14 sigma."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIGMA, ALPHA, N = 1.5, 0.3, 500


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.mark.parametrize("method,rho", [("METHOD_ALL_PAIRS", 0.6), ("METHOD_VERLET", 0.3),
                                        ("METHOD_LINKED_LIST_VERLET", 0.1), ("METHOD_LINKED_LIST", 0.1)])
@pytest.mark.parametrize("size", [100.0, 2.0 ** 10, -2.0 ** 14, 2.0 ** 20, 2.0 ** 28, 2.0 ** 30, 2.0 ** 33, -2.0 ** 38, 2.0 ** 45, 2.0 ** 50])
@pytest.mark.parametrize("model", [3, 4])
def test_rhs(spss, model, size, method, rho):
    print(f"[gpu] large phases {method} model={model} size={size}", flush=True)
    rng = np.random.default_rng(7)
    st = np.zeros((N, model))
    st[:, :2] = 0.05 + 0.9 * rng.random((N, 2))
    st[:, 2] = size + np.round(rng.uniform(-3, 3, N) / np.spacing(size)) * np.spacing(size)
    st[0] = [0.01, 0.02, 0.7] + [0.0] * (model - 3)
    st[1:, :2] = 0.5 + (st[1:, :2] - 0.5) * (0.5 if rho == 0.6 else 1.0)
    kw = dict(model=model, n=N, v0=0.0, xi=0.0, sigma=SIGMA, rho=rho, alpha=ALPHA, natfreq_local=1)
    g = spss.ParticleSystem(**kw)
    k = np.zeros(N * model)
    g.evaluate_rhs(getattr(spss, method), st.reshape(-1), np.zeros(N * model), k, 0.0, 0.01)
    g.close()
    d = np.abs(st[:, None, :2] - st[None, :, :2])
    near = (np.minimum(d, 1 - d) ** 2).sum(-1) <= rho ** 2
    np.fill_diagonal(near, False)
    own = near[:, 0] | near[0]  # pairs with particle 0: their differences are rounded
    s = np.sin(st[None, :, 2] - st[:, None, 2] - ALPHA)
    n = near.sum(1)
    want = SIGMA * np.where(near, s, 0.0).sum(1) / np.maximum(n, 1)
    fine = ~own
    fine[0] = False
    assert fine.sum() > 100 and n[fine].max() > 10
    err = np.abs(k.reshape(N, model)[:, -1] - want)[fine].max()
    assert err <= 1e-14 * SIGMA, err
