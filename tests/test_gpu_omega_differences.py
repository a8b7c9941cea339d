"""The complementary force of the FP64 neighbour methods, (1 / n) sigma sum (omega_j - omega_i) cos(phi_j - phi_i - alpha):
as exact as the differences of the omegas are, whatever other particles have and whatever all have in common.
Reference: numpy over all pairs with the differences, which are exact.

Bound: sums of some hundred terms in segments err by less than 64 roundings of 2^-53 of the largest |omega_j -
omega_i| in range."""
import numpy as np
import pytest

from spsslangevinintegration_amd import _capi

pytestmark = pytest.mark.gpu

SIGMA, ALPHA, N = 1.5, 0.3, 1500


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.mark.parametrize("method,rho", [("METHOD_ALL_PAIRS", 0.1), ("METHOD_VERLET", 0.1),
                                        ("METHOD_LINKED_LIST_VERLET", 0.1), ("METHOD_LINKED_LIST", 0.1)])
@pytest.mark.parametrize("kind", ["ordinary", "particle 0 far off", "some far off", "one side far off",
                                  "all far off"])
def test_complementary_force(spss, kind, method, rho):
    print(f"[gpu] omega differences {method} {kind}", flush=True)
    rng = np.random.default_rng(11)
    st = np.zeros((N, 4))
    st[:, :2] = rng.random((N, 2))
    st[:, 2] = 6.0 * rng.random(N)
    st[:, 3] = np.round(rng.normal(0, 1, N) * 2.0 ** 20) * 2.0 ** -20
    if kind == "particle 0 far off":
        st[0, 3] = 2.0 ** 27
    elif kind == "some far off":
        st[rng.choice(N, 12, replace=False), 3] = 2.0 ** 28
    elif kind == "one side far off":  # the first particles of the rows of cells
        st[st[:, 0] < 0.1, 3] = 2.0 ** 28
    elif kind == "all far off":
        st[:, 3] += 2.0 ** 28
    g = spss.ParticleSystem(model=4, n=N, v0=0.0, xi=1.0, sigma=SIGMA, rho=rho, alpha=ALPHA, natfreq_local=1)
    _capi.check(g.lib.spss_set_higher_order(g.h, 1))
    k = np.zeros(4 * N)
    g.evaluate_rhs(getattr(spss, method), st.reshape(-1), np.zeros(4 * N), k, 0.0, 0.01)
    got = g.complementary_force()
    g.close()
    d = np.abs(st[:, None, :2] - st[None, :, :2])
    near = (np.minimum(d, 1 - d) ** 2).sum(-1) <= rho ** 2
    np.fill_diagonal(near, False)
    dom = st[None, :, 3] - st[:, None, 3]
    n = near.sum(1)
    want = SIGMA * np.where(near, dom * np.cos(st[None, :, 2] - st[:, None, 2] - ALPHA), 0.0).sum(1) / np.maximum(n, 1)
    most = np.where(near, np.abs(dom), 0.0).max(1)
    tol = SIGMA * 64 * 2.0 ** -53 * most
    err = np.abs(got - want)
    assert np.all(err <= tol), (err.max(), (err[most > 0] / tol[most > 0]).max())
