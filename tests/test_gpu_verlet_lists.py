"""The export of FP32C Verlet lists around the first rebuild: a run that is prepared has entered its state but
built nothing yet, so its lists are empty, also where an earlier state's lists were built on the same
handle; after a step they are the oracle's.  On grids with row tiles and on wider ones.  Lists that outgrow the
width are reported, and asking for them leaves the run as it is."""
import numpy as np
import pytest

import oracle
from oracle.pyoracle import METHOD_LINKED_LIST_VERLET, VERLET_EXACT

pytestmark = pytest.mark.gpu

# a tiled grid of 27 cells a side, and one of 1,041 (wider than the tiles serve)
GRIDS = [(3000, 0.03), (5000, 0.0008)]


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _lists(g):
    return [sorted(l.tolist()) for l in g.verlet_lists()]


@pytest.mark.parametrize("n,rho", GRIDS)
def test_lists_before_the_first_rebuild(spss, n, rho):
    print(f"[gpu] verlet lists around the first rebuild n={n} rho={rho}", flush=True)
    kw = dict(model=4, n=n, v0=0.01, xi=2.0, sigma=1.0, rho=rho, verlet_mode=VERLET_EXACT, verlet_skin=0.2 * rho)
    g = spss.ParticleSystem(precision=spss.PRECISION_FP32C, **kw)
    for seed in (1, 2):
        st = np.random.default_rng(seed).random((n, 4))
        st[: n // 2, :2] = 0.4 + 4 * rho * st[: n // 2, :2]  # somewhere dense: lists on the fine grid too
        st = st.reshape(-1)
        g.set_state(st)
        g.prepare_run(spss.STEPPER_EULER, spss.METHOD_LINKED_LIST_VERLET, 0.002, spss.NOISE_PHILOX)
        assert all(len(l) == 0 for l in g.verlet_lists())
        assert np.array_equal(g.get_state(), st)
        g.prepare_run(spss.STEPPER_EULER, spss.METHOD_LINKED_LIST_VERLET, 0.002, spss.NOISE_PHILOX)
        g.run(spss.STEPPER_EULER, spss.METHOD_LINKED_LIST_VERLET, 1, 0.002, spss.NOISE_PHILOX)
        o = oracle.Oracle(**kw)
        o.euler_step(METHOD_LINKED_LIST_VERLET, st.copy(), 0.002, np.zeros(n))
        oi, oj = o.verlet_lists()
        want = [[] for _ in range(n)]
        for i, j in zip(oi.tolist(), oj.tolist()):
            want[i].append(j)
        got = _lists(g)
        assert sum(map(len, got)) > 0
        assert got == [sorted(w) for w in want]
    g.close()


def test_lists_past_the_width_are_reported(spss):
    """three adjacent cells of 400 particles each in a uniform background: their particles' lists outgrow the
    width that the mean density of the densest 3 x 3 cells asks for"""
    rho = 0.02
    h = 1.0 / int(1.0 / (1.2 * rho))
    rng = np.random.default_rng(77)
    xy = [rng.random((12000, 2))]
    for cx, cy in ((20, 20), (21, 20), (20, 21)):
        xy.append((np.array([cx, cy]) + 0.02 + 0.96 * rng.random((400, 2))) * h)
    xy = np.concatenate(xy)
    n = len(xy)
    st = np.concatenate([xy, rng.random((n, 2))], 1).reshape(-1)
    out = []
    for ask in (False, True):
        g = spss.ParticleSystem(precision=spss.PRECISION_FP32C, model=4, n=n, v0=0.05, xi=2.0, sigma=3.0, rho=rho,
                                verlet_mode=VERLET_EXACT, verlet_skin=0.2 * rho)
        g.set_state(st)
        for _ in range(4):
            g.run(spss.STEPPER_SRK, spss.METHOD_LINKED_LIST_VERLET, 3, 0.002, spss.NOISE_PHILOX)
            if ask:
                with pytest.raises(spss.SpssError, match="outgrew"):
                    g.verlet_lists()
        out.append((g.verlet_status(), g.get_state()))
        g.close()
    assert out[0][0] == out[1][0]
    assert np.array_equal(out[0][1], out[1][1])
