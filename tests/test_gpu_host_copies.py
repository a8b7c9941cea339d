"""States and frames copied to the host in threaded pieces: byte counts at and around the smallest staged
copy, ragged pieces, more than one turn of the pinned buffer, pinned destinations, several handles from
several threads.  The copies are exact: compared bit for bit with what was set."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _system(spss, n, model=4):
    g = spss.ParticleSystem(model=model, n=n, rho=0.9)
    st = np.random.default_rng(n).random(n * model)
    g.set_state(st)
    return g, st


@pytest.mark.parametrize("n", [131071, 131072, 131073, 200003, 524287, 524288, 524289, 1048576, 1048577, 2300001])
def test_state(spss, n):
    g, st = _system(spss, n)
    assert np.array_equal(g.get_state(), st)
    out = np.zeros(4 * n)
    assert np.array_equal(g.get_state(out), st)  # into memory that has its pages
    p = C.c_void_p()
    assert g.lib.hipHostMalloc(C.byref(p), C.c_size_t(32 * n), C.c_uint(0)) == 0  # of the library's runtime
    try:
        pinned = np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_double)), (4 * n,))
        assert np.array_equal(g.get_state(pinned), st)
    finally:
        assert g.lib.hipHostFree(p) == 0


@pytest.mark.parametrize("n", [349525, 349526, 1048575])
def test_frame(spss, n):
    g, st = _system(spss, n, model=6)
    frame = g.frame(1.5)  # model 6: the raw float copy behind a float time
    assert frame[0] == np.float32(1.5)
    assert np.array_equal(frame[1:], st.astype(np.float32))


def test_threads(spss):
    pairs = [_system(spss, n) for n in (400000, 500001, 600002)]
    bad = []

    def work(g, st):
        for _ in range(5):
            if not np.array_equal(g.get_state(), st):
                bad.append(g)

    team = [threading.Thread(target=work, args=p) for p in pairs]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad
