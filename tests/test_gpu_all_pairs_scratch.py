"""The workspace of the FP64 all-pairs sums: systems of other methods hold none, and one that needs it for the first
time while its stream is captured gets it there, as evaluations did that needed none."""
import ctypes as C

import numpy as np
import pytest

from spsslangevinintegration_amd import _capi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


@pytest.fixture(scope="module")
def hip():
    # the HIP runtime the library is linked against (already loaded in this process)
    _capi.load()
    return C.CDLL("libamdhip64.so.7")


def _free(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("rho", [0.9, 0.05])
def test_other_methods_hold_no_workspace(spss, hip, rho):
    """n = 4,099: the states, four derivatives, noise and sums of a model-4 system are 1.3 MB in some fifteen
    allocations; the workspace would be 10.7 MB"""
    n, count = 4099, 24
    spss.ParticleSystem(model=4, n=n, rho=rho).close()
    before = _free(hip)
    systems = [spss.ParticleSystem(model=4, n=n, rho=rho) for _ in range(count)]
    used = before - _free(hip)
    for g in systems:
        g.close()
    print(f"[gpu] {used / count / 1e6:.2f} MB a handle", flush=True)
    assert used <= count * 6e6


@pytest.mark.parametrize("mode", [0, 1, 2])  # global, thread-local, relaxed
def test_first_evaluation_in_a_capture(spss, hip, mode):
    n = 1500
    print(f"[gpu] all pairs first evaluated in a capture, mode {mode}", flush=True)
    rng = np.random.default_rng(mode)
    kw = dict(model=4, n=n, rho=0.9, xi=0.5, sigma=2.0, alpha=0.2)
    g, eager = spss.ParticleSystem(**kw), spss.ParticleSystem(**kw)
    x, k = spss.ParticleSystem(**kw), spss.ParticleSystem(**kw)  # their states: the evaluation's in- and output
    px, pk, pz = x.state_device_ptr(), k.state_device_ptr(), eager.state_device_ptr()
    x.synchronize(), k.synchronize(), g.synchronize()
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    _capi.check(g.lib.spss_set_stream(g.h, stream))
    assert hip.hipStreamBeginCapture(stream, mode) == 0
    try:
        g.evaluate_rhs_device(spss.METHOD_ALL_PAIRS, px, pz, pk, 0.0, 0.01)
    finally:
        assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for _ in range(4):
        st = np.concatenate([rng.random((n, 2)), 6.0 * rng.random((n, 1)), rng.normal(0, 1, (n, 1))], 1).reshape(-1)
        x.set_state(st)
        k.set_state(np.zeros(4 * n))
        x.synchronize(), k.synchronize()
        want = np.zeros(4 * n)
        eager.evaluate_rhs(spss.METHOD_ALL_PAIRS, st, np.zeros(4 * n), want, 0.0, 0.01)
        assert hip.hipGraphLaunch(run, stream) == 0 and hip.hipStreamSynchronize(stream) == 0
        assert np.array_equal(k.get_state(), want)
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    for s in (g, eager, x, k):
        s.close()
    assert hip.hipStreamDestroy(stream) == 0
