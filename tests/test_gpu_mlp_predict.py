"""Tables of more rows than a network keeps on the device at a time (64 MB of rows and outputs): the same outputs as
row by row chunks of the table, and no more memory held."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_table_beyond_the_workspace():
    import spsslangevinintegration_amd as spss
    dims, rows = (128, 16, 128), 200003
    print(f"[gpu] predict rows={rows} dims={dims}", flush=True)
    net = spss.MLP(dims, max_batch=64, seed=3)
    x = np.random.default_rng(1).uniform(-1, 1, (rows, dims[0])).astype(np.float32)
    few = net.predict(x[:100])
    hip = C.CDLL("libamdhip64.so.7")  # the runtime that the library is linked against
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    before = free.value
    y = net.predict(x)
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    print(f"  {(before - free.value) / 1e6:.1f} MB held", flush=True)
    assert before - free.value <= 80e6
    assert np.array_equal(y[:100], few)
    for a in (65500, 131000, 199900):
        assert np.array_equal(y[a:a + 103], net.predict(x[a:a + 103]))


@pytest.mark.parametrize("width", [1, 3, 5, 6, 17, 18, 64, 127])
def test_activations_that_overflow(width):
    """a hidden unit of the first layer overflows, all of the second and the output with it: infinite, as the sums
    of the real units are, whatever the widths leave of a tile"""
    import spsslangevinintegration_amd as spss
    dims = (1, width, width, 2)
    print(f"[gpu] predict overflow width={width}", flush=True)
    net = spss.MLP(dims, max_batch=64, seed=3)
    w1 = np.zeros((width, 1))
    w1[0] = 1e38
    w2 = np.full((width, width), 0.5)
    w3 = np.full((2, width), 0.25)
    w3[1] = -0.25
    parts = [w1, np.zeros(width), w2, np.zeros(width), w3, np.zeros(2)]
    net.params = np.concatenate([p.ravel() for p in parts]).astype(np.float32)
    y = net.predict(np.array([[10.0], [0.0], [20.0]], dtype=np.float32))
    assert np.all(np.isposinf(y[[0, 2], 0])) and np.all(np.isneginf(y[[0, 2], 1])) and np.all(y[1] == 0)


@pytest.mark.parametrize("dims", [(6, 128, 128, 128, 2), (128, 128, 128), (5, 17, 3), (1, 1, 1)])
def test_rows_by_16_and_by_64(dims):
    """a row's outputs are the same bits in a table of any length: tables up to 4,096 rows go 16 rows a workgroup,
    longer ones 64"""
    import spsslangevinintegration_amd as spss
    net = spss.MLP(dims, max_batch=64, seed=5)
    x = np.random.default_rng(2).uniform(-1, 1, (4163, dims[0])).astype(np.float32)
    print(f"[gpu] predict rows dims={dims}", flush=True)
    y = net.predict(x)
    for n in (1, 15, 16, 17, 63, 65, 4080, 4095, 4096, 4097):
        assert np.array_equal(net.predict(x[:n]), y[:n]), n
