"""The FP64 global field at the edges of its splits: one workgroup's register tiles (1, 256, 512, 1024,
2048 particles), the block sums beyond them, several passes of a workgroup; all steppers, models 3
and 4, the complementary force, phases beyond the range of the short reduction, a field of zero.
Reference: the oracle's restatement of ParticleSystemFirstOrderPtr.cpp:177-223 and of the steppers; for
phases of 2^31, where that expression's arg(Z) - phi_i itself rounds at 2^-22, the same formulas in
extended precision on the same double-precision stage states.

Bounds: a right-hand side's terms are at most a few units with rounding errors of a few 2^-53 and a
compensated or 11-level sum, 1e-12 relative to max(1, |k|) as for every FP64 right-hand side; three
steps add three times as much, 1e-11.  A run of several steps and the same steps one by one differ by the
order of the field's sums at most: 1e-12."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def spss():
    import spsslangevinintegration_amd as m
    return m


def _systems(spss, model, n, ho=0):
    import oracle
    kw = dict(model=model, n=n, v0=0.7, xi=0.3, sigma=1.3, rho=0.9, alpha=0.4, D_phi=0.2)
    o, g = oracle.Oracle(**kw), spss.ParticleSystem(**kw, seed=77)
    w = np.random.default_rng(n).normal(0, 1, n)
    o.set_natural_frequencies(w)
    g.set_natural_frequencies(w)
    if ho:
        o.set_higher_order(1)
        g.set_higher_order(1)
    return o, g


def _state(model, n, far=False):
    rng = np.random.default_rng(1000 * model + n)
    st = rng.random((n, model))
    st[:, 2] = 4.0 + 2 * np.pi * rng.random(n)
    if far:
        st[::3, 2] += 2.0 ** 31
    if model == 4:
        st[:, 3] = rng.normal(0, 1, n)
    return st.reshape(-1)


def _close(a, b, tol):
    assert np.all(np.isfinite(b))
    assert np.max(np.abs(a - b) / np.maximum(np.abs(b), 1.0)) <= tol


def _exact_rhs(st, model, w):
    x = st.reshape(-1, model)
    phi = x[:, 2].astype(np.longdouble)
    c, s = np.cos(phi), np.sin(phi)
    zx, zy = c.mean(), s.mean()
    A, B = zy * c - zx * s, zx * c + zy * s
    al = np.longdouble(0.4)
    force = w + np.longdouble(1.3) * (A * np.cos(al) - B * np.sin(al))
    v0 = np.longdouble(0.7)
    k = [v0 * c, v0 * s] + ([force] if model == 3 else [x[:, 3], -np.longdouble(0.3) * x[:, 3] + force])
    out = np.stack([np.asarray(q, dtype=np.float64) for q in k], axis=1).reshape(-1)
    W = x[:, -1].astype(np.longdouble)
    wx, wy = (W * c).mean(), (W * s).mean()
    sin_w = (wy * c - wx * s) / np.hypot(wx, wy)  # sin(arg W - phi)
    compl = np.longdouble(1.3) * ((wx * c + wy * s) * np.cos(al) + (wy * c - wx * s) * np.sin(al) -
                                  W * (B * np.cos(al) + np.hypot(zx, zy) * sin_w * np.sin(al)))
    return out, np.asarray(compl, dtype=np.float64)


def _exact_rk4(st, model, w, dt):
    k1 = _exact_rhs(st, model, w)[0]
    k2 = _exact_rhs(st + 0.5 * dt * k1, model, w)[0]
    k3 = _exact_rhs(st + 0.5 * dt * k2, model, w)[0]
    k4 = _exact_rhs(st + dt * k3, model, w)[0]
    return st + (k1 + 2.0 * k2 + 2.0 * k3 + k4) * dt / 6.0


SIZES = [1, 2, 255, 256, 257, 512, 513, 1024, 1025, 2048, 2049, 4097, 262145]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("model", [3, 4])
def test_rhs_and_steps(spss, model, n):
    for ho in ([0, 1] if model == 4 else [0]):
        o, g = _systems(spss, model, n, ho)
        far = n % 2 == 1
        st = _state(model, n, far)
        w = np.random.default_rng(n).normal(0, 1, n)
        kp = np.random.default_rng(5).normal(0, 1, model * n)
        ko, kg = np.zeros(model * n), np.zeros(model * n)
        o.evaluate_rhs(0, st, kp, ko, 0.5, 0.01)
        g.evaluate_rhs(spss.METHOD_GLOBAL_FIELD, st, kp, kg, 0.5, 0.01)
        co = o.complementary_force() if ho else None
        if far:
            ko, co = _exact_rhs(st + kp * (0.5 * 0.01), model, w)
        _close(kg, ko, 1e-12)
        if ho:
            _close(g.complementary_force(), co, 1e-12)
        so = st.copy()
        g.set_state(st)
        for _ in range(3):
            if far:
                so = _exact_rk4(so, model, w, 0.01)
            else:
                o.rk4_step(0, so, 0.01)
        g.run(spss.STEPPER_RK4, spss.METHOD_GLOBAL_FIELD, 3, 0.01, spss.NOISE_NONE)
        _close(g.get_state(), so, 1e-11)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("stepper", ["euler", "srk"])
def test_stochastic_steps(spss, stepper, n):
    for model in ([3, 4] if stepper == "euler" else [4]):
        o, g = _systems(spss, model, n)
        st = _state(model, n)
        so, rng = st.copy(), np.random.default_rng(9)
        g.set_state(st)
        for _ in range(3):
            z = rng.normal(0, 1, n if stepper == "euler" else 2 * n)
            getattr(o, stepper + "_step")(0, so, 0.01, z)
            getattr(g, stepper + "_step")(spss.METHOD_GLOBAL_FIELD, 0.01, spss.NOISE_HOST, z)
        _close(g.get_state(), so, 1e-11)
        if stepper == "srk":
            _close(g.complementary_force(), o.complementary_force(), 1e-11)
        # Philox noise: several steps in one call and one by one
        code = spss.STEPPER_EULER if stepper == "euler" else spss.STEPPER_SRK
        a, b = [spss.ParticleSystem(model=model, n=n, sigma=1.3, rho=0.9, alpha=0.4, D_phi=0.2, seed=5)
                for _ in range(2)]
        a.set_state(st)
        b.set_state(st)
        a.run(code, spss.METHOD_GLOBAL_FIELD, 4, 0.01, spss.NOISE_PHILOX)
        for _ in range(4):
            getattr(b, stepper + "_step")(spss.METHOD_GLOBAL_FIELD, 0.01, spss.NOISE_PHILOX)
        _close(a.get_state(), b.get_state(), 1e-12)


def test_field_of_zero_and_nonfinite(spss):
    """opposite phases cancel to a field near zero; a phase that is not finite spoils every force, as in
    the reference, and one left in k1 does so at the next step (state + 0 * k1)"""
    for n in (4, 4096):
        o, g = _systems(spss, 4, n, 1)
        st = np.zeros((n, 4))
        st[:, 2] = np.where(np.arange(n) % 2, np.pi, 0.0)
        ko, kg = np.zeros(4 * n), np.zeros(4 * n)
        o.evaluate_rhs(0, st.reshape(-1), np.zeros(4 * n), ko, 0.0, 0.01)
        g.evaluate_rhs(spss.METHOD_GLOBAL_FIELD, st.reshape(-1), np.zeros(4 * n), kg, 0.0, 0.01)
        _close(kg, ko, 1e-12)
        bad = st.copy()
        bad[n // 2, 2] = np.inf
        g.set_state(bad.reshape(-1))
        g.rk4_step(spss.METHOD_GLOBAL_FIELD, 0.01)
        assert np.all(np.isnan(g.get_state()[3::4]))
        g.set_state(st.reshape(-1))
        g.rk4_step(spss.METHOD_GLOBAL_FIELD, 0.01)
        assert np.all(np.isnan(g.get_state()[3::4]))


@pytest.mark.parametrize("model,n,mode", [(3, 1, 0), (4, 255, 1), (3, 257, 1), (4, 1025, 0), (3, 131073, 0),
                                          (4, 131072, 0), (4, 131073, 1)])
def test_dormand_prince(spss, model, n, mode):
    """the trials on planes of phases and positions: the same steps as the oracle's integration, the states
    within 1e-10 (right-hand sides that agree to 1e-12 over the same steps), with and without an observer;
    then lists, whose trials work on whole rows, in the same buffers"""
    from oracle import dopri5_oracle as D
    o, g = _systems(spss, model, n)
    st, zeros = _state(model, n), np.zeros(model * n)

    def rhs(x):
        out = np.zeros(model * n)
        o.evaluate_rhs(0, np.ascontiguousarray(x), zeros, out, 0.0, 0.0)
        return out

    integ = D.integrate_const if mode == 0 else D.integrate_adaptive
    want, want_seen, ost = integ(rhs, st, 0.0, 0.3, 0.05, 1e-7, 1e-7)
    seen = []
    for observer in (lambda t, x: seen.append((t, x)), None):
        g.set_state(st)
        steps, rejected = g.integrate_dopri5(0.0, 0.3, 0.05, 1e-7, 1e-7, method=spss.METHOD_GLOBAL_FIELD, mode=mode,
                                             observer=observer)
        assert (steps, rejected) == (ost.steps, ost.rejected)
        _close(g.get_state(), want, 1e-10)
    assert len(seen) == len(want_seen)
    for (_, x), (_, xw) in zip(seen, want_seen):
        _close(x, xw, 1e-10)
    if 1 < n < 2000:
        h = _systems(spss, model, n)[1]
        for s in (g, h):
            s.set_state(st)
            s.integrate_dopri5(0.0, 0.1, 0.05, 1e-7, 1e-7, method=spss.METHOD_ALL_PAIRS, mode=mode)
        assert np.array_equal(g.get_state(), h.get_state())
