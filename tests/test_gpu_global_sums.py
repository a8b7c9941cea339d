"""The global field's sums where large terms cancel and small ones are left: blocks of 256 particles at phases 0
and pi, whose cosines cancel exactly, and at +-pi/2, whose cosines of 6e-17 are the whole of Re Z (so the
sines at 0 and pi of Im Z).  A block's terms are equal or cancel in pairs; only sums that carry their rounding
errors from block to block keep the small ones.  Reference: the exact sums (math.fsum).  From rest
the phase velocities after a step are dt sigma |Z| sin(arg Z - phi) times 1 + O(dt)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIGMA, DT = 1.3, 1e-4


@pytest.mark.parametrize("stepper,n", [("euler", 768), ("euler", 1024), ("srk", 768), ("rk4", 768), ("rk4", 1280),
                                       ("rk4", 2048), ("euler", 1280), ("srk", 1280), ("rk4", 2304)])
def test_small_terms_beside_cancelling_ones(stepper, n):
    import spsslangevinintegration_amd as spss
    print(f"[gpu] global sums {stepper} n={n}", flush=True)
    blocks = n // 256
    phi = np.empty(n)
    for b in range(blocks):
        kind = b % 4  # 0, small, pi, small, ...; a last 0 without its pi is small too
        if kind in (0, 2) and not (kind == 0 and b + 2 >= blocks):
            phi[256 * b:256 * b + 256] = 0.0 if kind == 0 else np.pi
        else:
            phi[256 * b:256 * b + 256] = np.where(np.arange(256) % 2, 0.5, -0.5) * np.pi
    zx, zy = math.fsum(np.cos(phi)) / n, math.fsum(np.sin(phi)) / n
    assert 1e-18 < abs(zx) < 1e-15
    st = np.zeros((n, 4))
    st[:, 2] = phi
    g = spss.ParticleSystem(model=4, n=n, xi=0.1, sigma=SIGMA, rho=0.8, alpha=0.0, v0=0.0)
    g.set_state(st.reshape(-1))
    code = dict(euler=spss.STEPPER_EULER, srk=spss.STEPPER_SRK, rk4=spss.STEPPER_RK4)[stepper]
    g.run(code, spss.METHOD_GLOBAL_FIELD, 1, DT, spss.NOISE_NONE)
    om = g.get_state().reshape(-1, 4)[:, 3]
    g.close()
    want = DT * SIGMA * (zy * np.cos(phi) - zx * np.sin(phi))
    assert np.abs(om - want).max() <= 1e-3 * np.abs(want).max(), (om[:2], want[:2], om[256:258], want[256:258])
