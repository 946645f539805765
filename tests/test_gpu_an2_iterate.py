"""The AN2 update against its formula on the fields of the same run, step by
step through the Picard and the mixing steps: with the mixed iterate that the
residual pass wrote, and where that does not hold for the t at hand (t set by
the caller, or the state moved to the other precision, between the step and
the update).  t' = Q + s1 (P0 - Q) + s2 (P1 - Q), Q = t + m R: three products
and sums, within 16 ulps of the largest term (FP64 or FP32).
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("how", ["plain", "set_t", "fp32", "switch"])
def test_update(rism, golden, gpu, how):
    d = rism.read_xvk(f"{golden}/h2o_vv.xvk")
    w = random_walk_solute(6, seed=3, total_charge=0.0)
    su = {"usig": w["sig"], "ueps": w["eps"], "uq": w["q"],
          "uxyz": w["xyz"] - w["xyz"].mean(0)}
    grid = (20, 24, 32)
    low = how in ("fp32", "switch")
    g = rism.RISM3D(grid, tuple(0.5 * n for n in grid), d, su, count=2, m=0.6, mp=0.2,
                    precision=1 if low else 0)
    g.initialize()
    eps = 2.0 ** -24 if low else 2.0 ** -53
    rng = np.random.default_rng(4)
    P = [None, None]
    for step in range(7):
        g.calculate()
        _, s, count, b = g.an2_state()
        R = g.fields(rism.FIELD_R)
        if how == "set_t":
            for v in range(g.natv):
                g.set(rism.FIELD_T, v, g.get(rism.FIELD_T, v) + rng.normal(0, 0.1, g.N))
        if how == "switch":
            g.set_precision(1 - g.precision())
        t = g.fields(rism.FIELD_T)
        Q = t + 0.6 * R
        g.anderson()
        got = g.fields(rism.FIELD_T)
        if count > 0:
            want, size = t + R, np.abs(t).max() + np.abs(R).max()
        else:
            want = Q + s[0] * (P[0] - Q) + s[1] * (P[1] - Q)
            size = (1 + abs(s[0]) + abs(s[1])) * max(np.abs(x).max() for x in (Q, P[0], P[1]))
        P[b] = Q
        assert np.abs(got - want).max() <= 16 * eps * size, step
    g.close()
