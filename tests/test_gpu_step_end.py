"""The end of a step on the device: the sums of the residual pass read in one
workgroup or, past its limit, reduced first; the AN2 system; the Anderson(m)
least squares from one pair to the most the solver keeps, with the history
filling up and, later, retiring pairs.  Against the oracle's iteration on the
same potentials, 1e-9 of the largest value as in the other trajectory tests.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu


def _case(oracle, golden, xvk, natu):
    s = oracle.read_xvk(f"{golden}/{xvk}")
    d = {"natv": s.natv, "ntab": s.ntab, "dr": s.dr, "temper": s.temper, "xt": s.xt,
         "vsig": s.sig, "veps": s.eps, "vq": s.q, "vrho": s.rho, "xvv": s.xvv}
    w = random_walk_solute(natu, seed=12, total_charge=0.0)
    sol = oracle.Solute(w["sig"], w["eps"], 0.5 * w["q"], w["xyz"])
    sol.xyz, sol.shift = oracle.centering(sol.xyz)
    return s, d, sol, {"usig": sol.sig, "ueps": sol.eps, "uq": sol.q, "uxyz": sol.xyz}


@pytest.mark.parametrize("grid,xvk,am,steps", [
    ((24, 16, 32), "h2o_vv.xvk", 1, 8),
    ((24, 16, 32), "h2o_vv.xvk", 3, 14),
    ((24, 20, 32), "naclaq_vv.xvk", 10, 16),
    ((20, 16, 24), "h2o_vv.xvk", 16, 22),
    ((160, 80, 16), "naclaq_vv.xvk", 4, 9),    # 800 rows of 17 sums per site
    ((8, 8, 16), "h2o_vv.xvk", 0, 8),
    ((256, 144, 16), "naclaq_vv.xvk", 0, 7),   # 2304 rows of 6 sums per site
])
def test_trajectory(rism, oracle, golden, gpu, grid, xvk, am, steps):
    s, d, sol, su = _case(oracle, golden, xvk, 8)
    box = tuple(0.5 * n for n in grid)
    o = oracle.OracleRISM(grid, box, s, sol, "KH", 2, 0.6, 0.2, 1e-30, steps).setup()
    ro = o.solve(maxstep=steps) if am == 0 else o.solve_anderson_m(am, maxstep=steps)
    g = rism.RISM3D(grid, box, d, su, rism.KH, 2, 0.6, 0.2, anderson_m=am)
    g.initialize()
    st, n, rms = g.iterate(maxstep=steps, tol=1e-30)
    t = g.fields(rism.FIELD_T).reshape(-1)
    g.close()
    assert n == ro.steps == steps
    assert abs(rms - ro.rms[-1]) <= 1e-9 * ro.rms[-1]
    assert np.abs(t - ro.t.reshape(-1)).max() <= 1e-9 * np.abs(ro.t).max()
