"""Boxes with different sides take chi_vv from the octant table; the x pass
evaluating the spline at every k (chi_spline) is what the other tests hold to
the oracle.  One step of each must agree to rounding: the table holds the
same spline values, so the bound is a few hundred ulps of the largest value
(FP64) and of FP32 rounding for the mixed solve's bulk.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu


def _solvent(oracle, golden, sites):
    s = oracle.read_xvk(f"{golden}/naclaq_vv.xvk")
    xvv = np.asarray(s.xvv).reshape(s.ntab, 4, 4)
    idx = [i % 4 for i in range(sites)]
    return {"natv": sites, "ntab": s.ntab, "dr": s.dr, "temper": s.temper, "xt": s.xt,
            "vsig": s.sig[idx], "veps": s.eps[idx], "vq": s.q[idx], "vrho": s.rho[idx],
            "xvv": xvv[:, idx][:, :, idx]}


# row lengths with one and several (kx, -kx) pairs per thread, row slots with
# spare rows, few rows (taken one by one) and many (taken in mirror pairs)
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("grid,sites", [
    ((8, 12, 16), 1), ((8, 12, 16), 2), ((12, 8, 32), 3), ((20, 30, 16), 4), ((36, 8, 24), 6),
    ((72, 90, 60), 2), ((160, 20, 32), 4), ((90, 96, 128), 2), ((48, 128, 144), 4),
    ((64, 72, 96), 3), ((30, 16, 24), 8),
])
def test_octant_matches_spline(rism, oracle, golden, gpu, grid, sites, prec):
    d = _solvent(oracle, golden, sites)
    box = tuple(0.5 * n for n in grid)
    s = random_walk_solute(6, seed=33, total_charge=1.0)
    su = {"usig": s["sig"], "ueps": s["eps"], "uq": s["q"],
          "uxyz": 0.2 * (s["xyz"] - s["xyz"].mean(0))}
    out = []
    for spline in (False, True):
        g = rism.RISM3D(grid, box, d, su, chi_spline=spline, precision=prec)
        g.initialize()
        rms = g.calculate()
        out.append((rms, g.fields(rism.FIELD_R)))
        g.close()
    (ra, a), (rb, b) = out
    tol = 3e-5 if prec else 1e-13
    assert np.isfinite(rb) and abs(ra - rb) <= tol * rb
    assert np.abs(a - b).max() <= tol * np.abs(b).max()
