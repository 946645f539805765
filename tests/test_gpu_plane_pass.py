"""Small planes take the y, x and inverse y passes in one kernel.  One step of
it is compared with one step of the three passes, which the spline x pass of
the same context options runs (chi_spline); both transform the same values, so they agree to
rounding: a few hundred ulps of the largest value.  Every pair of lengths and site count that the kernel is
built for, the smallest nz, and the nearest grid that does not fit.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu

LENGTHS = (40, 48, 60, 64, 72, 80, 96)


def _fits(nx, ny, sites):
    return 16 * (sites * ny * (nx + 1) + 2 * (nx + ny)) <= 160 * 1024


CASES = [(nx, ny, nz, sites) for sites, nz in ((2, 16), (4, 24))
         for nx in LENGTHS for ny in LENGTHS if _fits(nx, ny, sites)]


def _solvent(oracle, golden, sites):
    s = oracle.read_xvk(f"{golden}/naclaq_vv.xvk")
    xvv = np.asarray(s.xvv).reshape(s.ntab, 4, 4)
    idx = [i % 4 for i in range(sites)]
    return {"natv": sites, "ntab": s.ntab, "dr": s.dr, "temper": s.temper, "xt": s.xt,
            "vsig": s.sig[idx], "veps": s.eps[idx], "vq": s.q[idx], "vrho": s.rho[idx],
            "xvv": xvv[:, idx][:, :, idx]}


@pytest.mark.parametrize("nx,ny,nz,sites", CASES + [(64, 80, 16, 2), (64, 64, 64, 2),
                                                    (48, 48, 48, 2), (48, 48, 48, 4)])
def test_plane_matches_passes(rism, oracle, golden, gpu, nx, ny, nz, sites):
    d = _solvent(oracle, golden, sites)
    grid = (nx, ny, nz)
    # equal lengths along x and y: a cubic box, so that chi comes from shells
    box = (0.5 * nx,) * 3 if nx == ny else tuple(0.5 * n for n in grid)
    s = random_walk_solute(6, seed=41, total_charge=1.0)
    su = {"usig": s["sig"], "ueps": s["eps"], "uq": s["q"],
          "uxyz": 0.2 * (s["xyz"] - s["xyz"].mean(0))}
    out = []
    for spline in (False, True):
        g = rism.RISM3D(grid, box, d, su, chi_spline=spline)
        g.initialize()
        rms = g.calculate()
        out.append((rms, g.fields(rism.FIELD_R)))
        g.close()
    (ra, a), (rb, b) = out
    assert np.isfinite(rb) and abs(ra - rb) <= 1e-13 * rb
    assert np.abs(a - b).max() <= 1e-13 * np.abs(b).max()
