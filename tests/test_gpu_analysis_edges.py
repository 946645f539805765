"""The per-atom integrals against numpy sums over the solver's own g, at the
edges of the kernel: solutes around the 8 atoms of a wave and the 32 of a
workgroup, 1 to 8 sites, grids that are no whole number of 256-point tiles,
atoms on grid points.  A lane adds up to some 1100 terms before the wave and
the compensated column sums, and a term is good to 64 units: 1300 units of
2^-53 of the sum of |terms|.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu
AVOGADRO, BOHR, HARTREE = 6.02214076e23, 0.5291771500001, 4.359744722207185e-18


@pytest.mark.parametrize("grid,natu,sites,ad,lam", [
    ((8, 8, 16), 1, 1, 0, 1.0), ((12, 20, 24), 8, 2, 0, 1.0), ((20, 12, 40), 9, 3, 1, 0.8),
    ((30, 20, 16), 32, 4, 2, 0.7), ((24, 36, 16), 33, 6, 0, 1.0), ((16, 30, 32), 70, 8, 1, 0.9),
])
def test_analysis(rism, golden, gpu, grid, natu, sites, ad, lam):
    s = rism.read_xvk(f"{golden}/naclaq_vv.xvk")
    idx = [i % 4 for i in range(sites)]
    d = dict(s, natv=sites, vsig=s["vsig"][idx], veps=s["veps"][idx], vq=s["vq"][idx],
             vrho=s["vrho"][idx], xvv=s["xvv"][:, idx][:, :, idx])
    w = random_walk_solute(natu, seed=9, total_charge=0.0)
    xyz = 0.5 * (w["xyz"] - w["xyz"].mean(0))
    xyz[0] = 0.0
    box = tuple(0.5 * n for n in grid)
    g = rism.RISM3D(grid, box, d, {"usig": w["sig"], "ueps": w["eps"], "uq": 0.1 * w["q"],
                                   "uxyz": xyz}, ad_switch=ad, lam=lam)
    g.initialize()
    g.calculate()
    G = g.fields(rism.FIELD_G)
    grad, euv, adv = (g.analysis(k) for k in (rism.ANALYSIS_GRAD, rism.ANALYSIS_EUV,
                                              rism.ANALYSIS_AD))
    g.close()
    ax = [(np.arange(n) - n // 2) * (b / n) for n, b in zip(grid, box)]
    z, y, x = (a.reshape(-1) for a in np.meshgrid(ax[2], ax[1], ax[0], indexing="ij"))
    dv, cc, tol = 0.125, HARTREE * BOHR * AVOGADRO, 1300 * 2.0 ** -53
    for a in range(natu):
        dr = np.stack([x, y, z]) - xyz[a][:, None]
        r2 = (dr ** 2).sum(0)
        i2 = 1.0 / np.where(r2 > 0, r2, 1.0)
        gr, gs = np.zeros(3), np.zeros(3)
        av, avs, e0, e0s = 0.0, 0.0, 0.0, 0.0
        for v in range(sites):
            sg = 0.5 * (w["sig"][a] + d["vsig"][v]) * (lam if ad == 1 else 1.0)
            eps = np.sqrt(w["eps"][a] * d["veps"][v])
            qq = cc * 0.1 * w["q"][a] * d["vq"][v]
            gv = np.where(r2 >= (0.5 * sg) ** 2, G[v], 0.0)
            s6 = (sg * sg * i2) ** 3
            f = (24 * eps * s6 * (2 * s6 - 1) * i2 + qq * i2 * np.sqrt(i2)) * gv * d["vrho"][v]
            fs = (24 * eps * s6 * (2 * s6 + 1) * i2 + abs(qq) * i2 * np.sqrt(i2)) * gv * d["vrho"][v]
            gr += (f * dr).sum(1)
            gs += (fs * np.abs(dr)).sum(1)
            e = dv * d["vrho"][v] * ((4 * eps * s6 * (s6 - 1) + qq * np.sqrt(i2)) * gv).sum()
            es = dv * d["vrho"][v] * ((4 * eps * s6 * (s6 + 1) + abs(qq) * np.sqrt(i2)) * gv).sum()
            assert abs(euv[a, 1 + v] - e) <= tol * es
            e0, e0s = e0 + e, e0s + es
            if ad == 1:
                gl = np.where(r2 >= (0.5 * sg * lam) ** 2, G[v], 0.0)
                av += (24 * eps * s6 * (2 * s6 - 1) / lam * gl).sum() * d["vrho"][v]
                avs += (24 * eps * s6 * (2 * s6 + 1) / lam * gl).sum() * d["vrho"][v]
            else:
                av += (qq * np.sqrt(i2) * gv).sum() * d["vrho"][v]
                avs += (abs(qq) * np.sqrt(i2) * gv).sum() * d["vrho"][v]
        assert abs(euv[a, 0] - e0) <= tol * e0s
        assert np.all(np.abs(grad[a] - gr * dv / 4184.0) <= tol * gs * dv / 4184.0)
        assert abs(adv[a] - av * dv / 4184.0) <= tol * avs * dv / 4184.0
