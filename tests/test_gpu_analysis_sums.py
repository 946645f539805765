"""The per-atom integrals against sums in 80-bit arithmetic over the solver's own
g, with a bound from what the kernel adds up.  On these grids a slab is 1024
points, of which a lane takes every 64th: 16 points, so 16 terms of a site's
energy and 16 natv of the other sums; the wave adds 6 levels and the columns are
summed with compensation.  Grid points are exact (0.5 A apart).  In units of
2^-53 r^2 is good to 5, 1/r to 4, r^-6 to 29, (sigma / r)^6 to 41 and its square
with the factors to 90; with g, the levels and the last products 128.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu
L = np.longdouble
AVOGADRO, BOHR, HARTREE = 6.02214076e23, 0.5291771500001, 4.359744722207185e-18


@pytest.mark.parametrize("grid,natu,sites,ad,lam", [
    ((8, 8, 16), 1, 1, 0, 1.0), ((20, 12, 40), 9, 3, 1, 0.8), ((30, 20, 16), 32, 4, 2, 0.7),
    ((24, 36, 32), 33, 2, 0, 1.0), ((16, 30, 32), 40, 8, 1, 0.9),
])
def test_sums(rism, golden, gpu, grid, natu, sites, ad, lam):
    s = rism.read_xvk(f"{golden}/naclaq_vv.xvk")
    idx = [i % 4 for i in range(sites)]
    d = dict(s, natv=sites, vsig=s["vsig"][idx], veps=s["veps"][idx], vq=s["vq"][idx],
             vrho=s["vrho"][idx], xvv=s["xvv"][:, idx][:, :, idx])
    w = random_walk_solute(natu, seed=19, total_charge=0.0)
    xyz = 0.5 * (w["xyz"] - w["xyz"].mean(0))
    xyz[0] = 0.0
    uq = 0.1 * w["q"]
    box = tuple(0.5 * n for n in grid)
    g = rism.RISM3D(grid, box, d, {"usig": w["sig"], "ueps": w["eps"], "uq": uq, "uxyz": xyz},
                    ad_switch=ad, lam=lam)
    g.initialize()
    g.calculate()
    G = g.fields(rism.FIELD_G).astype(L)
    grad, euv, adv = (g.analysis(k) for k in (rism.ANALYSIS_GRAD, rism.ANALYSIS_EUV,
                                              rism.ANALYSIS_AD))
    g.close()
    ax = [(np.arange(n) - n // 2).astype(L) * L(0.5) for n in grid]
    z, y, x = (a.reshape(-1) for a in np.meshgrid(ax[2], ax[1], ax[0], indexing="ij"))
    dv, cc = L(0.125), L(HARTREE * BOHR * AVOGADRO)
    eps64 = L(2.0) ** -53
    one, all_ = (16 + 128) * eps64, (16 * sites + 128) * eps64
    for a in range(natu):
        dr = np.stack([x, y, z]) - xyz[a].astype(L)[:, None]
        r2 = (dr ** 2).sum(0)
        ir = 1 / np.sqrt(np.where(r2 > 0, r2, L(1)))
        i2 = ir * ir
        gr, gs = np.zeros(3, L), np.zeros(3, L)
        av = avs = e0 = e0s = L(0)
        for v in range(sites):
            sg = L(0.5) * (L(w["sig"][a]) + L(d["vsig"][v])) * L(lam if ad == 1 else 1.0)
            e = np.sqrt(L(w["eps"][a]) * L(d["veps"][v]))
            qq = cc * L(uq[a]) * L(d["vq"][v])
            rho = L(d["vrho"][v])
            gv = np.where(r2 >= (sg / 2) ** 2, G[v], L(0))
            s6 = (sg * sg * i2) ** 3
            f = (24 * e * s6 * (2 * s6 - 1) * i2 + qq * i2 * ir) * gv * rho
            fs = (24 * e * s6 * (2 * s6 + 1) * i2 + abs(qq) * i2 * ir) * gv * rho
            gr += (f * dr).sum(1)
            gs += (fs * np.abs(dr)).sum(1)
            ev = dv * rho * ((4 * e * s6 * (s6 - 1) + qq * ir) * gv).sum()
            es = dv * rho * ((4 * e * s6 * (s6 + 1) + abs(qq) * ir) * gv).sum()
            assert abs(euv[a, 1 + v] - ev) <= one * es
            e0, e0s = e0 + ev, e0s + es
            if ad == 1:
                gl = np.where(r2 >= (sg * L(lam) / 2) ** 2, G[v], L(0))
                av += (24 * e * s6 * (2 * s6 - 1) / L(lam) * gl).sum() * rho
                avs += (24 * e * s6 * (2 * s6 + 1) / L(lam) * gl).sum() * rho
            else:
                av += (qq * ir * gv).sum() * rho
                avs += (abs(qq) * ir * gv).sum() * rho
        assert abs(euv[a, 0] - e0) <= all_ * e0s
        assert np.all(np.abs(grad[a] - gr * dv / 4184) <= all_ * gs * dv / 4184)
        assert abs(adv[a] - av * dv / 4184) <= all_ * avs * dv / 4184
