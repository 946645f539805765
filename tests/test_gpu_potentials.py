"""The r-space potentials and the k-space Coulomb term against sums in 80-bit
arithmetic, at the edges of their kernels: grids that are not whole tiles of
16 x 4 x 4 points (r space) or 32 ky x 32 kx (k space), solutes around the 64
atoms taken at once and the 4 of a matrix product, one and many atom types,
boxes so coarse that most pairs are beyond the smoothing's reach, atoms on and
next to grid points, and no Coulomb part.

Bounds, in units of 2^-53 of the sum of |terms|: a term's r^2 is good to 3
units, 1/r to 3 more, r^-12 to 12 times that and a few for its products (64
together), and n terms add n units.  fk: each k_d x_d is rounded twice, so a
phase is off by 2 sum |k_d x_d| units, plus 16 for the products and n.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu
L = np.longdouble
EPS = 2.0 ** -53
AVOGADRO, BOHR, BOLTZMANN, HARTREE = (6.02214076e23, 0.5291771500001, 1.380649e-23,
                                      4.359744722207185e-18)


@pytest.mark.parametrize("grid,spacing,natu,ntype,sites,lj_only", [
    ((8, 8, 16), 0.5, 1, 1, 1, False),
    ((20, 12, 24), 0.5, 5, 5, 2, False),
    ((30, 36, 40), 0.5, 63, 4, 4, False),
    ((36, 30, 32), 0.5, 64, 1, 3, False),
    ((40, 20, 24), 4.0, 65, 7, 4, False),      # mostly far pairs
    ((16, 72, 32), 3.0, 130, 130, 2, False),   # every atom a type of its own
    ((24, 20, 32), 2.0, 129, 3, 6, False),
    ((20, 36, 16), 0.5, 66, 2, 8, False),
    ((72, 40, 16), 0.5, 7, 3, 4, True),
])
def test_potentials(rism, golden, gpu, grid, spacing, natu, ntype, sites, lj_only):
    s = rism.read_xvk(f"{golden}/naclaq_vv.xvk")
    idx = [i % 4 for i in range(sites)]
    d = dict(s, natv=sites, vsig=s["vsig"][idx], veps=s["veps"][idx], vq=s["vq"][idx],
             vrho=s["vrho"][idx], xvv=s["xvv"][:, idx][:, :, idx])
    w = random_walk_solute(natu, seed=7, total_charge=1.0)
    rng = np.random.default_rng(5)
    kind = rng.integers(0, ntype, natu) if natu > ntype else np.arange(natu)
    sig, eps = 2.5 + 0.01 * kind, 300.0 + 7.0 * kind
    xyz = w["xyz"] - w["xyz"].mean(0)
    xyz[0] = 0.0                                        # on a grid point
    if natu > 2:
        xyz[1] = (spacing, 0.0, 0.004)                  # within the guards
        xyz[2] = (0.0, spacing + 5e-6, 0.0)
    box = tuple(spacing * n for n in grid)
    g = rism.RISM3D(grid, box, d, {"usig": sig, "ueps": eps, "uq": w["q"], "uxyz": xyz},
                    ad_switch=1 if lj_only else 0, lam=0.9)
    g.initialize()
    ax = [(np.arange(n) - n // 2).astype(L) * (L(b) / n) for n, b in zip(grid, box)]
    z, y, x = np.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
    ikbt = 1.0 / (AVOGADRO * BOLTZMANN * d["temper"])
    ub = HARTREE * BOHR / (BOLTZMANN * d["temper"])
    shape = x.shape
    de, ade, fr = (np.zeros(shape, L) for _ in range(3))
    lj, alj = np.zeros((sites,) + shape, L), np.zeros((sites,) + shape, L)
    for a in range(natu):
        p = xyz[a].astype(L)
        r2 = (x - p[0]) ** 2 + (y - p[1]) ** 2 + (z - p[2]) ** 2
        r = np.sqrt(r2)
        near = r < 1e-5
        rs = np.where(near, L(1), r)
        q = L(0 if lj_only else w["q"][a])
        de += np.where(near, 0, q / rs)
        ade += np.where(near, abs(q), abs(q) / rs)
        fr += np.where(near, q, -q * np.expm1(-rs) / rs)
        for v in range(sites):
            sg = L((sig[a] + d["vsig"][v]) * 0.5 * (0.9 if lj_only else 1.0))
            e4 = L(4.0 * np.sqrt(eps[a] * d["veps"][v]))
            s6 = np.maximum(r2 / sg ** 2, L(4e-6)) ** -3
            lj[v] += e4 * s6 * (s6 - 1)
            alj[v] += e4 * s6 * (s6 + 1)
    units = (64 + natu) * EPS
    for v in range(sites):
        qv = L(d["vq"][v])
        ref = lj[v] * ikbt + qv * de * ub
        bound = units * (alj[v] * ikbt + abs(qv) * ade * ub)
        err = abs(g.get(rism.FIELD_U, v).reshape(shape) - ref)
        assert np.all(err <= bound), (v, float((err / np.maximum(bound, 1e-300)).max()))
    err = abs(g.get(rism.FIELD_FR).reshape(shape) - fr * ub)
    assert np.all(err <= units * ade * ub)
    fk = g.fk_half()
    g.close()
    if lj_only:
        assert not fk.any()
        return
    M = grid[2] // 2
    k = [2 * L(np.pi) * (np.arange(n) - n // 2 + L(0.5)) / L(b) for n, b in zip(grid, box)]
    kz, ky, kx = np.meshgrid(k[2][M:], k[1], k[0], indexing="ij")
    S, off = np.zeros(kx.shape, np.clongdouble), np.zeros(kx.shape, L)
    for a in range(natu):
        p, q = xyz[a].astype(L), L(w["q"][a])
        ph = kx * p[0] + ky * p[1] + kz * p[2]
        S += q * (np.cos(ph) - 1j * np.sin(ph))
        off += abs(q) * (2 * (abs(kx * p[0]) + abs(ky * p[1]) + abs(kz * p[2])) + 16 + natu)
    k2 = kx ** 2 + ky ** 2 + kz ** 2
    f = 4 * L(np.pi) * ub / (k2 * (k2 + 1))
    assert np.all(np.abs(fk - f * S) <= EPS * f * off)
