"""The set-up kernels where a solute is unlike most: every atom of a type of its
own (a pair then costs what the site loop costs, so at most 1.75 times a pair
among few types: 14 operations and two sums against 14 and two sums, eight
products and the start of a run), and the k-space sum at the solute size up to
which a workgroup forms its own phases.
"""
import numpy as np
import pytest

from gen_inputs import cluster_solute
import test_gpu_potentials as potentials

pytestmark = pytest.mark.gpu


def _time(rism, d, su):
    grid = (128, 128, 128)
    g = rism.RISM3D(grid, tuple(0.5 * n for n in grid), d, su)
    g.initialize()
    out = []
    for _ in range(5):
        g.kernel_timing(True)
        g.initialize()
        n, ms = g.kernel_stats()["potential_r"]
        out.append(ms / n)
    g.close()
    return min(out)


def test_many_types(rism, golden, gpu):
    d = rism.read_xvk(f"{golden}/naclaq_vv.xvk")
    w = cluster_solute(500, 10.6, 5, 0.0)
    su = {"usig": w["sig"], "ueps": w["eps"], "uq": w["q"], "uxyz": w["xyz"]}
    few = _time(rism, d, su)
    own = _time(rism, d, dict(su, usig=w["sig"] * (1.0 + 1e-5 * np.arange(500))))
    assert own <= 1.75 * few


@pytest.mark.parametrize("grid,natu,ntype,sites", [
    ((36, 40, 24), 15, 15, 1), ((30, 72, 40), 16, 3, 2), ((72, 20, 24), 17, 17, 4),
])
def test_own_phases(rism, golden, gpu, grid, natu, ntype, sites):
    potentials.test_potentials(rism, golden, gpu, grid, 0.5, natu, ntype, sites, False)


def test_no_atoms(rism, golden, gpu):
    d = rism.read_xvk(f"{golden}/h2o_vv.xvk")
    none = np.zeros(0)
    g = rism.RISM3D((16, 20, 24), (8.0, 10.0, 12.0), d,
                    {"usig": none, "ueps": none, "uq": none, "uxyz": none})
    g.initialize()
    assert not g.fields(rism.FIELD_U).any() and not g.get(rism.FIELD_FR).any()
    assert not g.fk_half().any()
    assert g.calculate() == 0.0  # the bulk solvent: h = 0 everywhere
    g.close()
