"""The end of a step of a group whose partial sums are too many for one workgroup
per context (more than 49152) and are reduced first: 2304 rows of 6 sums for each
of 4 sites.  As separate solves, bit for bit.
"""
import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu


def test_reduced_in_group(rism, golden, gpu):
    grid, steps = (256, 144, 16), 11
    d = rism.read_xvk(f"{golden}/naclaq_vv.xvk")
    out = []
    for batch in (False, True):
        gs = []
        for seed in (21, 22):
            s = random_walk_solute(6, seed=seed, total_charge=0.0)
            gs.append(rism.RISM3D(grid, tuple(0.5 * n for n in grid), d, {
                "usig": s["sig"], "ueps": s["eps"], "uq": 0.5 * s["q"],
                "uxyz": s["xyz"] - s["xyz"].mean(0)}).initialize())
        if batch:
            rms = [r for _, _, r in rism.solve_batch(gs, maxstep=steps, tol=1e-30)]
        else:
            rms = [g.iterate(maxstep=steps, tol=1e-30)[2] for g in gs]
        out.append((rms, [g.fields(rism.FIELD_T) for g in gs]))
        for g in gs:
            g.close()
    assert out[0][0] == out[1][0] and all(np.isfinite(out[0][0]))
    for a, b in zip(out[0][1], out[1][1]):
        assert np.array_equal(a, b)
