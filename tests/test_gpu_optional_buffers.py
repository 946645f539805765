"""The buffers that a context can do without: the octant chi table of a box with
different sides and the third AN2 iterate.  Contexts without them (withheld by
RISM_OPTIONAL_BUFFERS=0) hold that much less memory and walk the same trajectory;
an allocation that finds no room takes them from idle contexts, wherever these
stand in the loop, and leaves those at work alone.

The table and the spline, and the iterate written by either kernel, agree to
rounding (some 1e-15 of the largest value a step), which the steps amplify: 1e-9
after up to 14, as in the other trajectory tests (FP32 1e-3).
"""
import os
import threading

import numpy as np
import pytest

from gen_inputs import random_walk_solute

pytestmark = pytest.mark.gpu
GRID = (96, 80, 64)


def _inputs(rism, golden, seed=3):
    s = random_walk_solute(6, seed=seed, total_charge=0.0)
    return rism.read_xvk(f"{golden}/naclaq_vv.xvk"), {
        "usig": s["sig"], "ueps": s["eps"], "uq": 0.5 * s["q"],
        "uxyz": s["xyz"] - s["xyz"].mean(0)}


def _make(rism, golden, withheld=False, grid=GRID, seed=3, **kw):
    d, su = _inputs(rism, golden, seed)
    if withheld:
        os.environ["RISM_OPTIONAL_BUFFERS"] = "0"
    try:
        return rism.RISM3D(grid, tuple(0.5 * n for n in grid), d, su, **kw)
    finally:
        os.environ.pop("RISM_OPTIONAL_BUFFERS", None)


def _optional_bytes(grid, sites, precision):
    n = grid[0] * grid[1] * grid[2]
    words = sites * n + (sites * sites * n // 8 if len(set(grid)) > 1 else 0)
    return words * (12 if precision else 8)


def _free():
    import torch
    return torch.cuda.mem_get_info()[0]


def _exhaust(rism):
    """An allocation that no device has room for."""
    with pytest.raises(rism.RismError) as e:
        rism.copy_bench(1 << 50)
    assert e.value.code == rism.RISM_ERR_NOMEM


@pytest.mark.parametrize("grid,kw", [
    (GRID, {}), ((96, 96, 96), {}), (GRID, {"precision": 1}),
    (GRID, {"precision": 1, "mixed_switch": 1e3, "mixed_block": 3}),
    (GRID, {"anderson_m": 3}),
])
def test_withheld(rism, golden, gpu, grid, kw):
    _make(rism, golden, grid=grid, **kw).close()  # kernels loaded, plans timed
    out, used = [], []
    for withheld in (False, True):
        f0 = _free()
        g = _make(rism, golden, withheld, grid, **kw)
        used.append(f0 - _free())
        g.initialize()
        _, n, _ = g.iterate(maxstep=9, tol=1e-30)
        assert n == 9
        out.append(g.fields(rism.FIELD_T))
        g.close()
    want = _optional_bytes(grid, 4, kw.get("precision", 0))
    if "anderson_m" in kw:
        want -= 4 * grid[0] * grid[1] * grid[2] * 8
    assert abs(used[0] - used[1] - want) <= 8 << 20  # whole pages
    tol = 1e-3 if kw.get("precision") else 1e-9
    assert np.abs(out[0] - out[1]).max() <= tol * np.abs(out[1]).max()


@pytest.mark.parametrize("withheld", [False, True])
def test_batch_without(rism, golden, gpu, withheld):
    """Groups of contexts without the buffers: as separate solves."""
    grid = (40, 48, 32)
    ref = []
    for seed in (3, 4):
        g = _make(rism, golden, withheld, grid, seed)
        g.initialize()
        g.iterate(maxstep=14, tol=1e-30)
        ref.append(g.fields(rism.FIELD_T))
        g.close()
    gs = [_make(rism, golden, withheld, grid, s) for s in (3, 4)]
    for g in gs:
        g.initialize()
    rism.solve_batch(gs, maxstep=14, tol=1e-30)
    for g, t in zip(gs, ref):
        assert np.array_equal(g.fields(rism.FIELD_T), t)
        g.close()


@pytest.mark.parametrize("precision", [0, 1])
def test_given_back(rism, golden, gpu, precision):
    """After every number of steps up to two periods of the slots' rotation,
    before and after the update, and before a graph of a former run is used
    again."""
    grid = (48, 40, 32)
    ref = _make(rism, golden, True, grid, precision=precision).initialize()
    t = []
    for _ in range(14):
        ref.calculate()
        ref.anderson()
        t.append(ref.fields(rism.FIELD_T))
    ref.close()
    tol = 1e-3 if precision else 1e-9
    gs = [_make(rism, golden, False, grid, precision=precision).initialize() for _ in range(26)]
    for i, g in enumerate(gs):
        for _ in range(i // 2):
            g.calculate()
            g.anderson()
        if i % 2:
            g.calculate()
    again = _make(rism, golden, False, grid).initialize()
    again.iterate(maxstep=13, tol=1e-30)
    again.initialize()
    big = _make(rism, golden)
    f0 = _free()
    _exhaust(rism)
    assert _free() - f0 >= _optional_bytes(GRID, 4, 0) - (8 << 20)
    for i, g in enumerate(gs):
        if i % 2:
            g.anderson()
        for _ in range(14 - i // 2 - i % 2):
            g.calculate()
            g.anderson()
        got = g.fields(rism.FIELD_T)
        assert np.abs(got - t[13]).max() <= tol * np.abs(t[13]).max(), i
        g.close()
    if not precision:
        again.iterate(maxstep=14, tol=1e-30)
        got = again.fields(rism.FIELD_T)
        assert np.abs(got - t[13]).max() <= tol * np.abs(t[13]).max()
    again.close()
    big.close()


def test_in_use(rism, golden, gpu):
    """Contexts that other threads run keep theirs: solves are undisturbed."""
    grid = (64, 48, 40)
    ref = _make(rism, golden, False, grid).initialize()
    ref.iterate(maxstep=200, tol=1e-30)
    want = ref.fields(rism.FIELD_T)
    ref.close()
    gs = [_make(rism, golden, False, grid).initialize() for _ in range(3)]
    out = [None] * 3

    def work(i):
        gs[i].iterate(maxstep=200, tol=1e-30)
        out[i] = gs[i].fields(rism.FIELD_T)

    th = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for x in th:
        x.start()
    while any(x.is_alive() for x in th):
        _exhaust(rism)
    for x, g, t in zip(th, gs, out):
        x.join()
        g.close()
        assert np.all(np.isfinite(t))
    # each solve ran with its buffers from its first step, or without them
    alt = _make(rism, golden, True, grid).initialize()
    alt.iterate(maxstep=200, tol=1e-30)
    other = alt.fields(rism.FIELD_T)
    alt.close()
    for t in out:
        assert np.array_equal(t, want) or np.array_equal(t, other)
