"""Refined meshes whose number of cells per direction is no power of two: midpoints of neighbours on
one level differ in the last bits across the mesh. Such a difference is no transverse offset, so no
slope launch reads slopes that it writes itself, and a step gives the same bits every time.
Against the oracle, which projects over the rounding: 1e-12 as in the parity tests."""
import numpy as np
import pytest

import oracle as O
from _util import pair, rel_err, rel_err_rows, say
from kitamr_hip import cases
from kitamr_hip.solver import kah_params

SHAPES = {
    "box": lambda: cases.box_3d(n=6, nv=12, ps_levels=1),
    "riemann": lambda: cases.riemann_2d(n=28, nv=10, ps_levels=2),
    "riemann-adapted": lambda: cases.riemann_2d(n=14, nv=10, ps_levels=2, vs_levels=1,
                                                vs_variants=5),
}


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(SHAPES))
def test_steps_repeat(name):
    case = SHAPES[name]()
    mid = np.asarray(case.topo["cell_mid"])
    say(f"[slope order] {name}: cells={case.n_cells} P={case.phase_cells}")
    assert np.any(mid * 2.0 ** 20 != np.round(mid * 2.0 ** 20))   # not exact in binary
    states = []
    for options in ({"branches": 1}, {"branches": 1}, {"branches": 3}, {"regular": 0}):
        dev, orc = pair(case, options=options)
        for s in range(4):
            dev.step(case.dt_xi, s)
        states.append(dev.get_state(sdf=True))
        dev.close()
    for s in range(4):
        orc.step(case.dt_xi, s)
    g, o = states[0], orc.get_state()
    for other in states[1:]:
        for k in ("w", "prim", "qf", "df", "sdf"):
            assert np.array_equal(g[k], other[k]), k
    nw = case.config.solver.DIM + 2
    assert rel_err(g["df"], o["df"]) <= 1e-12
    assert rel_err_rows(g["w"].reshape(-1, nw), o["w"].reshape(-1, nw), nw) <= 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("n", [6, 8, 12])
def test_narrow_levels(n):
    """Cells with a coarser neighbour on one side and finer ones on the other: the mean of the finer
    midpoints is the cell's own up to rounding, so there is no projection on that side. Measured
    against the oracle on the same mesh in units of its cells, where every midpoint is exact: slopes
    to 1e-12 of the largest (differences of values alike in both, divided by sizes that round)."""
    case = cases.riemann_2d(n=n, nv=8, ps_levels=2, halo=(2.0, 1.5, 1.0))
    state = np.asarray(case.topo["nb_state"]).reshape(-1, 2, 2)
    narrow = int(np.sum(np.any(state == -1, axis=2) & np.any(state == 2, axis=2)))
    say(f"[slope order] narrow n={n}: cells={case.n_cells}, {narrow} between coarse and fine")
    assert narrow > 0
    # a factor per cell that is curved along both directions: slopes across the faces and along them
    x, y = np.asarray(case.topo["cell_mid"]).reshape(-1, 2)[:case.n_cells].T
    size = np.diff(np.asarray(case.topo["vs_offset"])) * 2
    case.df = case.df * np.repeat(1.0 + 0.3 * np.sin(3.0 * x + 2.0 * y) + 0.2 * x * y, size)
    dev, orc = pair(case)
    for _ in range(2):   # the second sweep finds slopes in the finer cells
        dev.slope(case.dt_xi)
    g = dev.get_state(sdf=True)
    dev.close()
    orc.close()
    topo = dict(case.topo)
    for k in ("cell_mid", "cell_ds", "pair_mid"):
        topo[k] = np.round(np.asarray(topo[k]) * n * 1024) / 1024
    exact = O.Oracle(kah_params(case.config), topo)
    exact.set_state(case.w, case.prim, case.df)
    for _ in range(2):
        exact.slope()
    assert rel_err(g["sdf"], exact.get_state()["sdf"] * n) <= 1e-12
