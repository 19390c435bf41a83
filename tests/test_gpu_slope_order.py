"""Refined meshes whose number of cells per direction is no power of two: midpoints of neighbours on
one level differ in the last bits across the mesh. Such a difference is no transverse offset, so no
slope launch reads slopes that it writes itself, and a step gives the same bits every time.
Against the oracle, which projects over the rounding: 1e-12 as in the parity tests."""
import numpy as np
import pytest

from _util import pair, rel_err, rel_err_rows, say
from kitamr_hip import cases

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
