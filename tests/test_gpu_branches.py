"""Streams of the independent launches of a phase (KAH_OPT_BRANCHES): one, two and three streams and
the library's choice by shape give the same state bit for bit, on meshes of both sides of that
choice: meshes below and above 2,048,000 velocity cells (2D) and 786,432 (3D), adapted grids below
and above the largest grid from which the launches run side by side."""
import numpy as np
import pytest

from _util import say
from kitamr_hip import abi, cases
from kitamr_hip.solver import kah_params

# name: (case, velocity cells in all, largest grid)
SHAPES = {
    "shared": (lambda: cases.riemann_2d(n=10, nv=16, ps_levels=1), (0, 2048000), None),
    "shared-large": (lambda: cases.riemann_2d(n=28, nv=30, ps_levels=1), (2048000, None), None),
    "box": (lambda: cases.box_3d(n=4, nv=8, ps_levels=1), (0, 786432), None),
    "box-large": (lambda: cases.box_3d(n=6, nv=12, ps_levels=1), (786432, None), None),
    "adapted-small": (lambda: cases.riemann_2d(n=8, nv=8, ps_levels=2, vs_levels=1, vs_variants=5),
                      (0, 2048000), (0, 384)),
    "adapted-fp32": (lambda: cases.riemann_2d(n=8, nv=16, ps_levels=1, vs_levels=1, vs_variants=5,
                                              precision="fp32f"), (0, 2048000), (384, 768)),
    "adapted": (lambda: cases.riemann_2d(n=8, nv=16, ps_levels=1, vs_levels=2, vs_variants=5),
                (0, 2048000), (768, None)),
    "adapted-mesh": (lambda: cases.riemann_2d(n=44, nv=10, ps_levels=2, vs_levels=1, vs_variants=5),
                     (2048000, None), (0, 384)),
    "adapted-box": (lambda: cases.box_3d(n=3, nv=6, ps_levels=1, vs_levels=1, vs_variants=5),
                    (0, 786432), (512, None)),
}


def within(x, bounds):
    return bounds is None or (x >= bounds[0] and (bounds[1] is None or x < bounds[1]))


@pytest.mark.parametrize("name", list(SHAPES))
def test_shapes(name):
    """The meshes of the test below are on the side of the choice they stand for."""
    make, cells, grid = SHAPES[name]
    case = make()
    n = int(np.diff(np.asarray(case.topo["vs_offset"])).max())
    assert within(case.phase_cells, cells), case.phase_cells
    assert within(n, grid), n


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [0, 1])
@pytest.mark.parametrize("name", list(SHAPES))
def test_branches_agree(name, graphs):
    case = SHAPES[name][0]()
    say(f"[branches] {name} graphs={graphs}: cells={case.n_cells} P={case.phase_cells}")
    ctx = []
    for branches in ((1,), (), (2,), (3,), (1, 4)):   # the last: back to the library's choice
        dev = abi.HipContext(kah_params(case.config))
        dev.set_option("graphs", graphs)
        for b in branches:
            dev.set_option("branches", b)
        dev.set_topology(case.topo)
        dev.set_state(case.w, case.prim, case.df)
        ctx.append(dev)
    for s in range(4):   # both parities of a captured step, and their replays
        for dev in ctx:
            dev.step(case.dt_xi, s)
    one = ctx[0].get_state(sdf=True)
    for dev in ctx[1:]:
        g = dev.get_state(sdf=True)
        for k in ("w", "prim", "qf", "df", "sdf"):
            assert np.array_equal(one[k], g[k]), k
    for dev in ctx:
        dev.close()
