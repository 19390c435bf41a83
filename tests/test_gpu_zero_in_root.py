"""Adapted velocity grids whose root lattice has v = 0 inside a root cell. The solver's
configurations refuse such a lattice, the C ABI takes it: a coarse velocity cell at rest then
overlaps finer ones that leave their cells through opposite faces, so the micro flux a neighbour
stores at one of them need not be the one through the shared face.

The reference's walk over two such grids has no meaning (it counts the velocity cells of the
upwind sets), so the measure is the general gather, which reconstructs at the neighbour's own
velocities (KAH_OPT_REGULAR 0): the default, with and without overlap maps, equals it bit for bit."""
import numpy as np
import pytest

from _util import say
from kitamr_hip import abi, cases
from kitamr_hip.solver import kah_params

SHAPES = {
    "one-level": lambda p: cases.riemann_2d(n=8, nv=8, vs_levels=2, vs_variants=5, precision=p),
    "hanging": lambda p: cases.riemann_2d(n=8, nv=8, ps_levels=1, vs_levels=2, vs_variants=5,
                                          precision=p),
    "box-hanging": lambda p: cases.box_3d(n=4, nv=6, ps_levels=1, vs_levels=1, vs_variants=2,
                                          precision=p),
}


def at_rest_inside_a_root(case):
    """The case in a frame that moves by half a root cell: the lattice, the flow and its energy."""
    dim, topo = case.config.solver.DIM, dict(case.topo)
    lo, hi = np.array(topo["vs_lo"], dtype=float), np.array(topo["vs_hi"], dtype=float)
    s = 0.5 * (hi[0] - lo[0]) / topo["vs_trees_num"][0]
    topo["vs_lo"], topo["vs_hi"] = lo + s, hi + s
    topo["vs_mid"] = np.asarray(topo["vs_mid"]) + s   # root cells are cubes
    case.topo = topo
    w = np.array(case.w).reshape(-1, dim + 2)
    w[:, -1] += s * w[:, 1:-1].sum(axis=1) + 0.5 * dim * s * s * w[:, 0]
    w[:, 1:-1] += s * w[:, :1]
    prim = np.array(case.prim).reshape(-1, dim + 2)
    prim[:, 1:-1] += s
    case.w, case.prim = w.reshape(np.shape(case.w)), prim.reshape(np.shape(case.prim))
    return case


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32f"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_zero_in_root(name, precision):
    case = at_rest_inside_a_root(SHAPES[name](precision))
    mid = np.asarray(case.topo["vs_mid"])
    say(f"[zero in root] {name} {precision}: cells={case.n_cells}, at rest {np.sum(mid == 0.0)}, "
        f"slowest {np.abs(mid[mid != 0.0]).min():.3f}")
    dt = 0.5 * case.dt_xi   # the frame's speed adds to the fastest velocities
    states = []
    for options in ({"regular": 0}, {}, {"overlap_maps": 0}):
        dev = abi.HipContext(kah_params(case.config))
        for k, v in options.items():
            dev.set_option(k, v)
        dev.set_topology(case.topo)
        dev.set_state(case.w, case.prim, case.df)
        for s in range(2):
            dev.step(dt, s)
        states.append(dev.get_state(sdf=True))
        dev.close()
    assert np.all(np.isfinite(states[0]["df"]))
    for other in states[1:]:
        for k in ("w", "prim", "qf", "df", "sdf"):
            assert np.array_equal(states[0][k], other[k]), k
