"""The chunked slope kernels and the stored gathers at the edges of their launch shapes: grids just
below, at and above a wave, a workgroup and a chunk, refined meshes (hanging faces, blocks of their
own for the micro fluxes of a coarse side), adapted grids with overlap maps and with the key
search, walls, outflow and inflow sides and immersed boundaries beside regular cells.

FP64 against the oracle: sums of at most a few thousand terms in another order, 1e-12 as in the
parity tests. FP32 form: every f is rounded to float each step (6e-8), 2 steps stay within 1e-6
of the largest f; regular and general path bit for bit in both forms."""
import numpy as np
import pytest

from _util import pair, rel_err, rel_err_rows, say
from kitamr_hip import abi, cases
from kitamr_hip.solver import kah_params

SHAPES = {
    "wave": lambda p: cases.riemann_2d(n=6, nv=8, precision=p),
    "wave+": lambda p: cases.riemann_2d(n=6, nv=10, precision=p),
    "group": lambda p: cases.riemann_2d(n=6, nv=16, precision=p),
    "chunk-": lambda p: cases.riemann_2d(n=6, nv=24, precision=p),
    "chunk+": lambda p: cases.riemann_2d(n=6, nv=28, precision=p),
    "chunks": lambda p: cases.riemann_2d(n=5, nv=42, precision=p),
    "hanging": lambda p: cases.riemann_2d(n=8, nv=10, ps_levels=2, precision=p),
    "hanging-adapted": lambda p: cases.riemann_2d(n=8, nv=8, ps_levels=1, vs_levels=2,
                                                  vs_variants=5, precision=p),
    "period-adapted": lambda p: cases.periodic_box_2d(n=8, nv=8, ps_levels=1, vs_levels=2,
                                                      precision=p),
    "box": lambda p: cases.box_3d(n=4, nv=12, precision=p),
    "box-hanging": lambda p: cases.box_3d(n=4, nv=6, ps_levels=1, precision=p,
                                          bcs=("SuperSonicInflow", "UniformOutflow") * 3),
    "box-adapted": lambda p: cases.box_3d(n=4, nv=6, ps_levels=1, vs_levels=1, precision=p),
    "walls": lambda p: cases.box_3d(n=4, nv=6, precision=p, bcs=("Maxwellian",) * 2 +
                                    ("UniformOutflow",) * 4),
    "cylinder": lambda p: cases.cylinder_2d(n=16, nv=10, vs_levels=2, precision=p),
}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32f"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_edges(name, precision):
    case = SHAPES[name](precision)
    say(f"[slope chunks] {name} {precision}: cells={case.n_cells} P={case.phase_cells}")
    live = case.topo["bound_enc"] >= 0
    rows = np.repeat(live, np.diff(np.asarray(case.topo["vs_offset"])) * case.config.solver.NDF)
    states = []
    for options in ({}, {"regular": 0}, {"overlap_maps": 0}):
        dev, orc = pair(case, options=options)
        for s in range(2):
            dev.step(case.dt_xi, s)
            orc.step(case.dt_xi, s)
        states.append(dev.get_state(sdf=True))
        dev.close()
    g, o = states[0], orc.get_state()
    tol = 1e-12 if precision == "fp64" else 1e-6
    nw = case.config.solver.DIM + 2
    assert rel_err(g["df"][rows], o["df"][rows]) <= tol
    assert rel_err_rows(g["w"].reshape(-1, nw)[live], o["w"].reshape(-1, nw)[live], nw) <= tol
    for other in states[1:]:
        for k in ("w", "prim", "qf", "df", "sdf"):
            assert np.array_equal(g[k], other[k]), k


@pytest.mark.gpu
@pytest.mark.parametrize("vpt", [1, 2, 4, 6])
def test_chunk_sizes_agree(vpt):
    """Another number of velocity cells per thread changes the order of the sums only."""
    case = cases.riemann_2d(n=8, nv=28, ps_levels=1)
    out = []
    for options in ({}, {"slope_vpt": vpt}):
        dev = abi.HipContext(kah_params(case.config))
        for k, v in options.items():
            dev.set_option(k, v)
        dev.set_topology(case.topo)
        dev.set_state(case.w, case.prim, case.df)
        for s in range(2):
            dev.step(case.dt_xi, s)
        out.append(dev.get_state(sdf=True))
        dev.close()
    for k in ("w", "df", "sdf"):
        assert rel_err(out[1][k], out[0][k]) <= 1e-12, k
