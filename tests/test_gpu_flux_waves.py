"""The number of waves the flux/relaxation kernel picks by shape: shared grids with cells enough for
few waves per workgroup, CIP_Marching on 2 and 4, one velocity cell more than the waves cover evenly,
3D adapted grids whose LDS copy leaves one workgroup per CU and those in global memory (16 waves).

FP64 against the oracle and against 8 waves: sums in another order, 1e-12 as in the parity tests.
FP32 form: f rounded to float each step (6e-8), 2 steps within 1e-6 of the largest f."""
import numpy as np
import pytest

from _util import pair, rel_err, rel_err_rows, say
from kitamr_hip import cases

SHAPES = {
    "few-waves": lambda p: cases.riemann_2d(n=44, nv=14, precision=p),
    "few-waves-hanging": lambda p: cases.riemann_2d(n=24, nv=18, ps_levels=1, precision=p),
    "euler": lambda p: cases.riemann_2d(n=44, nv=10, marching="Euler", precision=p),
    "box": lambda p: cases.box_3d(n=12, nv=6, precision=p),
    "lds-copy": lambda p: cases.box_3d(n=4, nv=18, vs_levels=1, precision=p),
    "global-copy": lambda p: cases.box_3d(n=3, nv=26, vs_levels=1, precision=p),
    "cip-2": lambda p: cases.riemann_2d(n=40, nv=10, marching="CIP_Marching", precision=p),
    "cip-4": lambda p: cases.riemann_2d(n=40, nv=36, marching="CIP_Marching", precision=p),
}


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32f"])
@pytest.mark.parametrize("name", list(SHAPES))
def test_waves_by_shape(name, precision):
    case = SHAPES[name](precision)
    grid = int(np.diff(np.asarray(case.topo["vs_offset"])).max())
    say(f"[flux waves] {name} {precision}: cells={case.n_cells} largest grid={grid}")
    dev, orc = pair(case)
    eight, _ = pair(case, options={"flux_waves": 8})
    general, _ = pair(case, options={"regular": 0})
    for s in range(2):
        for d in (dev, eight, general, orc):
            d.step(case.dt_xi, s)
    g, e, r, o = dev.get_state(), eight.get_state(), general.get_state(), orc.get_state()
    for d in (dev, eight, general):
        d.close()
    tol = 1e-12 if precision == "fp64" else 1e-6
    nw = case.config.solver.DIM + 2
    for other in (o, e):
        assert rel_err(g["df"], other["df"]) <= tol
        assert rel_err_rows(g["w"].reshape(-1, nw), other["w"].reshape(-1, nw), nw) <= tol
    for k in ("w", "prim", "qf", "df"):
        assert np.array_equal(g[k], r[k]), k


# 16-wave workgroups in the FP64 form with the copy of f* in LDS: 2D cells with neighbours on other
# levels or at the domain's edge whose grids lie above 2,048 velocity cells (and below the 6,485 that
# fit 152 KiB), 3D grids whose copy takes more than 56 KiB and fits (3,585 to 9,728).
WIDE = {
    "2d": (lambda: cases.riemann_2d(n=6, nv=26, vs_levels=2), 2049, 6485),
    "2d-hanging": (lambda: cases.riemann_2d(n=5, nv=26, ps_levels=1, vs_levels=2, vs_variants=5),
                   2049, 6485),
    "3d": (lambda: cases.box_3d(n=3, nv=14, vs_levels=1), 3585, 9728),
}


@pytest.mark.parametrize("name", list(WIDE))
def test_wide_shapes(name):
    make, lo, hi = WIDE[name]
    sizes = np.diff(np.asarray(make().topo["vs_offset"]))
    assert lo <= sizes.min() and sizes.max() <= hi, (sizes.min(), sizes.max())


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(WIDE))
def test_wide_workgroups(name):
    case = WIDE[name][0]()
    say(f"[flux waves] wide {name}: cells={case.n_cells} P={case.phase_cells}")
    dev, orc = pair(case)
    eight, _ = pair(case, options={"flux_waves": 8})
    general, _ = pair(case, options={"regular": 0})
    for s in range(2):
        for d in (dev, eight, general, orc):
            d.step(case.dt_xi, s)
    g, e, r, o = dev.get_state(), eight.get_state(), general.get_state(), orc.get_state()
    for d in (dev, eight, general):
        d.close()
    nw = case.config.solver.DIM + 2
    for other in (o, e):   # sums of a few thousand terms in another order, as above
        assert rel_err(g["df"], other["df"]) <= 1e-12
        assert rel_err_rows(g["w"].reshape(-1, nw), other["w"].reshape(-1, nw), nw) <= 1e-12
    for k in ("w", "prim", "qf", "df"):
        assert np.array_equal(g[k], r[k]), k
