"""The fused multigrid sweeps against one launch per colour (mg_smoother 0 and
1), at grid sizes whose levels end on, just before and just past a tile edge
(tiles of 16 x 64 cells on the fine level, 8 x 64 on the coarse ones), in both
precisions, with and without calving fronts, cross terms and periodic sides.
Both forms do the same arithmetic, so the solves are equal bit for bit."""
import numpy as np
import pytest

import branch_cases
from imau_vel import config, geometry

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from imau_vel import solver
    c = solver.Context()
    yield c
    c.close()


SIZES = [(5, 7), (17, 65), (33, 34), (66, 130), (129, 127), (130, 128), (131, 129), (40, 257), (259, 34)]
CASES = [(s, p, "cap") for s in SIZES for p in ("fp64", "mixed")]
CASES += [(s, p, kind) for s in ((61, 21), (130, 66)) for p in ("fp64", "mixed") for kind in ("sans", "periodic")]
CASES += [((61, 21), p, "BC") for p in ("fp64", "mixed")]


@pytest.mark.parametrize("shape,precision,kind", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_fused_sweeps_equal_colour_launches(ctx, shape, precision, kind):
    nx, ny = shape
    if kind == "cap":
        g, cfg, st = geometry.random_geometry(nx, ny, seed=nx + ny, beta_sq=1e4)
    elif kind == "BC":
        _, g, cfg, st = branch_cases.bc_margin_case()
    else:
        kw = {"sans": dict(include_SSADIVA_crossterms=0),
              "periodic": {"DIVA_boundary_BC_%s_%s" % (c, d): "periodic" for c in "uv"
                           for d in ("west", "east", "south", "north")}}[kind]
        g, cfg, st = geometry.channel(nx=nx, ny=ny, dx=8e3, cfg=geometry.synthetic_config(**kw))
    config.set_config(cfg, stop_rule=1, nonlinear_rtol=1e-12, DIVA_visc_it_nit=3, precision=precision,
                      ksp_type=0 if kind == "BC" else 1)
    st.DIVA_PETSc_rtol, st.DIVA_PETSc_abstol, st.DIVA_SOR_nit = 1e-2, 0.0, 6
    out = []
    for smoother in (0, 1):
        config.set_config(cfg, mg_smoother=smoother)
        s = st.copy()
        ctx.solve_diva(g, cfg, s)
        out.append(s)
    assert np.abs(out[0]["u_vav_cx"]).max() > 0.0
    for f in ("u_vav_cx", "v_vav_cy", "visc_eff_3D_a"):
        np.testing.assert_array_equal(out[0][f], out[1][f], err_msg=f)
