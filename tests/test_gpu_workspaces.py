"""Kept device blocks and pinned staging of the host-array calls: what a call
returns does not depend on the calls before it (kept blocks come back zeroed; they
go back to the driver on demand),
on the size of its arrays against the staging buffers (2 MiB each), on another
thread's context or calls, on which context a problem's thickness update goes through, or
on whether the context is still open when a problem goes."""
import threading

import numpy as np
import pytest

from imau_vel import config, geometry
from imau_vel.state import Grid, ProducerState, ThicknessState

pytestmark = pytest.mark.gpu

FIELDS = ("u_vav_cx", "v_vav_cy", "visc_eff_3D_a", "u_3D_a", "w_3D_a", "taub_cx", "N_b", "DIVA_mask_combi")


def solve(ctx, nx, ny, dyn="DIVA"):
    g, cfg, st = geometry.dome(nx, ny, 1450e3 / max(nx, ny))
    config.set_config(cfg, choice_ice_dynamics=dyn, DIVA_visc_it_nit=5)
    (ctx.solve_diva if dyn == "DIVA" else ctx.solve_sia)(g, cfg, st)
    return {f: st[f].copy() for f in FIELDS}


def same(a, b):
    for f in FIELDS:
        np.testing.assert_array_equal(a[f], b[f], err_msg=f)


def test_results_do_not_depend_on_earlier_calls():
    from imau_vel import solver
    with solver.Context() as fresh:
        ref = solve(fresh, 29, 31)
    with solver.Context() as ctx:
        for nx, ny, dyn in ((61, 57, "DIVA"), (30, 30, "SIA"), (17, 90, "DIVA")):
            solve(ctx, nx, ny, dyn)
        same(solve(ctx, 29, 31), ref)
        same(solve(ctx, 29, 31), ref)


@pytest.mark.parametrize("nx,ny", [(31, 37), (129, 135), (4, 40000), (300, 301)])
def test_transfers_of_any_size(nx, ny):
    """The rheology's 3D fields are downloaded whole: below one staging buffer,
    several, rows longer than half a buffer, and more than the ring holds."""
    from imau_vel import solver
    g = Grid(nx, ny, 5e3)
    ps = ProducerState(g, 15)
    rng = np.random.default_rng(nx)
    for f in ("mask_ice_a", "mask_sheet_a"):
        ps[f] = 1
    ps["Ti_a"] = rng.uniform(240.0, 262.0, (15, ny, nx))
    with solver.Context() as ctx:
        ctx.calc_ice_rheology(g, config.producer_config(), ps)
    A = 1.14e-05 * np.exp(-6.0e+04 / (8.314 * ps["Ti_a"]))
    np.testing.assert_allclose(ps["A_flow_3D_a"], A, rtol=1e-13)
    np.testing.assert_array_equal(ps["A_flow_3D_cx"], (ps["A_flow_3D_a"][:, :, :-1] + ps["A_flow_3D_a"][:, :, 1:]) / 2)
    np.testing.assert_array_equal(ps["A_flow_3D_cy"], (ps["A_flow_3D_a"][:, :-1] + ps["A_flow_3D_a"][:, 1:]) / 2)


def test_contexts_of_two_threads():
    from imau_vel import solver
    sizes = [(29, 31), (45, 33)]
    ref, got, errs = [], [None, None], []
    for nx, ny in sizes:
        with solver.Context() as ctx:
            ref.append(solve(ctx, nx, ny))

    def work(q):
        try:
            with solver.Context() as ctx:
                for _ in range(3):
                    got[q] = solve(ctx, *sizes[q])
        except Exception as e:
            errs.append(e)
    threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errs, errs
    for q in range(2):
        same(got[q], ref[q])


def test_two_threads_in_one_context():
    """Host-array calls of two threads on the same context, bit for bit."""
    from imau_vel import solver
    g = Grid(281, 283, 8e3)
    rng = np.random.default_rng(7)
    ts, ps = ThicknessState(g), ProducerState(g, 15)
    ts["Hi_a"] = rng.uniform(500.0, 900.0, (g.ny, g.nx))
    ts["u_vav_cx"] = rng.uniform(-150.0, 150.0, (g.ny, g.nx - 1))
    ts["v_vav_cy"] = rng.uniform(-150.0, 150.0, (g.ny - 1, g.nx))
    ts["mask_ice_a"], ts["float_margin_frac_a"] = 1, 1.0
    for f in ("mask_ice_a", "mask_sheet_a"):
        ps[f] = 1
    ps["Ti_a"] = rng.uniform(240.0, 262.0, (15, g.ny, g.nx))
    tcfg, pcfg = config.thickness_config(choice_ice_integration_method="explicit"), config.producer_config()

    def thickness(ctx):
        out = ts.copy()
        ctx.thickness_update(g, tcfg, out, 2.0)
        return [out[f].copy() for f in ("dHi_dt_a", "Hi_tplusdt_a", "Qx_cx", "Qy_cy")]

    def rheology(ctx):
        ctx.calc_ice_rheology(g, pcfg, ps)
        return [ps[f].copy() for f in ("A_flow_3D_a", "A_flow_3D_cx", "A_flow_3D_cy", "A_flow_vav_a", "A_flow_vav_cy")]

    calls, errs, bad = (thickness, rheology), [], []
    with solver.Context() as ctx:
        ref = [f(ctx) for f in calls]

        def work(q):
            try:
                for _ in range(20):
                    if not all(np.array_equal(a, b) for a, b in zip(calls[q](ctx), ref[q])):
                        bad.append(q)
            except Exception as e:
                errs.append(e)
        threads = [threading.Thread(target=work, args=(q,)) for q in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not errs and not bad, (errs, bad)


def test_device_memory_goes_back():
    """What host-array calls keep is reported and given back on demand, and a
    destroyed problem's memory (10 MB and more here) goes back by itself."""
    import torch
    from imau_vel import solver
    with solver.Context() as ctx:
        ref = solve(ctx, 61, 57)
        assert ctx.keep_memory() > 0
        assert ctx.keep_memory(0) == 0
        same(solve(ctx, 61, 57), ref)
        assert ctx.keep_memory() == 0
        ctx.keep_memory(4 << 30)
        same(solve(ctx, 61, 57), ref)
        kept = ctx.keep_memory()
        assert 0 < kept <= 4 << 30
        g, cfg, st = geometry.dome(201, 203, 8e3)
        free = torch.cuda.mem_get_info()[0]
        prob = ctx.problem([g], cfg, [st])
        assert torch.cuda.mem_get_info()[0] < free
        prob.close()
        assert torch.cuda.mem_get_info()[0] >= free - (8 << 20)    # the driver's own granularity
        assert ctx.keep_memory() == kept


def test_problem_outlives_its_context():
    """A problem solved through another context, after its own is closed and
    with buffers allocated only then, gives what a context of its own gives."""
    from imau_vel import solver
    later = dict(stop_rule=1, nonlinear_rtol=1e-3, DIVA_visc_it_nit=40, anderson_m=2, ksp_type=1, precision="mixed_visc")
    g, cfg, st = geometry.dome()
    config.set_config(cfg, DIVA_visc_it_nit=3)
    ref = st.copy()
    first, second = solver.Context(), solver.Context()
    prob = first.problem([g], cfg, [st])
    prob.solve(cfg)
    first._check(first.L.imau_net_sync(first.h))
    first.close()
    config.set_config(cfg, **later)
    prob.ctx = second
    prob.reset_state()
    prob.solve(cfg)
    prob.download()
    prob.close()
    prob = second.problem([g], cfg, [ref])
    prob.solve(cfg)
    prob.download()
    prob.close()
    second.close()
    for f in ("u_vav_cx", "v_vav_cy", "visc_eff_3D_a", "u_3D_a"):
        np.testing.assert_array_equal(st[f], ref[f], err_msg=f)


def test_thickness_through_another_context():
    """reset_state does not wait; a thickness update through a second context
    still sees the restored velocities, also when the problem's own stream has
    work in front of the copies (network passes, a few ms)."""
    import torch
    from imau_vel import learned, solver
    g, cfg, st = geometry.dome()
    config.set_config(cfg, DIVA_visc_it_nit=3)
    with solver.Context() as first, solver.Context() as second:
        prob = first.problem([g], cfg, [st])
        net = learned.Net(first, seed=0)
        plan = learned.Plan(first, rows=[512] * 4, cols=[512] * 4)
        x = torch.zeros(plan.npix[0] * learned.NFEAT, dtype=torch.int16, device="cuda")
        torch.cuda.synchronize()
        tcfg, out = config.thickness_config(), []
        for ctx in (first, second):
            prob.ctx = first
            prob.solve(cfg)
            for _ in range(10):
                net.forward(plan, x)
            prob.reset_state()
            prob.ctx = ctx
            ts = ThicknessState(g)
            for f in ("Hi_a", "Hb_a", "SL_a", "mask_ice_a", "mask_shelf_a", "mask_ocean_a"):
                ts[f] = st[f]
            ts["SMB_year"], ts["float_margin_frac_a"] = 0.3, 1.0
            prob.thickness(0, tcfg, ts, 5.0)
            out.append(ts["dHi_dt_a"].copy())
        net.sync()
        net.release(plan)
        plan.close()
        prob.close()
    np.testing.assert_array_equal(out[0], out[1])
    # no velocity: the surface mass balance alone, away from the margin and the cleared boundary rows
    np.testing.assert_allclose(out[0][10:-10, 10:-10], 0.3, rtol=1e-9)
