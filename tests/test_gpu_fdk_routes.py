"""Each kernel that the FDK's rules choose, against the FP64 oracle, with the choice asserted: window
edges, tuned shapes, chunks of views, and the row projector's blocks of rows."""
import math

import numpy as np
import pytest

from conftest import oracle_geom, rel_l2, rel_max
from fdk_routes import routes

pytestmark = pytest.mark.gpu

TOL = 1e-5


def _t(x):
    import torch

    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


def _scan(back=False, **kw):
    from monte_amd import geometry as G

    base = dict(nu=96, nv=80, sod=30.0, sdd=60.0, du=0.1, dv=0.08, vx=0.04, vy=0.04, vz=2.6 / kw["nz"], u_off=0.02,
                v_off=-0.03, oz=0.01)
    return G.Geometry(**{**base, **kw}, dangle=-2.0 * math.pi / kw["n_views"] if back else None)


# name: (orbit, groups, zc, stack), scan.  The detectors are smaller than the volume's projection, so
# samples are clamped onto the guard zeros on all sides.
_PAST = {
    "quarter": ((4, 1, 16, 1), dict(nx=65, ny=65, nz=915, n_views=12, nu=40, nv=50)),
    "quarter_even_back": ((4, 1, 16, 1), dict(nx=66, ny=66, nz=910, n_views=8, nu=41, nv=40, back=True)),
    "quarter_8_four_groups": ((4, 4, 8, 1), dict(nx=65, ny=65, nz=130, n_views=16, nu=40, nv=50)),
    "quarter_two_groups": ((4, 2, 16, 1), dict(nx=66, ny=66, nz=840, n_views=8, nu=41, nv=200, dv=0.02)),
    "half": ((2, 1, 16, 1), dict(nx=51, ny=67, nz=705, n_views=10, nu=40, nv=50)),
    "one_32": ((1, 1, 32, 1), dict(nx=51, ny=66, nz=1301, n_views=5, nu=40, nv=40)),
    "one_16": ((1, 1, 16, 1), dict(nx=51, ny=66, nz=420, n_views=5, nu=40, nv=40)),
    "one_8_steep": ((1, 2, 8, 1), dict(nx=100, ny=90, nz=64, n_views=21, nu=60, nv=150, dv=0.021)),
    "one_4_four_groups": ((1, 4, 4, 1), dict(nx=64, ny=64, nz=40, n_views=17, nu=40, nv=40)),
    "stacked": ((1, 4, 16, 4), dict(nx=100, ny=72, nz=90, n_views=21, nu=150, du=0.02, nv=50)),
    "stacked_8": ((1, 1, 8, 4), dict(nx=129, ny=129, nz=257, n_views=5, nu=200, du=0.02, nv=200, dv=0.015)),
}


@pytest.mark.parametrize("name", list(_PAST))
def test_backprojection_past_the_detector(ctx, oracle, name):
    from monte_amd.fdk import fdk_backproject

    plan, kw = _PAST[name]
    g = _scan(**kw)
    assert routes(g)[:4] == plan
    f = np.random.default_rng(len(name)).standard_normal(g.filt_shape).astype(np.float32)
    ref = oracle.fdk_std_backproject(oracle_geom(oracle, g), f)
    got = fdk_backproject(_t(f), g, ctx).cpu().numpy()
    print(name, rel_max(got, ref), rel_l2(got, ref), "zeros", float((ref == 0).mean()))
    assert (ref == 0).any(), "the volume does not leave the detector"
    assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL


_TUNED = {
    "quarter": ((4, 1, 16, 1), dict(nx=65, ny=65, nz=915, n_views=12)),
    "quarter_8": ((4, 4, 8, 1), dict(nx=65, ny=65, nz=130, n_views=16)),
    "half": ((2, 1, 16, 1), dict(nx=51, ny=67, nz=705, n_views=10)),
    "half_four_groups": ((2, 4, 16, 1), dict(nx=51, ny=67, nz=300, n_views=18)),
    "one_32": ((1, 1, 32, 1), dict(nx=51, ny=66, nz=1301, n_views=5)),
    "one_four_groups": ((1, 4, 16, 1), dict(nx=100, ny=90, nz=64, n_views=71)),
    "stacked": ((1, 4, 16, 4), dict(nx=100, ny=72, nz=90, n_views=21, nu=400, du=0.02)),
    "direct": ((0, 1, 0, 1), dict(nx=33, ny=31, nz=45, n_views=9)),
}


@pytest.mark.parametrize("name", list(_TUNED))
def test_volume_does_not_depend_on_tuned_shapes(ctx, name):
    import torch

    from monte_amd.fdk import fdk_backproject

    plan, kw = _TUNED[name]
    g = _scan(**kw)
    assert routes(g)[:4] == plan
    f = _t(np.random.default_rng(3).standard_normal(g.filt_shape).astype(np.float32))
    saved, shapes = ctx.tuning, set()
    ref = fdk_backproject(f, g, ctx)
    try:
        for zc in (4, 8, 16):
            for tx in (8, 16, 32, 64):
                r = routes(g, bp_zchunk=zc, bp_tile_x=tx)
                assert (r.orbit, r.groups, r.stack) == (plan[0], plan[1], plan[3])
                shapes.add((r.zc, r.tile_x))
                ctx.set_tuning(bp_zchunk=zc, bp_tile_x=tx)
                assert torch.equal(fdk_backproject(f, g, ctx), ref), (zc, tx, r)
    finally:
        ctx.set_tuning(**saved)
    print(name, sorted(shapes))
    assert len(shapes) >= {"direct": 1, "stacked": 3, "quarter_8": 4}.get(name, 6)


@pytest.mark.parametrize("name,chunks", [("quarter", (1, 5, 11)), ("half", (3, 9)), ("one_four_groups", (1, 3, 70)),
                                         ("one_32", (2, 4)), ("stacked", (2, 20)), ("direct", (1, 4, 8))])
def test_backprojection_in_chunks_of_views(ctx, oracle, name, chunks):
    """Chunks take orbits apart, leave groups without views and end in a remainder."""
    from monte_amd.fdk import fdk_backproject

    plan, kw = _TUNED[name]
    g = _scan(**kw)
    f = np.random.default_rng(4).standard_normal(g.filt_shape).astype(np.float32)
    ref = oracle.fdk_std_backproject(oracle_geom(oracle, g), f)
    saved = ctx.tuning
    try:
        for n in chunks:
            assert routes(g, bp_view_chunk=n).orbit == min(plan[0], 1)
            ctx.set_tuning(bp_view_chunk=n)
            got = fdk_backproject(_t(f), g, ctx).cpu().numpy()
            print(name, n, rel_max(got, ref))
            assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL
    finally:
        ctx.set_tuning(**saved)


def test_bp3d20_in_chunks_of_views(ctx, oracle):
    from monte_amd import geometry as G
    from monte_amd.fdk import fdk
    from synth import bp3d20_sphere_stack

    for kw, orbit in ((dict(nx=120, ny=128, nz=140, vx=0.2, vy=0.2, vz=0.2, roi_x0=3, roi_x1=118), 1), (dict(), 0)):
        g = G.bp3d20_65(n_views=6).replace(**kw)
        assert routes(g, bp_view_chunk=4).orbit == orbit
        proj = bp3d20_sphere_stack(65, g.du)[:6]
        ref, _ = oracle.bp3d20_fdk(oracle_geom(oracle, g), proj)
        saved = ctx.tuning
        try:
            for n in (1, 4):
                ctx.set_tuning(bp_view_chunk=n)
                got = fdk(_t(proj), g, ctx).cpu().numpy()
                assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL
        finally:
            ctx.set_tuning(**saved)


def _row_scan(nu=60, step=0.9, nv=None, **kw):
    from monte_amd import geometry as G

    v = 4.0 / max(kw["nx"], kw["ny"], 8)
    return G.Geometry(**{**dict(nu=nu, nv=nv or int(kw["nz"] * step) + 14, sod=40.0, sdd=80.0, du=10.2 / nu, dv=0.04,
                                vx=v, vy=v, vz=step * 0.02, u_off=0.03, v_off=-0.02), **kw})


# name: (orbit, blocks of rows, rows / 64 of a block, voxels a row), scan
_ROWS = {
    "quarter_4": ((4, 1, 4, 3), dict(nx=21, ny=21, nz=230, n_views=88, nu=470)),
    "quarter_5": ((4, 1, 5, 3), dict(nx=20, ny=20, nz=300, n_views=88, nu=470)),
    "quarter_6": ((4, 1, 6, 2), dict(nx=21, ny=21, nz=300, n_views=88, nu=470, step=1.1, nv=420)),
    "half_4": ((2, 1, 4, 3), dict(nx=19, ny=23, nz=230, n_views=90, nu=70)),
    "half_5": ((2, 1, 5, 2), dict(nx=18, ny=24, nz=250, n_views=90, nu=70, step=1.1)),
    "half_6": ((2, 1, 6, 3), dict(nx=18, ny=24, nz=350, n_views=90, nu=70, step=1.0)),
    "one_4": ((1, 1, 4, 3), dict(nx=18, ny=14, nz=230, n_views=7)),
    "one_5": ((1, 1, 5, 2), dict(nx=18, ny=14, nz=260, n_views=7, step=1.1)),
    "one_two_blocks": ((1, 2, 4, 3), dict(nx=18, ny=14, nz=300, n_views=9, nu=70, oz=20.0, nv=1530, step=1.0, v_off=30.0)),
    "half_two_blocks": ((2, 2, 4, 3), dict(nx=18, ny=18, nz=300, n_views=90, nu=70, oz=18.0, nv=1500, step=1.0,
                                          v_off=30.0)),
    "quarter_two_blocks": ((4, 2, 4, 3), dict(nx=17, ny=17, nz=300, n_views=88, nu=470, oz=18.0, nv=1500, step=1.0,
                                             v_off=30.0)),
}


@pytest.mark.parametrize("name", list(_ROWS))
def test_projector_by_rows_blocks(ctx, oracle, name):
    from monte_amd.fdk import fdk_project

    plan, kw = _ROWS[name]
    g = _row_scan(**kw)
    assert routes(g)[8:] == plan
    y = np.random.default_rng(len(name)).standard_normal(g.vol_shape).astype(np.float32)
    ref = oracle.fdk_std_backproject_T(oracle_geom(oracle, g), y)
    got = fdk_project(_t(y), g, ctx).cpu().numpy()
    print(name, rel_max(got, ref), rel_l2(got, ref))
    assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL


@pytest.mark.parametrize("name,chunks", [("half_4", (1, 7, 89)), ("quarter_4", (13, 87)), ("one_two_blocks", (1, 4)),
                                         ("by_voxels", (1, 5, 11))])
def test_projector_in_chunks_of_views(ctx, oracle, name, chunks):
    """Chunks take orbits apart (one view a wave) and have windows of rows of their own."""
    from monte_amd.fdk import fdk_project

    if name == "by_voxels":
        g, orbit = _row_scan(nx=20, ny=18, nz=70, n_views=12, step=0.7), 0
    else:
        g, orbit = _row_scan(**_ROWS[name][1]), 1
    y = np.random.default_rng(5).standard_normal(g.vol_shape).astype(np.float32)
    ref = oracle.fdk_std_backproject_T(oracle_geom(oracle, g), y)
    saved = ctx.tuning
    try:
        for n in chunks:
            assert routes(g, bp_view_chunk=n).pj_orbit == orbit
            ctx.set_tuning(bp_view_chunk=n)
            got = fdk_project(_t(y), g, ctx).cpu().numpy()
            print(name, n, rel_max(got, ref))
            assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL
    finally:
        ctx.set_tuning(**saved)


@pytest.mark.parametrize("views,nx,ny", [(8, 4, 4), (9, 31, 17), (30, 12, 40)])
def test_projector_of_wide_fans(ctx, oracle, views, nx, ny):
    """A volume close to the source's orbit under a detector of 80 degrees either side: strips whose rays
    run along the slabs that the column lists are made of."""
    from monte_amd import geometry as G
    from monte_amd.fdk import fdk_project

    v = 30.0 / max(nx, ny)
    g = G.Geometry(n_views=views, nu=24, nv=13, nx=nx, ny=ny, nz=5, sod=24.0, sdd=33.0, du=17.0, dv=12.5, vx=v, vy=v,
                   vz=2.3)
    y = np.random.default_rng(views).standard_normal(g.vol_shape).astype(np.float32)
    ref = oracle.fdk_std_backproject_T(oracle_geom(oracle, g), y)
    got = fdk_project(_t(y), g, ctx).cpu().numpy()
    print(views, rel_max(got, ref), rel_l2(got, ref))
    assert rel_max(got, ref) < TOL and rel_l2(got, ref) < TOL
