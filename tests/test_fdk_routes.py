"""The rules that choose the FDK's kernels, without a GPU: a tile's patch holds every tap of its
voxels, whatever the scan and the tuning."""
import math

import numpy as np
import pytest

from fdk_routes import routes
from monte_amd import geometry as G

PAD_LO, PAD_HI = 1, 3
LDS_WORDS = {1: (64, 80), 2: (64, 144), 4: (32, 144)}  # columns of a patch, words of a row


def _draw(rng):
    """A scan: fine to coarse voxels, full and partial turns, offsets, all shapes."""
    n = lambda a, b: int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))  # noqa: E731
    nx = n(8, 600)
    ny = nx if rng.random() < 0.6 else n(1, 600)
    nz, V = n(1, 900), n(4, 720)
    if rng.random() < 0.6:
        V = max(4, V // 4 * 4)
    sod = rng.uniform(20, 80)
    sdd = sod * rng.uniform(1.2, 3)
    half = sod * rng.uniform(0.02, 0.98)
    vx = half * math.sqrt(2) / max(nx, ny)
    kw = dict(n_views=V, nu=n(1, 1024), nv=n(1, 1536), nx=nx, ny=ny, nz=nz, sod=sod, sdd=sdd, vx=vx,
              vy=vx if rng.random() < 0.7 else vx * rng.uniform(0.3, 1), vz=vx * math.exp(rng.uniform(-2, 1)))
    mag = sdd / sod
    kw["du"], kw["dv"] = vx * mag / math.exp(rng.uniform(-2, 1.5)), kw["vz"] * mag / math.exp(rng.uniform(-2, 2))
    if rng.random() < 0.3:
        kw.update(ox=vx * rng.uniform(-3, 3), oy=vx * rng.uniform(-3, 3))
    if rng.random() < 0.5:
        kw.update(oz=kw["vz"] * rng.uniform(-30, 30), u_off=kw["du"] * rng.uniform(-9, 9), v_off=kw["dv"] * rng.uniform(-9, 9))
    if rng.random() < 0.2:
        kw["dangle"] = rng.uniform(-0.2, 0.2)
    elif rng.random() < 0.3:
        kw["dangle"] = -2 * math.pi / V
    g = G.Geometry(**kw)
    if math.hypot(0.5 * g.nx * g.vx + abs(g.ox), 0.5 * g.ny * g.vy + abs(g.oy)) >= sod:
        return _draw(rng)  # (refused: it reaches the source's orbit)
    return g


def _taps_stay_inside(g, r, rng, tiles=64):
    nx = (g.nx + 1) // 2 if r.orbit == 4 else g.nx
    ny = (g.ny + 1) // 2 if r.orbit > 1 else g.ny
    tile_y, depth = 256 // (r.tile_x * r.stack), r.zc * r.stack
    tx = rng.integers(0, -(-nx // r.tile_x), tiles) * r.tile_x
    ty = rng.integers(0, -(-ny // tile_y), tiles) * tile_y
    tz = rng.integers(0, -(-g.nz // depth), tiles) * depth
    k = rng.integers(0, g.n_views, tiles)
    x1, y1 = np.minimum(tx + r.tile_x, nx) - 1, np.minimum(ty + tile_y, ny) - 1
    c = g.c()
    b = g.angle0 + k * c.dangle

    def sample(x, y, z):
        X, Y = g.ox - 0.5 * (g.nx - 1) * g.vx + x * g.vx, g.oy - 0.5 * (g.ny - 1) * g.vy + y * g.vy
        Z = g.oz - 0.5 * (g.nz - 1) * g.vz + z * g.vz
        U = X * np.cos(b) + Y * np.sin(b) + g.sod
        su = 0.5 * g.nu - g.u_off / g.du - 0.5 + g.sdd / g.du * (-X * np.sin(b) + Y * np.cos(b)) / U
        sv = 0.5 * g.nv - g.v_off / g.dv - 0.5 + g.sdd / g.dv * Z / U
        return np.clip(su, -1, g.nu), np.clip(sv, -1, g.nv)

    corners = [sample(x, y, z) for x in (tx, x1) for y in (ty, y1) for z in (tz, tz + depth - 1)]
    c0 = np.maximum(np.floor(np.min([s[0] for s in corners], axis=0) - 0.01) + PAD_LO, 0)
    r0 = np.maximum(np.floor(np.min([s[1] for s in corners], axis=0) - 0.01) + PAD_LO, 0)
    for s in corners + [sample(rng.integers(tx, x1 + 1), rng.integers(ty, y1 + 1), tz + rng.integers(0, depth, tiles))
                        for _ in range(20)]:
        col, row = np.floor(s[0]) + PAD_LO - c0, np.floor(s[1]) + PAD_LO - r0
        assert (col >= 0).all() and (col + 1 < r.cols).all(), (g, r)
        assert (row >= 0).all() and (row + 1 < r.rows).all(), (g, r)


@pytest.mark.parametrize("seed", range(8))
def test_patches_hold_every_tap(seed):
    rng = np.random.default_rng(seed)
    seen = set()
    for _ in range(120):
        g = _draw(rng)
        tuning = {}
        if rng.random() < 0.5:
            tuning = dict(bp_zchunk=int(rng.choice([4, 8, 16])), bp_tile_x=int(rng.choice([1, 8, 16, 32, 64, 256])))
        if rng.random() < 0.3:
            tuning["bp_view_chunk"] = int(rng.integers(1, g.n_views + 1))
        r = routes(g, **tuning)
        seen.add((r.orbit, r.stack))
        assert r.orbit in (0, 1, 2, 4)
        if r.orbit == 0:
            continue
        cols, words = LDS_WORDS[r.orbit]
        assert r.cols <= cols and 8 * r.rows * words * r.groups <= 156 * 1024
        assert r.zc in (4, 8, 16, 32) and r.groups in (1, 2, 4) and r.tile_x in (8, 16, 32)
        assert r.orbit == 1 or tuning.get("bp_view_chunk", g.n_views) >= g.n_views  # an orbit needs the whole turn
        _taps_stay_inside(g, r, rng)
    assert len(seen) >= 4
