"""What a scan's backprojection and projection run (monte_amd/csrc/fdk.hip, fdk_routes): needs no GPU."""
import ctypes as C
from collections import namedtuple

from monte_amd import _lib

Routes = namedtuple("Routes", "orbit groups zc stack tile_x rows cols blocks pj_orbit pj_blocks pj_nr pj_voxels")
DEFAULTS = dict(mc_block=256, mc_batch=64, mc_blocks_per_cu=6, bp_zchunk=16, bp_tile_x=16, bp_tile_y=16,
                bp_view_chunk=0, pj_zchunk=0, mc_ray_brick=4)


def routes(geom, **tuning):
    """orbit: columns a thread owns (0: straight from memory); pj_orbit: views a wave forms (0: by voxels)."""
    f = C.CDLL(_lib.LIB_PATH).monte_internal_fdk_routes
    f.argtypes, f.restype = [C.c_void_p, C.c_void_p, C.c_void_p], C.c_int
    out = (C.c_int32 * len(Routes._fields))()
    g, t = geom.c(), _lib.Tuning(**{**DEFAULTS, **tuning})
    rc = f(C.byref(g), C.byref(t), out)
    assert rc == 0, rc
    return Routes(*out)
