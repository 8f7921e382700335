"""How the tracer stages cut a grid's tiles, for devices (whole chips and partitions of them) of several
numbers of compute units: the tiles that are cut are those left over from full rounds of that device, and
the workspace, which is sized before the device is known, has a slot for every block of any of them."""
import ctypes as C

import pytest

from numericalearth_hip import _ctypes_abi as abi
from numericalearth_hip import _lib
from numericalearth_hip._lib import check

GRIDS = [(1, 1, 1), (1, 1, 50), (90, 40, 10), (353, 137, 19), (640, 410, 4), (640, 410, 1), (690, 416, 15),
         (720, 280, 10), (1440, 560, 10), (1440, 560, 1023), (4320, 1800, 33)]


def _chunks(Nz, levels):
    return -(-Nz // levels)


def _plan(Nx, Ny, Nz, waves, cus):
    out = (C.c_int32 * 4)()
    check(_lib.load().ne_stage_plan(Nx, Ny, Nz, waves, cus, out), "ne_stage_plan")
    return list(out)


def _residual_slots(Nx, Ny, Nz):
    """Slots of the workspace: what a mixed model's has beyond its other parts, all multiples of 256 bytes."""
    d = abi.ModelDesc()
    buf = C.create_string_buffer(8)   # the pointers are tested for null only
    for name, kind in abi.Grid._fields_:
        if kind is C.c_void_p:
            setattr(d.grid, name, C.addressof(buf))
    d.grid.Nx, d.grid.Ny, d.grid.Nz = Nx, Ny, Nz
    d.grid.topology_x = d.grid.topology_y = abi.NE_BOUNDED
    d.ocean.T = abi.View(C.addressof(buf), 1, Nx, Nx * Ny)
    d.precision = abi.NE_MIXED_FP32
    n = C.c_int64()
    check(_lib.load().ne_model_workspace_bytes(C.byref(d), C.byref(n)), "ne_model_workspace_bytes")
    up = lambda b: (b + 255) // 256 * 256
    return (n.value - 4 * up(4 * Nx * Ny * Nz) - up(Nx * Ny) - up(4 * (1 + Nx * Ny)) - up(16 * (Nz + 1))) // 32


@pytest.mark.parametrize("cus", [32, 64, 128, 256, 304])
def test_tiles_left_over_from_the_devices_rounds_are_cut(cus):
    for Nx, Ny, Nz in GRIDS:
        tiles = -(-Nx // 63) * -(-Ny // 4)
        for waves in (4, 5, 6, 7):
            n, first, levels, rest_levels = _plan(Nx, Ny, Nz, waves, cus)
            places, where = waves * cus, (Nx, Ny, Nz, waves, cus)
            assert n == tiles and 1 <= levels <= Nz and 1 <= rest_levels <= Nz, where
            rest = tiles - first
            blocks = first * _chunks(Nz, levels) + rest * _chunks(Nz, rest_levels)
            if tiles < places:
                # about 6 blocks for each compute unit: the chunks' number is rounded up to whole levels
                assert rest == 0 and blocks < 6 * min(cus, 256) + tiles, where
            else:
                left_over = tiles % places
                assert levels == Nz and rest in (0, left_over), where
                # cut when at least two chunks each have a place in the last round, and only then
                assert (rest > 0) == (0 < 2 * left_over <= places and Nz > 1), where
                assert rest * _chunks(Nz, rest_levels) <= places, where
            assert blocks <= _residual_slots(Nx, Ny, Nz), where


def test_plan_refuses_what_is_no_grid_or_device():
    out = (C.c_int32 * 4)()
    plan = _lib.load().ne_stage_plan
    assert plan(1, 1, 1, 4, 256, None) == abi.NE_ERR_NULL
    for bad in ((0, 1, 1, 4, 256), (1, 0, 1, 4, 256), (1, 1, 0, 4, 256), (1, 1, 1024, 4, 256), (1, 1, 1, 0, 256),
                (1, 1, 1, 4, 0)):
        assert plan(*bad, out) == abi.NE_ERR_SHAPE, bad
