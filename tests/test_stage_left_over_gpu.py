"""Tracer stages whose tiles left over from full rounds of the chip are cut into chunks of levels: both time
steppers and the two-colour forcing against the oracle's step, and the mixed form also by its heat budget,
whose rounding residual has a slot for every chunk."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from helpers import assert_rel
from numericalearth_hip._lib import check, load
from numericalearth_hip.generators import NE_PERIODIC, make_case
from numericalearth_hip.model import OceanOnlyModel
from numericalearth_hip.params import TwoColorRadiation, to_params

pytestmark = pytest.mark.gpu
DT = 1200.0


def _left_over(Nx, Ny, Nz, waves):
    """Tiles that a launch of an instance with `waves` blocks on each compute unit of this device cuts."""
    out = (C.c_int32 * 4)()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    check(load().ne_stage_plan(Nx, Ny, Nz, waves, cus, out), "ne_stage_plan")
    return out[0] - out[1]


def _case(Nx, Ny, Nz):
    return make_case(Nx, Ny, Nz, seed=13, topology_x=NE_PERIODIC, longitude=(0.0, 360.0), sigma_cells=6.0, n_times=2)


def _params(two_color):
    return to_params(radiative_forcing=TwoColorRadiation() if two_color else None)


# 1133 tiles, 109 left over from the FP64 instances' 1024 places (4 blocks on each of 256 compute units)
@pytest.mark.parametrize("two_color,stepper", [(True, "SplitRungeKutta3"), (False, "QuasiAdamsBashforth2"),
                                               (True, "QuasiAdamsBashforth2")])
def test_left_over_tiles_match_the_oracle(require_gpu, two_color, stepper):
    shape = (640, 410, 4)
    assert _left_over(*shape, 4) > 0
    case = _case(*shape)
    om = O.OracleModel(case, params=_params(two_color), timestepper=stepper).reconcile()
    gm = OceanOnlyModel(case, params=_params(two_color), timestepper=stepper)
    for _ in range(2):
        om.time_step(DT)
        gm.time_step(DT)
    assert_rel(gm.T.cpu().numpy(), om.T, 1e-12, "T")   # the parity bound of the step
    assert_rel(gm.S.cpu().numpy(), om.S, 1e-12, "S")
    gm.close()


# 1380 tiles: the two-colour instances have 5·256 places, 100 are left over in all three stages;
# 1625 tiles: the last stage has 6·256, 89 are left over, the other stages 7·256 and cut every tile
@pytest.mark.parametrize("shape,waves,two_color", [((700, 460, 6), 5, True), ((770, 500, 6), 6, False)])
def test_left_over_tiles_of_the_mixed_form(require_gpu, shape, waves, two_color):
    assert _left_over(*shape, waves) > 0
    case = _case(*shape)
    om = O.OracleModel(case, params=_params(two_color)).reconcile()
    gm = OceanOnlyModel(case, params=_params(two_color), precision="mixed")
    rho_c = gm.params.ocean_reference_density * gm.params.ocean_heat_capacity
    active = np.arange(shape[2])[:, None, None] >= case.grid.kmin[None]
    Az = case.grid.Az[:, None]
    V = Az[None] * case.grid.dz[:, None, None]
    C0, expected, bound = gm.conserved_heat(), 0.0, 0.0
    for _ in range(2):
        wet = case.grid.kmin < shape[2]
        J = gm.net["J_T"].cpu().numpy() - (gm.shortwave_surface_flux.cpu().numpy() if two_color else 0.0)
        expected -= DT * rho_c * float(np.sum(np.where(wet, J * Az, 0.0)))
        om.time_step(DT)
        gm.time_step(DT)
        torch.cuda.synchronize()
        # half an FP64 ulp of T per cell from the update, and as much from the shortwave's terms
        bound += 2.0 * rho_c * float(np.sum(np.where(active, V * np.spacing(np.abs(om.T)), 0.0)))
    # a chunk left out, or taken twice, is off by a stage's change of T, about 0.1 K; the FP32 tendency is
    # within 1e-5 of its terms
    for name, got, ref in (("T", gm.T, om.T), ("S", gm.S, om.S)):
        d = np.abs(got.cpu().numpy() - ref)[active]
        print(f"[left over] {name}: {d.max():.2e}", flush=True)
        assert d.max() <= 1e-5 * np.abs(ref).max(), name
    miss = abs(gm.conserved_heat() - C0 - expected)
    print(f"[left over] heat misses by {miss:.3e}, bound {bound:.3e}, change {expected:.3e}", flush=True)
    assert miss <= bound
    gm.close()
