"""Tracer stages whose columns are cut into chunks of levels: grids of few tiles, with chunks of one
level, of several, and a shorter last one, against the oracle's step (which knows no chunks)."""
import pytest

import oracle as O
from helpers import assert_rel
from numericalearth_hip.generators import NE_BOUNDED, NE_PERIODIC, make_case

pytestmark = pytest.mark.gpu

# tiles × levels against the 1536 blocks that a launch aims at: 6 × 23 → chunks of 1 level;
# 48 × 61 → 31 chunks of 2, the last one of 1; 69 × 50 → 17 chunks of 3, the last one of 2
SHAPES = [(70, 9, 23, NE_PERIODIC), (130, 64, 61, NE_BOUNDED), (127, 92, 50, NE_PERIODIC)]


@pytest.mark.parametrize("Nx,Ny,Nz,topology_x", SHAPES)
@pytest.mark.parametrize("stepper", ["SplitRungeKutta3", "QuasiAdamsBashforth2"])
def test_chunked_stages_match_the_oracle(require_gpu, Nx, Ny, Nz, topology_x, stepper):
    from numericalearth_hip.model import OceanOnlyModel
    lon = (0.0, 360.0) if topology_x == NE_PERIODIC else (10.0, 10.0 + 0.25 * Nx)
    case = make_case(Nx, Ny, Nz, seed=11, topology_x=topology_x, longitude=lon, sigma_cells=3.0)
    om = O.OracleModel(case, timestepper=stepper).reconcile()
    gm = OceanOnlyModel(case, timestepper=stepper)
    for _ in range(2):
        om.time_step(1200.0)
        gm.time_step(1200.0)
    # one step's FP64 round-off is a few ulp of the state; the parity bound of the step is 1e-12
    assert_rel(gm.T.cpu().numpy(), om.T, 1e-12, "T")
    assert_rel(gm.S.cpu().numpy(), om.S, 1e-12, "S")
    gm.close()


# 1133 and 1144 tiles of 63×4 cells: more than the 1024 blocks the chip holds, so that the last 109 (120)
# tiles alone are cut, into chunks of one level, and of two with a last one of one
@pytest.mark.parametrize("Nx,Ny,Nz", [(640, 410, 4), (690, 416, 15)])
def test_stages_of_more_tiles_than_places_match_the_oracle(require_gpu, Nx, Ny, Nz):
    from numericalearth_hip.model import OceanOnlyModel
    case = make_case(Nx, Ny, Nz, seed=12, topology_x=NE_PERIODIC, longitude=(0.0, 360.0), sigma_cells=6.0, n_times=2)
    om = O.OracleModel(case).reconcile()
    gm = OceanOnlyModel(case)
    om.time_step(1200.0)
    gm.time_step(1200.0)
    assert_rel(gm.T.cpu().numpy(), om.T, 1e-12, "T")
    assert_rel(gm.S.cpu().numpy(), om.S, 1e-12, "S")
    gm.close()
