"""The flux solve at the limits of the parameters that its logarithmic iteration takes, and beyond them,
against the oracle's closed forms."""
import numpy as np
import pytest
import torch

import oracle as O
from numericalearth_hip import _ctypes_abi as abi
from numericalearth_hip.model import OceanOnlyModel
from numericalearth_hip.params import FixedIterations, SimilarityTheoryFluxes, to_params
from test_flux_table_gpu import _case
from test_gpu_parity import RTOL, _compare_fluxes

pytestmark = pytest.mark.gpu

# The gustiness β∛(−u★b★h) depends on β³h alone: the first set is the default one with β and h of other
# sizes, whose arguments of the cube root lie below 1e-30. The others are the ranges' two ends.
SETS = {
    "gustiness of other sizes": dict(gustiness_parameter=1.2e10, boundary_layer_height=512e-30),
    "small": dict(minimum_gustiness=1e-4, gustiness_parameter=1e-3, roughness_gravitational_acceleration=1e3,
                  air_kinematic_viscosity=1e-7, charnock_parameter=1e-4, smooth_wall_parameter=1e-2,
                  maximum_momentum_roughness=1e-3, reynolds_scaling_A=1e-8, reynolds_scaling_b=-4.0,
                  maximum_scalar_roughness=1e-6),
    "large": dict(minimum_gustiness=1.0, gustiness_parameter=1e2, boundary_layer_height=1e5,
                  roughness_gravitational_acceleration=1.0, air_kinematic_viscosity=1e-3, charnock_parameter=1.0,
                  smooth_wall_parameter=10.0, reynolds_scaling_A=1e-2, reynolds_scaling_b=4.0,
                  maximum_scalar_roughness=0.1),
}


# Four iterates, no stop test. The 1e-12 bound of the flux rows is 4500 ulp; here an iterate's errors are
# a few ulp of logarithms up to 40, and a nudge of one constant grows by at most 60 over the four.
@pytest.mark.parametrize("name", SETS)
def test_flux_solve_at_the_ranges_of_its_parameters(require_gpu, name):
    case = _case(20.0, 1e-3)
    calm = np.random.default_rng(34).uniform(size=case.atmos["u"].shape) < 0.4
    case.atmos["u"][calm] = case.atmos["v"][calm] = 0.0
    p = to_params(SimilarityTheoryFluxes(solver_stop_criteria=FixedIterations(4)))
    for key, value in SETS[name].items():
        setattr(p, key, value)
    om = O.OracleModel(case, params=abi.Params.from_buffer_copy(p)).reconcile()
    gm = OceanOnlyModel(case, params=abi.Params.from_buffer_copy(p))
    torch.cuda.synchronize()
    print(f"[ranges] {name}", flush=True)
    _compare_fluxes(gm, om, RTOL)
    gm.close()
