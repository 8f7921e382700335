"""The flux solve's table of the stability functions on the GPU, by its users: parameters of every
flux path over air–sea differences and winds that put ζ on both sides of zero, in the table, at its
edges and beyond them, against the oracle's closed forms; and the solver counters, which the kernels
keep in many copies."""
import numpy as np
import pytest
import torch

import oracle as O
from numericalearth_hip import _ctypes_abi as abi
from numericalearth_hip.generators import make_case
from numericalearth_hip.model import OceanOnlyModel
from numericalearth_hip.params import FixedIterations, SimilarityTheoryFluxes, to_params
from test_gpu_parity import RTOL, _compare_fluxes

pytestmark = pytest.mark.gpu


def _case(largest_difference, calmest):
    case = make_case(70, 37, 2, seed=31)
    rng = np.random.default_rng(32)
    shape = case.atmos["T"].shape
    wind = np.exp(rng.uniform(np.log(calmest), np.log(60.0), shape))
    angle = rng.uniform(0.0, 2.0 * np.pi, shape)
    case.atmos["u"][...], case.atmos["v"][...] = wind * np.cos(angle), wind * np.sin(angle)
    case.atmos["T"][...] += rng.uniform(-1.0, 1.0, shape) ** 3 * largest_difference   # many near neutral
    case.atmos["q"][...] *= rng.uniform(0.3, 1.2, shape)
    return case


def _params(path):
    if path == "default constants":
        return to_params()
    p = to_params(SimilarityTheoryFluxes(solver_stop_criteria=FixedIterations(4)))   # four iterates: no stop test
    if path == "positive constants":
        p.charnock_parameter, p.reynolds_scaling_A = 0.014, 6.5e-5
    else:   # a constant scalar roughness length: the quotient form
        p.temperature_roughness = p.water_vapor_roughness = abi.NE_ROUGHNESS_CONSTANT
        p.temperature_roughness_length = p.water_vapor_roughness_length = 1e-4
    return p


# The bound of the flux rows, 1e-12 relative, is 4500 ulp: an iterate's few ulp times the iteration's
# sensitivity (about ten in the strongly unstable and stable columns here).
@pytest.mark.parametrize("path,difference,calmest", [("default constants", 20.0, 0.5), ("positive constants", 40.0, 1e-3),
                                                     ("quotient form", 40.0, 1e-3)])
def test_flux_paths_match_the_closed_forms(require_gpu, path, difference, calmest):
    case = _case(difference, calmest)
    p = _params(path)
    om = O.OracleModel(case, params=abi.Params.from_buffer_copy(p)).reconcile()
    gm = OceanOnlyModel(case, params=abi.Params.from_buffer_copy(p))
    torch.cuda.synchronize()
    print(f"[table] {path}", flush=True)
    _compare_fluxes(gm, om, RTOL)
    gm.close()


def test_counters_sum_over_their_copies(require_gpu):
    case = make_case(130, 70, 3, seed=33)
    gm = OceanOnlyModel(case)
    gm.ctx.counters(reset=True)
    for _ in range(3):
        gm.update_state()
    got = gm.ctx.counters(reset=True)
    wet = int(np.sum(case.grid.kmin < 3))
    it = gm.iterations.cpu().numpy()[case.grid.kmin < 3]
    assert got["solved_columns"] == 3 * wet and got["max_iterations"] == it.max()
    assert got["total_iterations"] == 3 * int(it.sum())
    assert got["nonconverged_columns"] == 0 and got["nan_columns"] == 0
    assert all(v == 0 for v in gm.ctx.counters().values())
    gm.close()
