"""The budget's loop over levels, which loads four at a time: columns of fewer levels than that, of whole
groups and of a remainder, whose lowest active level falls anywhere in a group."""
import pytest

import oracle as O
from numericalearth_hip.generators import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("Nz", [1, 3, 4, 5, 11])
def test_budget_matches_the_oracle(require_gpu, Nz, precision):
    from numericalearth_hip.model import OceanOnlyModel
    case = make_case(67, 13, Nz, seed=50 + Nz, n_times=2, sigma_cells=2.0)
    om = O.OracleModel(case).reconcile()
    gm = OceanOnlyModel(case, precision=precision)
    for field in (gm.T, gm.S):
        s, c = om.budget(field.cpu().numpy().astype("float64"), 3.0)
        # both sum in twice the working precision, all terms of one sign: the result's own rounding, 2 ulp
        assert abs(gm.budget(field, 3.0) - (s + c)) <= 4.5e-16 * abs(s + c)
    gm.close()
