"""The FP32 reconstructions of tracers whose neighbouring values differ by 10⁵ and more (units other than °C
and g/kg): the products of their smoothness indicators and the squares of the weights stay in FP32's range."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle as O
from helpers import assert_rel_terms
from numericalearth_hip import _ctypes_abi as abi
from numericalearth_hip.generators import make_case
from numericalearth_hip.model import OceanOnlyModel, stream_handle, torch_view
from test_f32_phases_gpu import RTOL32, _rounded

pytestmark = pytest.mark.gpu


def _noise(shape, rng):
    """Differences up to M: the product of three indicators, at most 8.3³M⁶, stays below 2¹²⁶."""
    return 5.5e5 * rng.random(shape)


def _steps(shape, rng):
    """Steps of D between constant values: a weight's (τ/ε)², with τ = 10/3·D², stays below 2¹²⁸."""
    coarse = rng.integers(0, 2, (-(-shape[0] // 4), -(-shape[1] // 5), -(-shape[2] // 7)))
    return 1e5 + 2.2e5 * np.kron(coarse, np.ones((4, 5, 7)))[:shape[0], :shape[1], :shape[2]]


@pytest.mark.parametrize("field", [_noise, _steps])
def test_f32_tendency_of_large_differences(require_gpu, field):
    case = make_case(60, 32, 8, seed=18)
    gm = OceanOnlyModel(case, precision="mixed")
    om = O.OracleModel(_rounded(case)).reconcile()
    rng = np.random.default_rng(19)
    T, S = (np.ascontiguousarray(field(om.T.shape, rng).astype(np.float32)) for _ in range(2))
    gm.T.copy_(torch.from_numpy(T))
    gm.S.copy_(torch.from_numpy(S))
    for k in O.NET_NAMES:
        gm.net[k].copy_(torch.from_numpy(om.net_arrays[k]))
    GT, GS = torch.zeros_like(gm.T), torch.zeros_like(gm.S)
    print(f"[f32] {field.__name__}", flush=True)
    assert gm.lib.ne_tracer_tendency_weno5_f32(gm.ctx.handle, C.byref(gm.grid.struct), C.byref(gm.params),
                                               C.byref(gm.desc.ocean), C.byref(gm.desc.net), torch_view(GT),
                                               torch_view(GS), stream_handle()) == abi.NE_OK
    torch.cuda.synchronize()
    om.T[...], om.S[...] = T, S
    GT_o, GS_o, sT, sS = om.tendency(scales=True)
    # the bound of the FP32 tendency at ordinary sizes: apart from ε the reconstruction scales with its values
    assert_rel_terms(GT.cpu().numpy(), GT_o, sT, RTOL32, "G_T")
    assert_rel_terms(GS.cpu().numpy(), GS_o, sS, RTOL32, "G_S")
    gm.close()
