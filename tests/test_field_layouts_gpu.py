"""Fields of one layout, which the surface kernels address with shared 32-bit offsets, against fields of
layouts of their own: the same step, bit for bit, for every flux path and both storage types, with an
output and a source field moved to a padded row stride and a strided (every second value) layout."""
import copy
import ctypes as C

import pytest
import torch

from numericalearth_hip import _ctypes_abi as abi
from numericalearth_hip._lib import check
from numericalearth_hip.generators import make_case
from numericalearth_hip.model import OceanOnlyModel, stream_handle, torch_view
from numericalearth_hip.params import CoefficientBasedFluxes, LargeYeagerTransferCoefficients, to_params

pytestmark = pytest.mark.gpu


def _params(path):
    p = to_params(CoefficientBasedFluxes(LargeYeagerTransferCoefficients()) if path == "coefficients" else None)
    if path == "positive":
        p.charnock_parameter = 0.015
    if path == "general":
        p.similarity_form = abi.NE_SIMILARITY_COARE_LOG
    return p


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("path", ["default", "positive", "coefficients", "general"])
def test_layouts_give_the_same_bits(require_gpu, path, precision):
    case = make_case(67, 21, 4, seed=41, n_times=2)
    unit = OceanOnlyModel(copy.deepcopy(case), params=_params(path), precision=precision)
    own = OceanOnlyModel(copy.deepcopy(case), params=_params(path), precision=precision)
    check(own.lib.ne_model_destroy(own.handle), "ne_model_destroy")
    own.handle = None
    d = own.desc
    Ny, Nx = own.fluxes["latent_heat"].shape
    padded = torch.zeros((Ny, Nx + 5), dtype=torch.float64, device=own.device)[:, :Nx]
    strided = torch.zeros((Ny, 2 * Nx), dtype=torch.float64, device=own.device)[:, ::2]
    own.fluxes["latent_heat"], own.net["J_H"] = padded, strided
    d.fluxes.latent_heat, d.net.J_H = torch_view(padded), torch_view(strided)
    v = own.atm["v"]
    moved = torch.zeros((*v.shape[:2], v.shape[2] + 3), dtype=v.dtype, device=v.device)[:, :, :v.shape[2]]
    moved.copy_(v)
    own.atm["v"] = moved
    d.atmosphere.v = torch_view(moved)
    own.T.copy_(torch.from_numpy(case.T))
    h = C.c_void_p()
    check(own.lib.ne_model_create(own.ctx.handle, C.byref(d), C.byref(h), stream_handle()), "ne_model_create")
    own.handle = h
    for _ in range(2):
        unit.time_step(1200.0)
        own.time_step(1200.0)
    torch.cuda.synchronize()
    for name, a, b in [("T", unit.T, own.T), ("S", unit.S, own.S), ("iterations", unit.iterations, own.iterations),
                       *((k, unit.fluxes[k], own.fluxes[k]) for k in unit.fluxes),
                       *((k, unit.net[k], own.net[k]) for k in unit.net),
                       *((k, unit.radiative[k], own.radiative[k]) for k in unit.radiative)]:
        # the logarithmic profile of the general path has no solution in some columns: NaN on both sides
        assert torch.equal(torch.isnan(a), torch.isnan(b)), (path, precision, name)
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)), (path, precision, name)
    unit.close()
    own.close()


def _padded(t, extra):
    out = torch.zeros((*t.shape[:-1], t.shape[-1] + extra), dtype=t.dtype, device=t.device)[..., :t.shape[-1]]
    out.copy_(t)
    return out


def _quotient_params():
    """The default stability functions with a constant scalar roughness length: the quotient form."""
    p = to_params()
    p.temperature_roughness = p.water_vapor_roughness = abi.NE_ROUGHNESS_CONSTANT
    p.temperature_roughness_length = p.water_vapor_roughness_length = 1e-4
    return p


def _rebuilt(m, moved=None, precipitation=True):
    """The model `m` with the fields that `moved` names in padded layouts, and without rain and snow if asked."""
    check(m.lib.ne_model_destroy(m.handle), "ne_model_destroy")
    m.handle, d = None, m.desc
    if moved == "radiation":
        m.rad["downwelling_longwave"] = _padded(m.rad["downwelling_longwave"], 3)
        d.radiation.downwelling_longwave = torch_view(m.rad["downwelling_longwave"])
    elif moved == "iterations":
        m.iterations = _padded(m.iterations, 5)
        d.fluxes.iterations = torch_view(m.iterations)
    elif moved == "state":   # its views have row strides of their own in the shared-offset kernels too
        m.T, m.S, m.u = _padded(m.T, 3), _padded(m.S, 3), _padded(m.u, 7)
        d.ocean.T, d.ocean.S, d.ocean.u = torch_view(m.T), torch_view(m.S), torch_view(m.u)
        d.workspace, d.workspace_bytes = None, 0   # the model's own stage buffers, of T's layout
    elif moved == "output":
        m.fluxes["latent_heat"] = _padded(m.fluxes["latent_heat"], 5)
        d.fluxes.latent_heat = torch_view(m.fluxes["latent_heat"])
    if not precipitation:
        d.atmosphere.rain = d.atmosphere.snow = abi.View(None, 0, 0, 0)
    m.T.copy_(torch.from_numpy(m.case.T))
    m.S.copy_(torch.from_numpy(m.case.S))
    h = C.c_void_p()
    check(m.lib.ne_model_create(m.ctx.handle, C.byref(d), C.byref(h), stream_handle()), "ne_model_create")
    m.handle = h
    return m


def _assert_same_bits(a, b, what):
    torch.cuda.synchronize()
    for name, x, y in [("T", a.T, b.T), ("S", a.S, b.S), ("iterations", a.iterations, b.iterations),
                       *((k, a.fluxes[k], b.fluxes[k]) for k in a.fluxes),
                       *((k, a.net[k], b.net[k]) for k in a.net),
                       *((k, a.radiative[k], b.radiative[k]) for k in a.radiative)]:
        assert torch.equal(x, y), (what, name)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("moved,precipitation", [("radiation", True), ("iterations", True), ("state", True),
                                                 ("output", False)])
def test_other_layouts_of_the_quotient_form_give_the_same_bits(require_gpu, moved, precipitation, precision):
    case = make_case(67, 21, 4, seed=42, n_times=2)
    unit = OceanOnlyModel(copy.deepcopy(case), params=_quotient_params(), precision=precision)
    if not precipitation:
        unit = _rebuilt(unit, precipitation=False)
    own = _rebuilt(OceanOnlyModel(copy.deepcopy(case), params=_quotient_params(), precision=precision), moved,
                   precipitation)
    for _ in range(2):
        unit.time_step(1200.0)
        own.time_step(1200.0)
    _assert_same_bits(unit, own, (moved, precision))
    unit.close()
    own.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_ensemble_with_a_member_of_another_layout(require_gpu, precision):
    """One member's own layout takes the whole ensemble to the kernels with each view's strides."""
    from numericalearth_hip.ensemble import Ensemble
    shapes, paths = [(67, 21, 4), (33, 12, 5), (20, 9, 3)], ("default", "positive", "coefficients")

    def members():
        return [OceanOnlyModel(make_case(*s, seed=43 + k, n_times=2), params=_params(path), precision=precision)
                for k, (s, path) in enumerate(zip(shapes, paths))]

    alone, batched = members(), members()
    _rebuilt(batched[1], "output")
    ens = Ensemble(batched)
    for _ in range(2):
        ens.time_step(1200.0)
        for m in alone:
            m.time_step(1200.0)
    for k, (a, b) in enumerate(zip(alone, batched)):
        _assert_same_bits(a, b, (precision, k))
    ens.close()
    for m in alone + batched:
        m.close()
