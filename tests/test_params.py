"""CPU tests of the parameters that a call packs: the values that pf_args holds at the time of the call, in any form."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from pfkit import _lib
from pfkit.allen_cahn import StateRHS
from pfkit.config import make_params
from problems import args, gaussian, quench, rosenthal

FIELDS = ("m_g", "gamma", "kappa_g", "ad_hoc", "L0", "Qg", "gas_const", "T_liquidus", "T_clip", "zeta_sharpness",
          "anisotropy", "liquid_shift")


def _rhs(a):
    pc = SimpleNamespace(mesh_h_xyz=(1.0, 1.0, 1.0), unique_grain_directions=np.zeros((3, 4, 3)))
    return StateRHS(pc, a, dtype=torch.float64, device="cpu")


@pytest.mark.parametrize("name", FIELDS)
@pytest.mark.parametrize("make", [lambda v: np.array(v), lambda v: torch.tensor(v, dtype=torch.float64)],
                         ids=["array", "tensor"])
def test_a_value_changed_in_place_takes_effect(name, make):
    v = make(1.5)
    rhs = _rhs(args(8, 6, 4, 4, **{name: v}))
    for T in (gaussian(8, 6, 4), torch.full((8 * 6 * 4, 1), 900.0)):
        before = getattr(rhs.params_for(T)[0], name)
        v *= 2
        assert getattr(rhs.params_for(T)[0], name) == 2 * before == float(v)


def test_a_cell_size_changed_in_place_takes_effect():
    h = np.ones(3)
    rhs = _rhs(args(8, 6, 4, 4))
    rhs.h_xyz = h
    assert list(rhs.params_for(gaussian(8, 6, 4))[0].h) == [1.0, 1.0, 1.0]
    h[1] = 0.5
    assert list(rhs.params_for(gaussian(8, 6, 4))[0].h) == [1.0, 0.5, 1.0]


def test_values_without_the_defaults():
    """A parameter dict put in later needs no more keys than one that a solver is made with."""
    rhs = _rhs(args(8, 6, 4, 4))
    rhs.pf_args = {k: v for k, v in args(8, 6, 4, 4).items() if k not in ("gamma", "T_clip", "zeta_sharpness", "force_liquid",
                                                                          "liquid_shift", "anisotropy", "ad_hoc")}
    p = rhs.params_for(gaussian(8, 6, 4))[0]
    assert (p.gamma, p.T_clip, p.zeta_sharpness, p.force_liquid, p.liquid_shift, p.anisotropy, p.ad_hoc) == (
        1.0, 2000.0, 1e10, 0, 1.0, 0.0, 1.0)
    with pytest.raises(KeyError):
        make_params(dict(Nx=8, Ny=6, Nz=4), (1.0, 1.0, 1.0))


@pytest.mark.parametrize("make", [gaussian, rosenthal, lambda nx, ny, nz: quench(nz)], ids=["gaussian", "rosenthal", "quench"])
def test_every_field_as_its_own_assignment(make):
    """The packed struct against one assignment per field, for every type that a yaml file or a program gives."""
    a = args(7, 5, 3, 9, force_liquid=True, T_liquidus="1623.5", m_g=np.float32(1.1), L0=3500, gamma=torch.tensor(0.75))
    L = make(7, 5, 3)
    p = make_params(a, np.array([0.5, 1.5, 2.5]), L)
    q = _lib.ParamsT()
    q.nz, q.ny, q.nx, q.num_oris, q.force_liquid = 3, 5, 7, 9, 1
    for d, v in enumerate((0.5, 1.5, 2.5)):
        q.h[d] = v
    for name in FIELDS:
        setattr(q, name, float(a[name]))
    q.laser.model = {"gaussian": _lib.PF_T_GAUSSIAN, "rosenthal": _lib.PF_T_ROSENTHAL, "quench": _lib.PF_T_QUENCH}[
        L.as_dict()["model"]]
    for name, v in L.as_dict().items():
        if name in ("pos0", "dir"):
            for d in range(3):
                getattr(q.laser, name)[d] = v[d]
        elif name != "model":
            setattr(q.laser, name, v)
    assert bytes(p) == bytes(q)
    q = _lib.ParamsT()
    q.laser.model, q.laser.T_dtype = _lib.PF_T_BUFFER, _lib.PF_F64
    assert bytes(make_params(a, (1.0, 1.0, 1.0)))[-_lib.ParamsT.laser.size:] == bytes(q.laser)


@pytest.mark.parametrize("make,name", [(gaussian, "sigma_z"), (rosenthal, "Q"), (rosenthal, "vel"), (lambda nx, ny, nz: quench(nz), "T_ref")])
@pytest.mark.parametrize("value", [None, "300", 1j])
def test_a_source_parameter_that_is_no_number_is_a_type_error(make, name, value):
    L = make(7, 5, 3)
    setattr(L, name, value)
    with pytest.raises(TypeError):
        make_params(args(7, 5, 3, 9), (1.0, 1.0, 1.0), L)
