"""Parameter handling: the reference's yaml dict, plus the constants it hard-codes.

The reference loads ``pf_params.yaml`` into a plain dict (jax_am/common.py:24-31) and
mutates it at run time (Nx/Ny/Nz from the mesh, utils.py:47-49; data_dir from the
app).  This module keeps that dict as the interface and fills in, under explicit
keys, what the reference hard-codes:

=================  =======  =========================================
key                default  reference
=================  =======  =========================================
gamma              1.0      allen_cahn.py:43 ``gamma = 1``
T_clip             2000.0   allen_cahn.py:56
zeta_sharpness     1e10     allen_cahn.py:57
force_liquid       False    allen_cahn.py:142 (call commented out)
liquid_shift       1.0      allen_cahn.py:124
anisotropy         0.0      pf_params.yaml
=================  =======  =========================================
"""
import math
import struct
from operator import itemgetter

import yaml

from . import _lib

HARD_CODED = dict(gamma=1.0, T_clip=2000.0, zeta_sharpness=1e10, force_liquid=False, liquid_shift=1.0)


def yaml_parse(path):
    """Load a reference pf_params.yaml into a dict (jax_am/common.py:24-31; SafeLoader here)."""
    with open(path) as f:
        args = yaml.load(f, Loader=yaml.SafeLoader)
    return args


def with_defaults(pf_args):
    """Copy of pf_args with the hard-coded constants filled in where absent."""
    out = dict(HARD_CODED)
    out.setdefault("anisotropy", 0.0)
    out.setdefault("ad_hoc", 1.0)
    out.update(pf_args)
    return out


def mobility(T, pf_args):
    """Arrhenius mobility L0 exp(-Qg / (R T)) at T clipped to T_clip (allen_cahn.py:56,83)."""
    a = with_defaults(pf_args)
    T = min(T, a["T_clip"])
    return a["L0"] * math.exp(-a["Qg"] / (T * a["gas_const"]))


def stable_dt(pf_args, h_xyz, fraction=0.2, c_local=None):
    """Explicit-Euler step at `fraction` of the linear stability limit.

    dt_max = 2 / (L_max (4 kappa_max sum_d 1/h_d^2 + m_g c)), with L_max the mobility at
    T_clip, kappa_max = kappa_g ad_hoc (1 + anisotropy), and c a bound on the diagonal
    of the local-term Jacobian: 4 for a just-melted one-hot cell plus 4*gamma for the
    cross terms (c_local overrides).  Returns (dt, dt_max, c).
    """
    a = with_defaults(pf_args)
    c = 4.0 + 4.0 * a["gamma"] if c_local is None else c_local
    L_max = mobility(a["T_clip"], a)
    kap = a["kappa_g"] * a["ad_hoc"] * (1.0 + max(a["anisotropy"], 0.0))
    stiff = 4.0 * kap * sum(1.0 / (h * h) for h in h_xyz) + a["m_g"] / a["ad_hoc"] * c
    dt_max = 2.0 / (L_max * stiff)
    return fraction * dt_max, dt_max, c


# The values of pf_params_t in the order of its fields, without its mesh size and laser, and the layout up to its laser.
_VALUES = itemgetter("Nz", "Ny", "Nx", "num_oris", "m_g", "gamma", "kappa_g", "ad_hoc", "L0", "Qg", "gas_const",
                     "T_liquidus", "T_clip", "zeta_sharpness", "anisotropy", "force_liquid", "liquid_shift")
_HEAD = struct.Struct("@4i14dixxxxd")
assert _HEAD.size == _lib.ParamsT.laser.offset


def make_params(pf_args, h_xyz, laser=None):
    """Pack pf_args (+ a laser descriptor) into the C struct pf_params_t.

    Every call reads the values that pf_args holds then: they may be arrays or tensors that are changed in
    place.  Packed by one call of struct (a small step is launched every few microseconds)."""
    try:
        if type(pf_args) is not dict:
            raise KeyError
        values = _VALUES(pf_args)
    except KeyError:
        values = _VALUES(with_defaults(pf_args))
    nz, ny, nx, k, m_g, gamma, kappa_g, ad_hoc, L0, Qg, gas_const, T_l, T_clip, sharp, aniso, force, shift = values
    force = 1 if force else 0
    p = _lib.ParamsT()
    try:
        _HEAD.pack_into(p, 0, nz, ny, nx, k, h_xyz[0], h_xyz[1], h_xyz[2], m_g, gamma, kappa_g, ad_hoc, L0, Qg,
                        gas_const, T_l, T_clip, sharp, aniso, force, shift)
    except (struct.error, TypeError):
        # values of other types (text from a yaml file, sizes as floats); sizes to 32 bits as ctypes takes them
        size = [(int(n) + 2 ** 31) % 2 ** 32 - 2 ** 31 for n in (nz, ny, nx, k)]
        _HEAD.pack_into(p, 0, *size, *(float(x) for x in (h_xyz[0], h_xyz[1], h_xyz[2], *values[4:15])), force, float(shift))
    if laser is not None:
        laser.fill(p.laser)
    else:
        p.laser.model = _lib.PF_T_BUFFER
        p.laser.T_dtype = _lib.PF_F64
    return p
