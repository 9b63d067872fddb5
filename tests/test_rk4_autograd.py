"""CPU tests of what rk4 hands to the stage kernels, which compute no derivatives: not a state or a time that autograd
follows.  The right-hand side stands in for pf_rhs, whose result is a new tensor outside of autograd."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from pfkit.allen_cahn import StateRHS, rk4
from problems import args, gaussian


@pytest.fixture
def rhs(monkeypatch):
    pc = SimpleNamespace(mesh_h_xyz=(1.0, 1.0, 1.0), unique_grain_directions=np.zeros((3, 3, 3)))
    f = StateRHS(pc, args(4, 3, 2, 3), dtype=torch.float64, device="cpu")
    f.native = 0

    def rk4_step(self, eta, T, t_prev, t_crt):
        self.native += 1
        return -0.5 * eta.detach()

    monkeypatch.setattr(StateRHS, "rk4_step", rk4_step)
    monkeypatch.setattr(StateRHS, "__call__", lambda self, y, t, p: 2.0 * y.detach() + float(t))
    return f


def _state():
    return torch.rand(24, 3, dtype=torch.float64, generator=torch.Generator().manual_seed(2))


def _combination(y, t, h):
    f = lambda y, t: 2.0 * y + t  # noqa: E731
    k1 = h * f(y, t)
    k2 = h * f(y + k1 / 2, t + h / 2)
    k3 = h * f(y + k2 / 2, t + h / 2)
    k4 = h * f(y + k3, t + h)
    return k1, k2, k3, k4


def test_untracked_states_take_the_stage_kernels(rhs):
    y = _state()
    for eta, t in ((y, 0.1), (y, torch.tensor(0.1)), (y.clone().requires_grad_(), 0.1)):
        with torch.no_grad():
            rk4((eta, t), 0.2, rhs, [gaussian(4, 3, 2)])
    assert rhs.native == 3


def test_a_tangent_of_the_state_follows(rhs):
    y, v = _state(), torch.ones(24, 3, dtype=torch.float64)
    with fwAD.dual_level():
        (out, _), _ = rk4((fwAD.make_dual(y, v), 0.1), 0.2, rhs, [gaussian(4, 3, 2)])
        value, tangent = fwAD.unpack_dual(out)
        want = y + sum(c * k for c, k in zip((1 / 6, 2 / 6, 2 / 6, 1 / 6), _combination(y, 0.1, 0.1)))
        assert rhs.native == 0 and torch.equal(tangent, v) and torch.allclose(value, want, rtol=1e-14, atol=0)


@pytest.mark.parametrize("which", ["t_prev", "t_crt"])
def test_a_gradient_of_a_time_follows(rhs, which):
    """The right-hand sides are outside of autograd, so the derivative by a time is that of the step h in front of them."""
    y = _state()
    t = {"t_prev": 0.1, "t_crt": 0.2}
    t[which] = torch.tensor(t[which], dtype=torch.float64, requires_grad=True)
    (out, _), _ = rk4((y, t["t_prev"]), t["t_crt"], rhs, [gaussian(4, 3, 2)])
    out.sum().backward()
    ks = _combination(y, 0.1, 0.1)
    want = sum(c * k.sum() / 0.1 for c, k in zip((1 / 6, 2 / 6, 2 / 6, 1 / 6), ks)) * (1 if which == "t_crt" else -1)
    assert rhs.native == 0 and t[which].grad == pytest.approx(float(want), rel=1e-12)


def test_a_gradient_of_the_state_follows(rhs):
    y = _state().requires_grad_()
    (out, _), _ = rk4((y, 0.1), 0.2, rhs, [gaussian(4, 3, 2)])
    out.sum().backward()
    assert rhs.native == 0 and torch.equal(y.grad, torch.ones_like(y))
