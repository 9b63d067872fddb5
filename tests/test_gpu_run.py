"""GPU tests of PFSolver.run (pf_run): the same states as a loop over stepper, for odd and even step counts, any form
of time grid, a temperature buffer, a state at an unaligned address, and parameters changed between calls."""
import numpy as np
import pytest
import torch

from pfkit import PFSolver
from pfkit.allen_cahn import RUN_BLOCK
from problems import args, gaussian, poly

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [0, 1, 2, 5])
@pytest.mark.parametrize("form", ["array", "list", "tensor", "column"])
def test_run_is_the_stepper_loop(cuda, n, form):
    nx, ny, nz, k = 21, 18, 9, 6
    a = args(nx, ny, nz, k, anisotropy=0.15, force_liquid=True)
    s = PFSolver(a, poly(nx, ny, nz, k), dtype="float32", device=cuda, clean=False)
    buf = torch.rand(nx * ny * nz * k + 1, device=cuda, generator=torch.Generator(cuda).manual_seed(n))
    eta0 = buf[1:].view(-1, k)          # 4-byte aligned
    keep = eta0.clone()
    ts = 0.1 + np.arange(n + 1) * 1e-3
    given = dict(array=ts, list=list(ts), tensor=torch.as_tensor(ts, device=cuda), column=ts.reshape(-1, 1))[form]
    T = torch.rand(nx * ny * nz, 1, device=cuda, dtype=torch.float64) * 1500.0 + 300.0
    for temp in (gaussian(nx, ny, nz), T):
        want = keep.clone()
        for i in range(n):
            (want, _), _ = s.stepper((want, ts[i]), ts[i + 1], [temp])
        got = s.run(eta0, given, temp)
        assert got.data_ptr() != eta0.data_ptr()
        assert torch.equal(got, want) and torch.equal(eta0, keep)


def test_parameters_changed_between_calls_take_effect(cuda):
    nx, ny, nz, k = 16, 12, 8, 5
    a = args(nx, ny, nz, k, anisotropy=0.15)
    pc, L = poly(nx, ny, nz, k), gaussian(nx, ny, nz)
    s = PFSolver(a, pc, dtype="float64", device=cuda, clean=False)
    eta = torch.rand(nx * ny * nz, k, device=cuda, dtype=torch.float64)
    first = s.run(eta, [0.1, 0.101], L)
    s.state_rhs.pf_args["m_g"] = 2.5
    got = s.run(eta, [0.1, 0.101], L)
    want = PFSolver(dict(a, m_g=2.5), pc, dtype="float64", device=cuda, clean=False).run(eta, [0.1, 0.101], L)
    assert torch.equal(got, want) and not torch.equal(got, first)


@pytest.mark.parametrize("dtype,extra", [("float32", 1), ("bfloat16", 2)])
def test_a_run_of_several_blocks(cuda, dtype, extra):
    nx, ny, nz, k = 13, 9, 6, 5
    s = PFSolver(args(nx, ny, nz, k, anisotropy=0.15), poly(nx, ny, nz, k), dtype=dtype, device=cuda, clean=False)
    n = 2 * RUN_BLOCK + extra
    ts, L, eta0 = 0.1 + np.arange(n + 1) * 1e-4, gaussian(nx, ny, nz), s.ini_cond()
    want = eta0
    for i in range(n):
        (want, _), _ = s.stepper((want, ts[i]), ts[i + 1], [L])
    assert torch.equal(s.run(eta0, ts, L), want) and torch.equal(eta0, s.ini_cond())
