"""CPU tests of how PFSolver.run hands a long run to pf_run: blocks that go on from each other, and a Ctrl-C that takes
effect between them.  A stand-in for the native call applies pf_run's contract to host memory."""
import ctypes
import gc
import signal
import weakref
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from pfkit import _lib, allen_cahn
from pfkit.allen_cahn import RUN_BLOCK, PFSolver
from problems import args, gaussian


@pytest.fixture
def solver(monkeypatch):
    pc = SimpleNamespace(mesh_h_xyz=(1.0, 1.0, 1.0), unique_grain_directions=np.zeros((3, 3, 3)))
    s = PFSolver(args(4, 3, 2, 3), pc, dtype="float64", device="cpu", tile=-1, zchunk=0, clean=False)
    s.calls = []

    def pf_run(src, b0, b1, dtype, T, p, axes, ts, steps, tile, zchunk, stream):
        assert b0 not in (src, b1) and steps >= 1
        s.calls.append(steps)
        view = lambda a: np.frombuffer((ctypes.c_double * 72).from_address(a))  # noqa: E731
        t = np.frombuffer((ctypes.c_double * (steps + 1)).from_address(ts))
        for i in range(steps):
            out = view((b0, b1)[i % 2])
            out[:] = 0.75 * view(src) + (t[i + 1] - t[i]) * t[i]
            src = (b0, b1)[i % 2]
        if s.interrupt_at == len(s.calls):
            signal.raise_signal(signal.SIGINT)
        return 0

    s.interrupt_at = 0
    monkeypatch.setattr(allen_cahn._lib, "load", lambda: SimpleNamespace(pf_run=pf_run))
    monkeypatch.setattr(allen_cahn._lib, "stream_handle", lambda d: 0)
    return s


@pytest.mark.parametrize("n", [0, 1, 2, RUN_BLOCK - 1, RUN_BLOCK, RUN_BLOCK + 1, RUN_BLOCK + 2, 3 * RUN_BLOCK + 5])
def test_blocks_go_on_from_each_other(solver, n):
    eta0 = torch.rand(24, 3, dtype=torch.float64, generator=torch.Generator().manual_seed(n))
    keep = eta0.clone()
    ts = 0.1 + np.cumsum(np.random.default_rng(n).random(n + 1))
    got = solver.run(eta0, ts, gaussian(4, 3, 2))
    want = keep.numpy().copy()
    for i in range(n):
        want = 0.75 * want + (ts[i + 1] - ts[i]) * ts[i]
    assert np.array_equal(got.numpy(), want) and torch.equal(eta0, keep) and got.data_ptr() != eta0.data_ptr()
    assert sum(solver.calls) == n and max(solver.calls, default=0) <= RUN_BLOCK


def test_an_interrupt_takes_effect_between_blocks(solver):
    solver.interrupt_at = 2
    with pytest.raises(KeyboardInterrupt):
        solver.run(torch.zeros(24, 3, dtype=torch.float64), np.arange(50 * RUN_BLOCK + 1.0), gaussian(4, 3, 2))
    assert len(solver.calls) == 2


def test_a_run_holds_its_temperature(solver):
    """The converted copy of a temperature array stays while the run's blocks read it, also if another call on the same
    solver (another thread's) converts one of its own between them."""
    held = []

    class Between:
        def __init__(self, pf_run):
            self.pf_run = pf_run

        def __call__(self, *a):
            held.append(held[0] if held else weakref.ref(solver.state_rhs._T_keep))
            solver.state_rhs.params_for(np.zeros(24, np.float16))
            gc.collect()
            assert held[-1]() is not None
            return self.pf_run(*a)

    lib = SimpleNamespace(pf_run=Between(allen_cahn._lib.load().pf_run))
    allen_cahn._lib.load = lambda: lib
    solver.run(torch.zeros(24, 3, dtype=torch.float64), np.arange(2 * RUN_BLOCK + 1.0), np.full(24, 900.0, np.float16))
    assert len(held) == 2 and held[0]() is None


def test_pf_run_refuses_aliased_buffers_without_gpu():
    from pfkit.config import make_params
    p = make_params(args(8, 8, 8, 4), (1.0, 1.0, 1.0))
    ts = np.zeros(3)
    for src, b0, b1 in ((16, 16, 32), (16, 32, 32)):
        rc = _lib.load().pf_run(src, b0, b1, _lib.PF_F32, None, p, None, ts.ctypes.data, 2, -1, 0, None)
        assert rc == _lib.PF_E_ARG and b"alias" in _lib.load().pf_last_error()
    # eta_in may be buf1: refused further on (no temperature buffer), not for its address
    rc = _lib.load().pf_run(32, 16, 32, _lib.PF_F32, None, p, None, ts.ctypes.data, 2, -1, 0, None)
    assert rc == _lib.PF_E_ARG and b"T buffer" in _lib.load().pf_last_error()
