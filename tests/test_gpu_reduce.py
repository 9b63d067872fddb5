"""GPU parity of pf_argmax and pf_reduce where their channel groups and runs of cells end: K below,
at and between multiples of a thread's channels, planes that are not whole runs, chunked z, states that
start at an address of the element's own alignment only."""
import numpy as np
import pytest
import torch

from oracle import pf_oracle as O
from pfkit import PFSolver, _lib
from problems import args, gaussian, poly, quench, rosenthal

pytestmark = pytest.mark.gpu

DT = {"float64": torch.float64, "float32": torch.float32, "bfloat16": torch.bfloat16}


def _state(n, k, dtype, cuda, seed):
    """Random state with zeros and ties, one element past the start of its buffer."""
    rng = np.random.default_rng(seed)
    e = np.where(rng.random((n, k)) < 0.4, 0.0, np.round(rng.random((n, k)) * 16) / 16)
    buf = torch.zeros(n * k + 1, dtype=DT[dtype], device=cuda)
    eta = buf[1:].view(n, k)
    eta.copy_(torch.as_tensor(e, device=cuda))
    return eta


@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("k,n", [(1, 700), (2, 333), (3, 1025), (4, 1024), (5, 51), (17, 977), (20, 204 * 3), (33, 64),
                                 (255, 7), (256, 1), (513, 5), (1030, 3)])
def test_argmax_groups(cuda, dtype, k, n):
    eta = _state(n, k, dtype, cuda, 7 * k + n)
    eta[n // 2, k // 2] = float("nan")
    eta[0, k - 1] = float("inf")
    if n > 2:
        eta[n - 1] = -float("inf")
        eta[1] = -0.0
        eta[1, k - 1] = 0.0
    out = torch.full((n + 2,), -7, dtype=torch.int32, device=cuda)
    _lib.check(_lib.load().pf_argmax(eta.data_ptr(), _lib.TORCH_TO_PF[eta.dtype], n, k, out[1:].data_ptr(),
                                     _lib.stream_handle(cuda)), "pf_argmax")
    assert np.array_equal(out[1:-1].cpu().numpy(), np.argmax(eta.double().cpu().numpy(), axis=1))
    assert out[0] == -7 and out[-1] == -7


@pytest.mark.parametrize("dtype", list(DT))
@pytest.mark.parametrize("nx,ny,nz,k", [(1, 1, 1, 1), (5, 1, 9, 2), (1, 7, 70, 3), (37, 11, 6, 5), (16, 16, 3, 16),
                                        (13, 4, 33, 17), (51, 3, 21, 20), (9, 8, 4, 256)])
def test_reduce_groups(cuda, dtype, nx, ny, nz, k):
    a = args(nx, ny, nz, k, anisotropy=0.0)
    pc = poly(nx, ny, nz, k)
    n = nx * ny * nz
    eta = _state(n, k, dtype, cuda, k + n)
    eta0 = torch.roll(eta, 1, 0).contiguous()
    e = eta.double().cpu().numpy()
    s = PFSolver(a, pc, dtype=DT[dtype], device=cuda, clean=False)
    for L in (gaussian(nx, ny, nz), rosenthal(nx, ny, nz), quench(nz)):
        d = s.diagnostics(eta, L, t=0.3, eta0=eta0)
        T = O.laser_T(L.as_dict(), O.centroids(nz, ny, nx, pc.mesh_h_xyz), 0.3)
        Fl, Fg = O.free_energy(e, T, a, pc.mesh_h_xyz)
        # FP64 sums of at most n k terms of one sign in any order: far below n k eps = 3e-11 of the sum of sizes
        size = np.sum(np.abs(e) + e ** 2 + e ** 4) + np.sum(e ** 2) ** 2 / n + 1
        assert abs(d["F_local"] - Fl) <= 1e-12 * size * 8
        assert abs(d["F_grad"] - Fg) <= 1e-12 * max(abs(Fg), 1e-300)
        assert np.allclose(d["volumes"], O.volumes(e, pc.mesh_h_xyz), rtol=1e-13, atol=0)
        assert d["eta_sum"] == pytest.approx(e.sum(), rel=1e-13)
        am = np.argmax(e, axis=1)
        assert np.array_equal(d["argmax_counts"], np.bincount(am, minlength=k))
        assert d["changed"] == int(np.sum(am != np.argmax(eta0.double().cpu().numpy(), axis=1)))
        assert d["liquid"] == int(np.sum(T >= a["T_liquidus"])) and d["nonfinite"] == 0
        assert d["max_T"] == pytest.approx(np.max(T), rel=1e-13)
    eta[n // 2, k // 2] = float("inf")
    eta[n - 1, k - 1] = float("nan")
    assert s.diagnostics(eta, quench(nz), t=0.3)["nonfinite"] == (1 if n == 1 else 2)
