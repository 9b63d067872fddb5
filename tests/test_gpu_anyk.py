"""GPU parity of the kernels for any K (pf_step without a tiled instantiation, pf_rhs): K around a
thread's channel group, up to and past the largest K of one workgroup, on grids whose planes are not
whole runs of cells and whose planes are not whole marches."""
import numpy as np
import pytest
import torch

from oracle import pf_oracle as O
from pfkit import PFSolver, rk4
from problems import args, gaussian, poly, quench

pytestmark = pytest.mark.gpu

# K: single channels, tails of every length, whole groups, the last K of the channel-group march in
# FP64 (256) and FP32 (512) and the first past them
CASES = [(7, 5, 9, 1), (19, 7, 3, 3), (23, 9, 40, 25), (11, 13, 5, 26), (10, 6, 9, 27), (16, 8, 21, 28), (29, 31, 7, 33),
         (1, 1, 30, 40), (37, 1, 1, 64), (5, 4, 3, 256), (4, 3, 3, 257), (3, 3, 2, 512), (3, 2, 2, 513)]


@pytest.mark.parametrize("nx,ny,nz,k", CASES)
@pytest.mark.parametrize("aniso", [0.0, 0.15])
def test_step_and_rhs_any_k(cuda, nx, ny, nz, k, aniso):
    a = args(nx, ny, nz, k, anisotropy=aniso, force_liquid=True)
    pc = poly(nx, ny, nz, k)
    n = nx * ny * nz
    rng = np.random.default_rng(n + k)
    eta = np.where(rng.random((n, k)) < 0.3, 0.0, rng.random((n, k)))
    cent = O.centroids(nz, ny, nx, pc.mesh_h_xyz)
    for L in (gaussian(nx, ny, nz), quench(nz)):
        T = O.laser_T(L.as_dict(), cent, 0.1)
        # FP64: rounding of sums of up to k squares; FP32 storage: inputs rounded alike, one stochastic
        # rounding (2^-23) of the result and FP32 sums of k terms of one sign, k 2^-24 of the sum S <= k
        for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 2e-6)):
            e = torch.as_tensor(eta, dtype=dtype, device=cuda)
            ed = e.double().cpu().numpy()
            s = PFSolver(a, pc, dtype=dtype, device=cuda, clean=False, tile=-2, zchunk=0)
            (out, _), _ = s.stepper((e, 0.1), 0.1001, [L])
            ref = O.explicit_euler(ed, 0.1, 0.1001, T, a, pc.mesh_h_xyz, pc.unique_grain_directions)
            assert np.max(np.abs(out.double().cpu().numpy() - ref)) <= tol * max(1.0, np.max(np.abs(ref)))
            rhs = s.state_rhs(e, 0.1, [L]).double().cpu().numpy()
            want = O.state_rhs(ed, T, a, pc.mesh_h_xyz, pc.unique_grain_directions)
            assert np.max(np.abs(rhs - want)) <= max(tol, k * (6e-8 if dtype == torch.float32 else 0)) * max(1.0, np.max(np.abs(want)))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [3, 9, 10, 17, 20])
def test_rhs_reads_unaligned_states(cuda, dtype, k):
    nx, ny, nz = 21, 10, 7
    a = args(nx, ny, nz, k, anisotropy=0.15)
    s = PFSolver(a, poly(nx, ny, nz, k), dtype=dtype, device=cuda, clean=False)
    n = nx * ny * nz
    buf = torch.rand(n * k + 1, device=cuda, generator=torch.Generator(cuda).manual_seed(k)).to(dtype)
    e = buf[1:].view(n, k)
    assert torch.equal(s.state_rhs(e, 0.1, [gaussian(nx, ny, nz)]), s.state_rhs(e.clone(), 0.1, [gaussian(nx, ny, nz)]))


# both sides of the library's choice (channel groups / which tile) for tile -1, by dtype and K
@pytest.mark.parametrize("dtype,k,dims", [
    ("float32", 20, (64, 64, 22)), ("float32", 20, (64, 64, 24)), ("float32", 17, (57, 61, 30)), ("float32", 17, (57, 61, 31)),
    ("float32", 10, (67, 63, 40)), ("float32", 2, (90, 70, 60)), ("bfloat16", 20, (64, 64, 24)), ("bfloat16", 10, (61, 50, 27)),
    ("bfloat16", 12, (80, 60, 40)), ("float64", 10, (50, 50, 41)), ("float64", 10, (50, 50, 39)), ("float64", 16, (63, 50, 41)),
    ("float64", 16, (63, 50, 45)), ("float64", 13, (91, 77, 85)), ("float64", 17, (33, 33, 20)), ("float64", 19, (91, 77, 62))])
def test_library_choice_is_bitwise_the_tiled_step(cuda, dtype, k, dims):
    nx, ny, nz = dims
    a = args(nx, ny, nz, k, anisotropy=0.15, force_liquid=True)
    pc = poly(nx, ny, nz, k, grains=20)
    s = PFSolver(a, pc, dtype=dtype, device=cuda, clean=False, tile=-1, zchunk=0)
    L = gaussian(nx, ny, nz)
    eta = s.ini_cond()
    eta[::3] += torch.rand(eta[::3].shape, device=cuda, generator=torch.Generator(cuda).manual_seed(k)).to(eta.dtype) * 0.2
    outs = []
    for tile, zc in ((-1, 0), (-1, 5), (-1, 0x10000), (0, 4), (-2, 0), (-2, 3)):
        out = torch.empty_like(eta)
        s.state_rhs.step(eta, out, L, 0.1, 0.101, tile, zc)
        outs.append(out)
    for o in outs[1:]:
        assert torch.equal(o, outs[0])


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("nx,ny,nz,k", [(9, 7, 5, 1), (21, 10, 7, 5), (16, 16, 11, 16), (33, 5, 9, 17), (12, 11, 20, 20),
                                        (4, 3, 3, 256), (3, 2, 2, 513)])
def test_rk4_matches_the_oracle(cuda, dtype, nx, ny, nz, k):
    a = args(nx, ny, nz, k, anisotropy=0.15)
    pc = poly(nx, ny, nz, k)
    n = nx * ny * nz
    s = PFSolver(a, pc, dtype=dtype, device=cuda, clean=False)
    rng = np.random.default_rng(k)
    buf = torch.zeros(n * k + 1, dtype=dtype, device=cuda)
    e = buf[1:].view(n, k)                      # aligned to one element only
    e.copy_(torch.as_tensor(np.where(rng.random((n, k)) < 0.3, 0.0, rng.random((n, k)) / np.sqrt(k)), device=cuda))
    ed = e.double().cpu().numpy()
    T = rng.uniform(900.0, 1900.0, (n, 1))      # a temperature array is held over the step, as the oracle does
    h = 2e-3
    (got, t), _ = rk4((e, 0.1), 0.1 + h, s.state_rhs, [torch.as_tensor(T, device=cuda)])
    want = O.rk4(ed, 0.1, 0.1 + h, T, a, pc.mesh_h_xyz, pc.unique_grain_directions)
    assert t == 0.1 + h
    # one rounding of the result to the storage type, stage states rounded alike times h |d rhs| << 1; FP64 as the step
    tol = {torch.float64: 1e-12, torch.float32: 2e-6, torch.bfloat16: 2.0 ** -7}[dtype]
    assert np.max(np.abs(got.double().cpu().numpy() - want)) <= tol * max(1.0, np.max(np.abs(want)))
    # a source that moves within the step: the stages' own temperatures (four pf_rhs calls)
    L = gaussian(nx, ny, nz)
    f = lambda y, tt: s.state_rhs(y, tt, [L]).double()  # noqa: E731
    y = e.double()
    k1 = f(e, 0.1)
    k2 = f((y + h / 2 * k1).to(dtype), 0.1 + h / 2)
    k3 = f((y + h / 2 * k2).to(dtype), 0.1 + h / 2)
    k4 = f((y + h * k3).to(dtype), 0.1 + h)
    (got, _), _ = rk4((e, 0.1), 0.1 + h, s.state_rhs, [L])
    ref = y + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    assert float((got.double() - ref).abs().max()) <= tol * max(1.0, float(ref.abs().max()))
