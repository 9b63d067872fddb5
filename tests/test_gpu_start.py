"""GPU tests of what a solve starts from and is coupled to: the Voronoi grain map (against every seed for every
cell), the one-hot state and the CFD temperature, at the edges of their boxes, runs and squares."""
import numpy as np
import pytest
import torch

from pfkit import _lib
from pfkit.config import make_params
from pfkit.coupling import cfd_temperature
from problems import args

pytestmark = pytest.mark.gpu


def _brute(seeds, nx, ny, nz, h):
    z, y, x = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    c = [(i + 0.5) * hh for i, hh in zip((x, y, z), h)]
    best, ind = np.full((nz, ny, nx), np.inf), np.zeros((nz, ny, nx), np.int32)
    for g, s in enumerate(seeds):
        dx, dy, dz = c[0] - s[0], c[1] - s[1], c[2] - s[2]
        d = dx * dx + dy * dy + dz * dz
        near = d < best
        best[near], ind[near] = d[near], g
    return ind.reshape(-1)


@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (16, 8, 4), (17, 9, 5), (37, 3, 21), (15, 7, 3)])
@pytest.mark.parametrize("kind", ["one", "random", "crowd", "ties", "outside", "broken"])
def test_voronoi_is_every_seed_for_every_cell(cuda, nx, ny, nz, kind):
    rng = np.random.default_rng(nx + ny)
    h = (0.5, 1.0, 1.75)
    L = np.array([nx * h[0], ny * h[1], nz * h[2]])
    seeds = {"one": lambda: rng.random((1, 3)) * L, "random": lambda: rng.random((300, 3)) * L,
             "crowd": lambda: 0.5 * L + rng.random((1300, 3)) * 1e-3,      # more candidates than a box keeps
             "ties": lambda: np.repeat(np.round(rng.random((40, 3)) * L), 3, axis=0),
             "outside": lambda: rng.normal(size=(60, 3)) * 40 * L,
             "broken": lambda: np.concatenate(([[np.nan] * 3, [np.inf, 0, 0]], rng.random((20, 3)) * L))}[kind]()
    gori = rng.integers(0, 9, len(seeds)).astype(np.int32)
    p = make_params(args(nx, ny, nz, 2), h, None)
    sd, go = torch.as_tensor(seeds, device=cuda), torch.as_tensor(gori, device=cuda)
    out = torch.full((nx * ny * nz + 1,), -3, dtype=torch.int32, device=cuda)
    want = _brute(seeds, nx, ny, nz, h)
    lib, st = _lib.load(), _lib.stream_handle(cuda)
    for g, ref in ((None, want), (go, gori[want])):
        _lib.check(lib.pf_voronoi(sd.data_ptr(), len(seeds), _lib.ptr(g), p, out.data_ptr(), st), "pf_voronoi")
        assert np.array_equal(out[:-1].cpu().numpy(), ref) and out[-1] == -3


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,k", [(1, 1), (255, 3), (256, 20), (257, 17), (700, 7), (3, 1000)])
def test_onehot_runs(cuda, dtype, n, k):
    rng = np.random.default_rng(n)
    ori = rng.integers(-1, k + 1, n).astype(np.int32)       # -1 and k name no channel: a row of zeros
    buf = torch.full((n * k + 2,), 5.0, dtype=dtype, device=cuda)
    od = torch.as_tensor(ori, device=cuda)
    _lib.check(_lib.load().pf_init_onehot(buf[1:].data_ptr(), _lib.TORCH_TO_PF[dtype], od.data_ptr(), n, k,
                                          _lib.stream_handle(cuda)), "pf_init_onehot")
    got = buf.double().cpu().numpy()
    assert got[0] == 5.0 and got[-1] == 5.0
    assert np.array_equal(got[1:-1].reshape(n, k), (np.arange(k) == ori[:, None]).astype(float))


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("nx,ny,nz", [(1, 1, 1), (32, 2, 32), (33, 5, 31), (7, 40, 65), (100, 3, 1)])
def test_cfd_temperature_squares(cuda, dtype, nx, ny, nz):
    g = torch.Generator(cuda).manual_seed(nx)
    a, b = (torch.rand(nx, ny, nz, dtype=dtype, device=cuda, generator=g) * 2000 for _ in range(2))
    got = cfd_temperature(a, b, 0.25, 1.0, 2.0)
    r = (1.0 - 0.25) / 2.0
    want = (r * a.double() + (1.0 - r) * b.double()).to(dtype).permute(2, 1, 0).reshape(-1, 1)
    assert torch.equal(got, want)
