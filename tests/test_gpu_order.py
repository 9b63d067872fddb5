"""GPU tests of the order in which a step's tiles go to the XCDs, and of the tiles that the library chooses for long and
flat grids: bitwise the step of the march of channel groups, whatever the order."""
import pytest
import torch

from pfkit import PFSolver
from problems import args, gaussian, poly

pytestmark = pytest.mark.gpu


def _states(cuda, nx, ny, nz, k, dtype):
    a = args(nx, ny, nz, k, anisotropy=0.15, force_liquid=True)
    s = PFSolver(a, poly(nx, ny, nz, k, grains=20), dtype=dtype, device=cuda, clean=False, tile=-1, zchunk=0)
    eta = s.ini_cond()
    eta[::3] += torch.rand(eta[::3].shape, device=cuda, generator=torch.Generator(cuda).manual_seed(k)).to(eta.dtype) * 0.2
    return s, eta


# whole rows and even shares: rows that overflow an XCD, fewer rows than XCDs, one row, rows that fit, a cut last row
@pytest.mark.parametrize("dtype,k,dims", [
    ("float32", 20, (320, 72, 48)), ("float32", 20, (1024, 16, 32)), ("float32", 17, (200, 56, 64)), ("float32", 16, (700, 9, 40)),
    ("bfloat16", 20, (333, 71, 25)), ("bfloat16", 13, (240, 88, 40)), ("float64", 16, (1024, 16, 32)), ("float64", 10, (130, 77, 33)),
    ("float32", 10, (2000, 5, 3))])
def test_orders_of_tiles_are_bitwise_the_same(cuda, dtype, k, dims):
    s, eta = _states(cuda, *dims, k, dtype)
    L = gaussian(*dims)
    outs = []
    for tile, zc in ((-2, 0), (-1, 0), (0, 0), (1, 4), (1, 0x10000 | 6), (2 if dtype != "float64" else 0, 1)):
        out = torch.full_like(eta, float("nan"))
        s.state_rhs.step(eta, out, L, 0.1, 0.101, tile, zc)
        outs.append(out)
    for o in outs[1:]:
        assert torch.equal(o, outs[0])


# each side of the library's choice of tile on few planes
@pytest.mark.parametrize("dtype,k,dims", [
    ("float32", 16, (300, 310, 1)), ("float32", 13, (201, 220, 1)), ("float32", 13, (64, 700, 1)), ("bfloat16", 13, (400, 403, 3)),
    ("bfloat16", 13, (201, 203, 3)), ("bfloat16", 16, (250, 255, 8)), ("bfloat16", 16, (250, 255, 13)), ("float32", 20, (251, 249, 4)),
    ("float32", 20, (251, 249, 7)), ("float32", 16, (300, 500, 6)), ("bfloat16", 12, (250, 251, 12)), ("float64", 16, (300, 310, 1))])
def test_choice_on_few_planes_is_bitwise_the_same(cuda, dtype, k, dims):
    s, eta = _states(cuda, *dims, k, dtype)
    L = gaussian(*dims)
    out, want = torch.full_like(eta, float("nan")), torch.full_like(eta, float("nan"))
    s.state_rhs.step(eta, want, L, 0.1, 0.101, -2, 0)
    s.state_rhs.step(eta, out, L, 0.1, 0.101, -1, 0)
    assert torch.equal(out, want)


@pytest.mark.parametrize("tile", [0, 1, 2])
def test_one_long_row_of_tiles(cuda, tile):
    """A row of 19 million tiles: dealt by whole rows it would be padded to eight of them, past the largest launch."""
    nx = 300_000_000
    a = args(nx, 1, 1, 1)
    eta = torch.rand(nx, 1, device=cuda, generator=torch.Generator(cuda).manual_seed(5))

    class One:
        Nx, Ny, Nz, mesh_h_xyz, num_oris, unique_grain_directions = nx, 1, 1, (1.0, 1.0, 1.0), 1, None

    s = PFSolver(a, One(), dtype="float32", device=cuda, clean=False, tile=-1, zchunk=0)
    L = gaussian(nx, 1, 1)
    out, want = torch.full_like(eta, float("nan")), torch.full_like(eta, float("nan"))
    s.state_rhs.step(eta, want, L, 0.1, 0.101, -2, 0)
    s.state_rhs.step(eta, out, L, 0.1, 0.101, tile, 0)
    assert torch.equal(out, want)
