"""Grain segmentation (pfkit.segment on the GPU; oracle/segmentation.py restates
jax_am/phase_field/utils.py:217-310)."""
import numpy as np
import pytest

from oracle import pf_oracle as O
from oracle import segmentation as S
from problems import args, gaussian, poly


def test_oracle_pca_matches_sklearn():
    from sklearn.decomposition import PCA
    rng = np.random.default_rng(4)
    for n in (5, 9, 40):
        X = rng.normal(size=(n, 3)) * np.array([3.0, 1.0, 0.2]) + rng.normal(size=3) * 10
        ref = PCA(n_components=3).fit(X).explained_variance_
        np.testing.assert_allclose(S.pca_variances(X), ref, rtol=1e-10)


def test_oracle_bfs_order_by_hand():
    # 4 x 3 x 1 grid (x fastest), orientations:
    #   y=0: 0 0 1 1
    #   y=1: 0 1 1 0
    #   y=2: 0 0 0 0     cell 5 (x=1, y=1) is liquid
    ori = np.array([0, 0, 1, 1, 0, 1, 1, 0, 0, 0, 0, 0])
    nonliquid = np.ones(12, bool)
    nonliquid[5] = False
    g = S.bfs_grains(ori, nonliquid, 2, 1, 3, 4)
    # orientation 0: {0,1,4,8,9,10,11,7} from cell 0; orientation 1: {2,3,6} from cell 2
    assert [sorted(x) for x in g] == [[0, 1, 4, 7, 8, 9, 10, 11], [2, 3, 6]]
    # BFS visiting order of the first grain (x-, x+, y-, y+ neighbour order)
    assert g[0][:3] == [0, 1, 4]


def test_oracle_box_aspect_ratio_closed_form():
    Nx, Ny, Nz = 10, 6, 5
    ori = np.zeros(Nx * Ny * Nz, int)
    z, y, x = np.meshgrid(np.arange(Nz), np.arange(Ny), np.arange(Nx), indexing="ij")
    box = (x >= 2) & (x < 8) & (y >= 1) & (y < 4) & (z >= 1) & (z < 3)   # 6 x 3 x 2 cells
    ori[box.reshape(-1)] = 1
    grains, vols, ars = S.segment(ori, np.ones(len(ori), bool), 2, Nz, Ny, Nx, (1.0, 1.0, 1.0))
    i = [k for k, gg in enumerate(grains) if ori[gg[0]] == 1][0]
    assert vols[i] == 36.0
    expected = 2 * np.sqrt(6**2 - 1) / (np.sqrt(3**2 - 1) + np.sqrt(2**2 - 1))
    assert abs(ars[i] - expected) < 1e-12


def test_host_statistics_match_oracle_on_random_grains():
    from pfkit.segment import _covariances, aspect_ratios
    rng = np.random.default_rng(2)
    Nx, Ny, Nz, h = 9, 7, 6, (0.5, 1.0, 2.0)
    ori = rng.integers(0, 2, size=Nx * Ny * Nz)
    grains, vols, ars = S.segment(ori, np.ones(len(ori), bool), 2, Nz, Ny, Nx, h)
    mom = []
    for g in grains:
        iz, r = np.divmod(np.array(g), Ny * Nx)
        iy, ix = np.divmod(r, Nx)
        mom.append([len(g), ix.sum(), iy.sum(), iz.sum(), (ix * ix).sum(), (iy * iy).sum(), (iz * iz).sum(),
                    (ix * iy).sum(), (ix * iz).sum(), (iy * iz).sum()])
    mom = np.array(mom, dtype=np.int64)
    got = aspect_ratios(_covariances(mom, h), mom[:, 0])
    np.testing.assert_allclose(got, ars, rtol=1e-9)


def _state(Nx, Ny, Nz, K, seed):
    a = args(Nx, Ny, Nz, K)
    pc = poly(Nx, Ny, Nz, K, grains=max(4, Nx * Ny * Nz // 60), seed=seed)
    eta = O.ini_cond(pc.cell_ori_inds, K) * 0.9 + 0.05 * np.random.default_rng(seed).random((Nx * Ny * Nz, K))
    return a, pc, eta


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(20, 16, 12, 4, 1), (33, 9, 7, 3, 2), (1, 1, 30, 2, 3)])
def test_gpu_segmentation_matches_oracle(shape, cuda):
    import torch
    from pfkit import PFSolver
    from pfkit.segment import grains
    Nx, Ny, Nz, K, seed = shape
    a, pc, eta = _state(Nx, Ny, Nz, K, seed)
    L = gaussian(Nx, Ny, Nz)                    # melts a pool under the top surface
    t = 0.3
    T = O.laser_T(L.as_dict(), O.centroids(Nz, Ny, Nx, pc.mesh_h_xyz), t).reshape(-1)
    ref_g, ref_v, ref_a = S.segment(np.argmax(eta, axis=1), T < a["T_liquidus"], K, Nz, Ny, Nx, pc.mesh_h_xyz)
    s = PFSolver(a, pc, dtype=torch.float64, device=cuda, clean=False)
    got = grains(s, eta, L, t)
    assert len(got.root) == len(ref_g)
    assert got.root.tolist() == [min(g) for g in ref_g]
    assert got.n_cells.tolist() == [len(g) for g in ref_g]
    np.testing.assert_allclose(got.volumes, ref_v, rtol=1e-12)
    np.testing.assert_allclose(got.aspect_ratios, ref_a, rtol=1e-9)
    lab = got.labels.cpu().numpy()
    for g in ref_g:
        assert np.all(lab[g] == min(g))
    liquid = ~(T < a["T_liquidus"])
    assert np.all(lab[liquid] == -1)


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,nz,k", [(1, 1, 1, 1), (31, 7, 3, 2), (32, 8, 4, 2), (33, 9, 5, 2), (65, 17, 9, 3),
                                        (100, 1, 1, 2), (1, 50, 33, 2), (64, 40, 37, 2)])
@pytest.mark.parametrize("kind", ["noise", "one", "snake"])
def test_labels_across_tiles(cuda, nx, ny, nz, k, kind):
    """Labels, roots and moments where components wind through many tiles: random cells (hundreds of grains
    to a tile, far more than its slots for moments), one component, and a comb whose teeth join at one
    end.  Orientation values may be any int32.  Integer results: equal, not close."""
    import ctypes
    import torch
    from scipy import ndimage
    from pfkit import _lib
    from pfkit.config import make_params
    n = nx * ny * nz
    rng = np.random.default_rng(n)
    shape = (nz, ny, nx)
    if kind == "noise":
        ori = np.array([-7, 2 ** 31 - 1, -2 ** 31], np.int32)[rng.integers(0, k, shape)]
    elif kind == "one":
        ori = np.zeros(shape, np.int32)
    else:
        ori = (np.arange(ny)[None, :, None] % 2 + np.zeros(shape)).astype(np.int32)
        ori[:, :, -1] = 0
    T = rng.choice([300.0, 300.0, 300.0, 1700.0], n) if kind == "noise" else np.full(n, 300.0)
    solid = T.reshape(shape) < 1623.0
    want = np.full(shape, -1, np.int64)
    idx = np.arange(n).reshape(shape)
    for o in np.unique(ori):
        lab, m = ndimage.label(solid & (ori == o))
        if m:
            first = ndimage.minimum(idx, lab, np.arange(1, m + 1)).astype(np.int64)
            want[lab > 0] = first[lab[lab > 0] - 1]
    a = args(nx, ny, nz, k)
    p = make_params(a, (1.0, 1.0, 1.0), None)
    p.laser.model, p.laser.T_dtype = _lib.PF_T_BUFFER, _lib.PF_F64
    dev = lambda v: torch.as_tensor(v, device=cuda)  # noqa: E731
    od, Td = dev(ori.reshape(-1)), dev(T)
    out = [torch.full((n,), -9, dtype=torch.int32, device=cuda) for _ in range(3)]
    ws, ng = torch.full((2,), 77, dtype=torch.int32, device=cuda), ctypes.c_int32(-1)
    lib, st = _lib.load(), _lib.stream_handle(cuda)
    _lib.check(lib.pf_segment(od.data_ptr(), Td.data_ptr(), p, 0.0, out[0].data_ptr(), out[1].data_ptr(),
                              out[2].data_ptr(), ws.data_ptr(), 1, ctypes.byref(ng), st), "pf_segment")
    labels, cid, root = (v.cpu().numpy() for v in out)
    assert np.array_equal(labels, want.reshape(-1))
    roots = np.unique(labels[labels >= 0])
    assert ng.value == len(roots) and np.array_equal(np.sort(root[:ng.value]), roots)
    assert np.array_equal(cid[root[:ng.value]], np.arange(ng.value))
    if ng.value:
        mom = torch.full((ng.value, 10), -5, dtype=torch.int64, device=cuda)
        _lib.check(lib.pf_segment_moments(out[0].data_ptr(), out[1].data_ptr(), p, ng.value, mom.data_ptr(), st), "moments")
        c = np.flatnonzero(labels >= 0)
        z, y, x = np.unravel_index(c, shape)
        cols = [np.ones_like(x), x, y, z, x * x, y * y, z * z, x * y, x * z, y * z]
        ref = np.stack([np.bincount(cid[labels[c]], v, ng.value) for v in cols], axis=1).astype(np.int64)
        assert np.array_equal(mom.cpu().numpy(), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("ng", [1, 30_000_001, 2 ** 32 // 10 + 5])
def test_moments_of_very_many_grains(cuda, ng):
    """More moments than a launch has threads (2^32; 34 GB), and than its blocks clear in one turn: zero but for the
    rows of the grains that have cells."""
    import torch
    from pfkit import _lib
    from pfkit.config import make_params
    nx, ny, nz = 5, 3, 2
    p = make_params(args(nx, ny, nz, 2), (1.0, 1.0, 1.0), None)
    labels = torch.zeros(nx * ny * nz, dtype=torch.int32, device=cuda)
    labels[nx * ny:] = 20
    cid = torch.zeros(nx * ny * nz, dtype=torch.int32, device=cuda)
    cid[20] = ng - 1
    mom = torch.full((ng, 10), -5, dtype=torch.int64, device=cuda)
    _lib.check(_lib.load().pf_segment_moments(labels.data_ptr(), cid.data_ptr(), p, ng, mom.data_ptr(),
                                              _lib.stream_handle(cuda)), "moments")
    z, y, x = np.unravel_index(np.arange(nx * ny * nz), (nz, ny, nx))
    cols = np.stack([np.ones_like(x), x, y, z, x * x, y * y, z * z, x * y, x * z, y * z], axis=1)
    halves = cols[:nx * ny].sum(0), cols[nx * ny:].sum(0)
    if ng == 1:
        assert np.array_equal(mom[0].cpu().numpy(), halves[0] + halves[1])
    else:
        assert np.array_equal(mom[0].cpu().numpy(), halves[0]) and np.array_equal(mom[-1].cpu().numpy(), halves[1])
        for part in mom[1:-1].split(1 << 26):
            assert not bool(part.any())
