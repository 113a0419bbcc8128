"""Untruncated RBF splat and gradient (matrix products over RBFs and over grid
rows) against the CPU oracle, at the edges of their tiles: 16 z slices and 32
columns (forward), 16 rows, 16 x and 32 RBFs (gradient), chunks of 32 RBFs per
wave, groups of 3 attributes (forward) and channel pairs (gradient).

Tolerance 1e-5 relative L2 against FP64: a Gaussian's exponent k r^2 carries
about four roundings of 2^-24 relative, terms that matter against the 1e-8
guard have |k r^2| < 27, so their relative error stays below
27 ln 2 * 4 * 2^-24 = 4.5e-6."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.cases import rel_l2

VS, VE = (-1.0, -1.0, 0.5), (1.0, 1.0, 2.5)

CASES = [  # B, N, A, (D, H, W)
    (1, 1, 0, (1, 1, 1)),
    (1, 31, 1, (15, 3, 11)),
    (2, 33, 2, (16, 4, 8)),
    (1, 32, 3, (17, 5, 13)),
    (1, 64, 4, (33, 1, 31)),
    (1, 300, 8, (49, 6, 16)),
    (2, 65, 1, (65, 7, 17)),
    (1, 1500, 1, (12, 10, 9)),     # few voxels, many RBFs: the RBFs are split
    (1, 40, 1, (40, 41, 15)),      # few RBFs, many rows: the rows are split
]


def _rbf(rng, B, N, A):
    return np.concatenate([rng.uniform(-1, 1, (B, N, 2)), rng.uniform(0.5, 2.5, (B, N, 1)),
                           rng.uniform(0.08, 0.3, (B, N, 1)), rng.random((B, N, A))],
                          2).astype(np.float32)


def _calls(rbf, res, G, ws):
    """Forward and gradient through the C entry points, with or without scratch."""
    from totrilib_amd import _lib
    lib = _lib.load()
    B, N, C = rbf.shape
    A, (D, H, W) = C - 4, res
    r, g = torch.from_numpy(rbf).cuda(), torch.from_numpy(G).cuda()
    vol, grad = torch.empty_like(g), torch.empty_like(r)
    st = torch.cuda.current_stream().cuda_stream
    nf = lib.totri_rbf2volume_gaussian_forward_workspace(B, N, A, D, H, W, 0.0) if ws else 0
    ng = lib.totri_rbf2volume_gaussian_grad_workspace(B, N, A, D, H, W, 0.0) if ws else 0
    buf = torch.empty(max(nf, ng, 4), dtype=torch.uint8, device="cuda")
    p = lambda n: buf.data_ptr() if n else None  # noqa: E731
    assert lib.totri_rbf2volume_gaussian_forward(
        r.data_ptr(), B, N, A, vol.data_ptr(), D, H, W, _lib.f3(VS), _lib.f3(VE), 0.0, p(nf), nf,
        ctypes.c_void_p(st)) == 0
    assert lib.totri_rbf2volume_gaussian_grad_split(
        r.data_ptr(), B, N, A, vol.data_ptr(), g.data_ptr(), grad.data_ptr(), D, H, W,
        _lib.f3(VS), _lib.f3(VE), 0.0, p(ng), ng, ctypes.c_void_p(st)) == 0
    torch.cuda.synchronize()
    return vol.cpu().numpy(), grad.cpu().numpy(), nf, ng


@pytest.mark.gpu
@pytest.mark.parametrize("B,N,A,res", CASES)
def test_full_splat_tiles(B, N, A, res):
    rng = np.random.default_rng(N + A)
    rbf = _rbf(rng, B, N, A)
    G = rng.standard_normal((B, 1 + A) + res).astype(np.float32)
    ref = O.splat_forward(rbf, res, VS, VE, mode=O.PURE64)
    gref = O.splat_grad(rbf, ref, G, VS, VE, mode=O.PURE64)
    split = []
    for ws in (True, False):
        vol, grad, nf, ng = _calls(rbf, res, G, ws)
        assert rel_l2(vol, ref) < 1e-5
        assert rel_l2(grad, gref) < 1e-5
        split.append((nf, ng))
    if N == 1500:
        assert split[0][0] > 0
    if N == 40:
        assert split[0][1] > 0


@pytest.mark.gpu
def test_full_splat_zero_sigma():
    """An RBF of sigma 0 on a voxel gives NaN there and nothing elsewhere."""
    rng = np.random.default_rng(3)
    res = (9, 5, 7)
    rbf = _rbf(rng, 1, 40, 1)
    clean = rbf[:, :39].copy()
    rbf[0, 39] = (0.0, 0.0, 1.5, 0.0, 1.0)      # the grid's middle voxel
    G = rng.standard_normal((1, 2) + res).astype(np.float32)
    vol, _, _, _ = _calls(rbf, res, G, True)
    want = O.splat_forward(clean, res, VS, VE, mode=O.PURE64)
    at = np.zeros(res, bool)
    at[4, 2, 3] = True
    assert np.isnan(vol[0, :, at]).all()
    assert np.isfinite(vol[0, :, ~at]).all()
    assert rel_l2(vol[0][:, ~at], want[0][:, ~at]) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("ws", [True, False])
@pytest.mark.parametrize("at", [0, 300, 1499])
def test_full_splat_zero_sigma_split(at, ws):
    """The same where the RBFs are split over workgroups, in any split's chunks."""
    rng = np.random.default_rng(4)
    res = (13, 11, 9)
    rbf = _rbf(rng, 1, 1500, 1)
    rbf[0, at] = (0.0, 0.0, 1.5, 0.0, 1.0)      # the grid's middle voxel
    G = np.zeros((1, 2) + res, np.float32)
    vol, _, nf, _ = _calls(rbf, res, G, ws)
    assert (nf > 0) == ws
    want = O.splat_forward(np.delete(rbf, at, 1), res, VS, VE, mode=O.PURE64)
    mid = np.zeros(res, bool)
    mid[6, 5, 4] = True
    assert np.isnan(vol[0][:, mid]).all()
    assert rel_l2(vol[0][:, ~mid], want[0][:, ~mid]) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("A", [1, 3])
@pytest.mark.parametrize("big", [1.0, 1e3, 1e7])
def test_full_splat_grad_attribute_range(big, A):
    """An RBF's gradient does not suffer from the attribute of one out of its
    reach.  Tolerance per entry: 64 * 2^-24 of the sum of its terms' magnitudes
    (a weight's exponent carries four roundings of |k r^2| < 27, at most 75 *
    2^-24 and on average a few; products and sums the rest)."""
    rng = np.random.default_rng(6)
    res, N = (24, 20, 28), 30
    rbf = np.concatenate([rng.uniform(-0.7, 0.2, (N, 2)), rng.uniform(0.7, 1.6, (N, 1)),
                          rng.uniform(0.08, 0.12, (N, 1)), rng.uniform(0.5, 1.5, (N, A))], 1)
    rbf[17] = [0.95, 0.95, 2.45, 0.05] + [big] * A
    rbf = rbf.astype(np.float32)[None]
    G = rng.standard_normal((1, 1 + A) + res).astype(np.float32)
    vol, grad, _, _ = _calls(rbf, res, G, True)
    v64 = vol.astype(np.float64)
    ref = O.splat_grad(rbf, v64, G, VS, VE, mode=O.PURE64)[0]
    z, y, x = np.meshgrid(*(np.linspace(VS[2 - k], VE[2 - k], res[k]) for k in range(3)),
                          indexing="ij")
    inv = 1.0 / np.where(v64[0, 0] < 1e-8, 1.0, v64[0, 0])
    for i in range(N):
        if i == 17:
            continue
        px, py, pz, s, *a = rbf[0, i].astype(np.float64)
        d = np.stack([x - px, y - py, z - pz])
        r2 = (d ** 2).sum(0)
        g = np.exp(-0.5 * r2 / s ** 2)
        mag = np.abs(G[0, 0]) + sum(
            np.abs(G[0, 1 + k]) * inv * (abs(a[k]) + np.abs(v64[0, 1 + k])) for k in range(A))
        bound = [(mag * g * np.abs(d[k])).sum() / s ** 2 for k in range(3)]
        bound += [(mag * g * r2).sum() / s ** 3]
        bound += [(np.abs(G[0, 1 + k]) * inv * g).sum() for k in range(A)]
        assert (np.abs(grad[0, i] - ref[i]) <= 64 * 2.0 ** -24 * np.array(bound)).all(), i


@pytest.mark.gpu
def test_full_splat_large_plane():
    """2^28 voxels in one slice: more tiles than a launch's grid takes."""
    from totrilib_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(5)
    res = (1, 16384, 16384)
    rbf = _rbf(rng, 1, 3, 0)
    rbf[..., 2] = 0.5
    r = torch.from_numpy(rbf).cuda()
    vol = torch.full((1, 1) + res, -1.0, device="cuda")
    assert lib.totri_rbf2volume_gaussian_forward(
        r.data_ptr(), 1, 3, 0, vol.data_ptr(), *res, _lib.f3(VS), _lib.f3(VE), 0.0, None, 0,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert (vol >= 0).all()
    vox = np.concatenate([[0, 2 ** 28 - 1], rng.integers(0, 2 ** 28, 2000)])
    got = vol.flatten()[torch.from_numpy(vox).cuda()].cpu().numpy()
    ref = O.splat_forward(rbf, res, VS, VE, mode=O.PURE64, vox=vox)
    assert rel_l2(got, ref.reshape(-1)[vox]) < 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("N,A,res", [(40, 1, (2, 2, 300)), (33, 3, (1, 3, 130)),
                                     (5, 0, (2, 1, 1000)), (3, 8, (3, 20, 128))])
def test_full_splat_few_long_rows(N, A, res):
    """Grids of few rows: the gradient's rows are split along x, with a
    remainder of a chunk and of a step."""
    rng = np.random.default_rng(N)
    rbf = _rbf(rng, 1, N, A)
    G = rng.standard_normal((1, 1 + A) + res).astype(np.float32)
    ref = O.splat_forward(rbf, res, VS, VE, mode=O.PURE64)
    gref = O.splat_grad(rbf, ref, G, VS, VE, mode=O.PURE64)
    for ws in (True, False):
        vol, grad, _, _ = _calls(rbf, res, G, ws)
        assert rel_l2(vol, ref) < 1e-5
        assert rel_l2(grad, gref) < 1e-5
