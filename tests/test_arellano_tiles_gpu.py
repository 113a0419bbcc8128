"""Ellipsoid backprojection at the edges of its kernel: column tiles of 64 with
a remainder and across rows, volumes past the LDS limit (256 rows), a single
entry, runs of one entry per scan/laser pair, coincident scan and laser
points, foci inside the box, boxes that most ellipsoids miss or that lie
behind the wall.  With a transient of ones every voxel counts its hits, which
must equal the oracle's FP32 decisions exactly."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,S,L,T,keep,vs,ve,w,off,same", [
    ((8, 8, 8), 3, 2, 120, 1.0, (-1, -1, 0.5), (1, 1, 2.5), 0.06, 0.0, False),
    ((16, 9, 7), 4, 3, 90, 0.3, (-1, -1, 0.5), (1, 1, 2.5), 0.08, 0.1, False),   # 63 columns
    ((5, 13, 5), 7, 1, 200, 0.01, (-1, -1, 0.5), (1, 1, 2.5), 0.04, 0.0, False),  # 65 columns
    ((260, 6, 6), 3, 2, 300, 0.2, (-1, -1, 0.5), (1, 1, 2.5), 0.025, 0.0, False),
    ((256, 8, 9), 2, 2, 300, 0.2, (-1, -1, 0.5), (1, 1, 2.5), 0.025, 0.0, False),
    ((12, 10, 70), 5, 5, 100, 0.5, (-1, -1, 0.5), (1, 1, 2.5), 0.07, 0.0, True),
    ((9, 11, 12), 4, 2, 150, 1.0, (-1, -1, -0.5), (1, 1, 1.5), 0.04, 0.0, False),  # foci inside
    ((9, 11, 12), 4, 2, 400, 1.0, (0.4, -0.1, 1.5), (0.6, 0.1, 1.6), 0.012, 0.0, False),
    ((10, 8, 8), 4, 2, 150, 1.0, (-1, -1, -2.5), (1, 1, -0.5), 0.05, 0.0, False),
    ((10, 8, 8), 4, 2, 150, 1.0, (-1, -1, 2.5), (1, 1, 0.5), 0.05, 0.0, False),   # reversed
    ((8, 8, 8), 1, 1, 40, 0.03, (-1, -1, 0.5), (1, 1, 2.5), 0.15, 0.0, True),
])
def test_hits_equal_the_oracle(res, S, L, T, keep, vs, ve, w, off, same):
    from totrilib_amd.reconstruct import BackprojectionExhaustiveArellano
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(S * T + res[0])
    scan = rng.uniform(-1, 1, (1, 3, S)).astype(np.float32)
    scan[:, 2] *= 0.01
    laser = rng.uniform(-1, 1, (1, 3, L)).astype(np.float32)
    laser[:, 2] *= 0.01
    if same:
        n = min(S, L)
        laser[:, :, :n] = scan[:, :, :n]
    tr = (rng.random((1, T, S, L)) < keep).astype(np.float32)
    vs, ve = tuple(map(float, vs)), tuple(map(float, ve))
    dev = torch.device("cuda:0")
    got = BackprojectionExhaustiveArellano.apply(
        torch.from_numpy(tr).to(dev), torch.from_numpy(scan).to(dev),
        torch.from_numpy(laser).to(dev), VolumeDef(vs, ve, res), BinDef(w, off, T))
    ref = O.arellano(tr, scan, laser, None, None, res, vs, ve, w, off, mode=O.FP32)
    got = got.detach().cpu().numpy().reshape(ref.shape)
    assert np.isfinite(ref).all()
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.parametrize("shift", [(3e3, -2e3, 1e3), (1e5, -1e5, 1e5), (1e6, 2e6, -1e6)])
@pytest.mark.parametrize("w", [0.06, 0.25])
def test_hits_far_from_the_origin(shift, w):
    """The formula rounds a pair's centre to the coordinates' spacing: no hit
    that this moves into a column is left out."""
    from totrilib_amd.reconstruct import BackprojectionExhaustiveArellano
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(int(abs(shift[0])))
    res, S, L, T = (9, 11, 12), 6, 3, int(9 / w)
    sh = np.array(shift)
    scan = (np.concatenate([rng.uniform(-1, 1, (1, 2, S)), np.zeros((1, 1, S))], 1)
            + sh[None, :, None]).astype(np.float32)
    laser = (np.concatenate([rng.uniform(-1, 1, (1, 2, L)), np.zeros((1, 1, L))], 1)
             + sh[None, :, None]).astype(np.float32)
    vs = tuple(float(v) for v in np.array([-1, -1, 0.5]) + sh)
    ve = tuple(float(v) for v in np.array([1, 1, 2.5]) + sh)
    tr = np.ones((1, T, S, L), np.float32)
    dev = torch.device("cuda:0")
    got = BackprojectionExhaustiveArellano.apply(
        torch.from_numpy(tr).to(dev), torch.from_numpy(scan).to(dev),
        torch.from_numpy(laser).to(dev), VolumeDef(vs, ve, res), BinDef(w, 0.0, T))
    ref = O.arellano(tr, scan, laser, None, None, res, vs, ve, w, 0.0, mode=O.FP32)
    got = got.detach().cpu().numpy().reshape(ref.shape)
    assert ref.any() and np.isfinite(ref).all()
    assert np.array_equal(got.astype(np.float64), ref)
