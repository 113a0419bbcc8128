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
