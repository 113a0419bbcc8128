"""float64 render and adjoint at the edges of their tiles (64 bins of a scan
point and 24 columns a round; 64 rows, 256 bins and three scan points a
round), bit for bit against the oracle's double dispatch."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu

ORIGIN, SIZE = (-1.0, -1.0, 0.5), (2.0, 2.0, 2.0)


def t64(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to("cuda:0")


@pytest.mark.parametrize("shape,n,T,w,off", [
    ((5, 7, 8), 1, 31, 0.1, 0.0),        # few bins: a lane per bin
    ((5, 5, 8), 3, 32, 0.1, 0.0),        # one partial tile, 25 columns
    ((4, 6, 7), 4, 64, 0.05, 0.01),      # 24 columns; few rows: a lane per voxel
    ((3, 4, 9), 5, 65, 0.05, 0.3),       # a second tile of one bin
    ((6, 5, 63), 4, 129, 0.025, 0.0),
    ((5, 10, 64), 6, 300, 0.011, 0.02),
    ((4, 5, 65), 7, 320, 0.011, 0.0),    # a second row tile of one voxel
    ((3, 3, 130), 2, 1500, 0.0021, 0.0),  # several 256-bin units per tile
    ((4, 4, 1), 3, 80, 0.04, 0.0),       # a single row: nothing is active
    ((4, 5, 20), 5, 330, 0.011, -0.4),   # radii of both signs
    ((4, 5, 20), 5, 200, -0.015, 3.1),   # radii that fall
])
@pytest.mark.parametrize("wall", ["flat", "inside"])
def test_render_and_adjoint_tiles(shape, n, T, w, off, wall):
    from totrilib_amd.totri_cpp.render import (volume_confocal_forward,
                                               volume_confocal_grad_volume)
    X, Y, Z = shape
    rng = np.random.default_rng(T + Z)
    vol = rng.standard_normal(shape)
    mp = rng.uniform(-1, 1, (3, n))
    mp[2] = 0.0 if wall == "flat" else rng.uniform(0.0, 3.0, n)  # some inside or past the box
    tr = torch.full((n, T), float("nan"), dtype=torch.float64, device="cuda:0")
    volume_confocal_forward(t64(vol), t64(mp), tr, ORIGIN, SIZE, w, off)
    assert np.array_equal(tr.cpu().numpy(), O.r1_forward_f64(vol, mp, T, ORIGIN, SIZE, w, off))
    G = rng.standard_normal((n, T))
    out = torch.full(shape, float("nan"), dtype=torch.float64, device="cuda:0")
    volume_confocal_grad_volume(out, t64(mp), t64(G), ORIGIN, SIZE, w, off)
    assert np.array_equal(out.cpu().numpy(),
                          O.a1_transpose_f64(G, mp, X, Y, Z, ORIGIN, SIZE, w, off))


@pytest.mark.parametrize("shape,n,T", [
    ((3, 4, 9), 10, 65),       # tiles from 640 samples on
    ((3, 4, 9), 9, 71),        # one sample fewer
    ((4, 5, 8), 20, 40),
    ((4, 4, 15), 30, 24),      # short tiles from 24 bins on
    ((4, 4, 15), 30, 23),
    ((4, 4, 16), 40, 16),
    ((6, 5, 63), 8, 129),
    ((5, 5, 8), 3, 320),
])
def test_adjoint_tiles_of_few_samples(shape, n, T):
    from totrilib_amd.totri_cpp.render import volume_confocal_grad_volume
    X, Y, Z = shape
    rng = np.random.default_rng(T + Z)
    mp = rng.uniform(-1, 1, (3, n))
    mp[2] = rng.uniform(-0.1, 0.1, n)
    G = rng.standard_normal((n, T))
    w = 3.3 / T
    out = torch.full(shape, float("nan"), dtype=torch.float64, device="cuda:0")
    volume_confocal_grad_volume(out, t64(mp), t64(G), ORIGIN, SIZE, w, 0.0)
    ref = O.a1_transpose_f64(G, mp, X, Y, Z, ORIGIN, SIZE, w, 0.0)
    assert ref.any() and np.array_equal(out.cpu().numpy(), ref)
