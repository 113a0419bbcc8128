"""Rows of the confocal walks.

* The render and the scan-point gradient visit only the rows that a column's
  nonzero voxels reach, from 2^28 samples on: volumes whose occupied rows sit
  at the ends, in the middle, nowhere, or hold a NaN, against the oracle.
* A1's row walks settle a sample exactly only at the end of its row where one
  bin moves it by more than four guard widths, and at every sample otherwise:
  bin widths on both sides of that line, bit for bit against the oracle.
* Calls too small to fill the chip are split down to one mirror quad (pair) of
  scan points per range and to small column chunks: sizes around the limits.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.cases import ORIGIN, SIZE, rel_l2, wall_grid

pytestmark = pytest.mark.gpu

TOL = 1e-5


def dev():
    return torch.device("cuda:0")


@pytest.mark.parametrize("scan", ["mirror", "random"])
@pytest.mark.parametrize("fill", ["first", "last", "middle", "ends", "none", "nan"])
def test_occupied_rows(fill, scan):
    from totrilib_amd.totri_cpp.render import (volume_confocal_forward,
                                               volume_confocal_grad_measurement_points)
    X, Y, Z, T, w = 32, 32, 70, 1024, 0.003  # X Y N T = 2^28
    rng = np.random.default_rng(5)
    mp = wall_grid(16)
    if scan == "random":
        mp = np.stack([rng.uniform(-1, 1, 256), rng.uniform(-1, 1, 256),
                       rng.uniform(-0.1, 0.1, 256)]).astype(np.float32)
    vol = np.zeros((X, Y, Z), np.float32)
    rows = {"first": [0], "last": [Z - 1], "middle": [33], "ends": [0, Z - 1], "none": [],
            "nan": [33]}[fill]
    for z in rows:
        vol[::3, 1::2, z] = rng.random(vol[::3, 1::2, z].shape)
    if fill == "middle":
        vol[4, 4, 64:66] = -1.0
        vol[5, 5, :] = -0.0
    if fill == "nan":
        vol[7, 9, 40] = np.nan
    v = torch.from_numpy(vol).to(dev())
    m = torch.from_numpy(np.ascontiguousarray(mp)).to(dev())
    out = torch.full((256, T), float("nan"), device=dev())
    volume_confocal_forward(v, m, out, ORIGIN, SIZE, w, 0.0)
    G = rng.standard_normal((256, T)).astype(np.float32)
    gp = torch.full((3, 256), float("nan"), device=dev())
    volume_confocal_grad_measurement_points(gp, v, m, torch.from_numpy(G).to(dev()), ORIGIN,
                                            SIZE, w, 0.0)
    got, gotp = out.cpu().numpy(), gp.cpu().numpy()
    pts = (0, 100, 255)
    refp = np.zeros((3, 256))
    for i in pts:
        ref = O.r1_forward(vol, mp, T, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=i, i1=i + 1)[0]
        nan = np.isnan(ref)
        assert nan.any() == (fill == "nan") and np.isnan(got[i][nan]).all()
        ok = ~np.isnan(got[i])
        assert ok.any() and rel_l2(got[i][ok], ref[ok]) < TOL
        refp += O.a6(vol, mp, G, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=i, i1=i + 1)
    if fill == "nan":
        assert np.isnan(gotp[:, pts]).all()
    else:
        assert rel_l2(gotp[:, pts], refp[:, pts]) < TOL
    if fill == "none":
        assert not got.any() and not gotp.any()


@pytest.mark.parametrize("scan", ["quads", "random"])
@pytest.mark.parametrize("T", [600, 1500])
@pytest.mark.parametrize("w", [2e-4, 6e-4])
def test_a1_bins_within_the_guard(w, T, scan):
    """32 rows per metre 40 m away: the guard is 2.5e-3 rows, and a bin moves
    z_hat by 6.4e-3 or 1.9e-2 rows."""
    from totrilib_amd.totri_cpp.render import volume_confocal_grad_volume
    X, Y, Z = 8, 8, 64
    origin = (-1.0, -1.0, 40.0)
    off = 40.5
    rng = np.random.default_rng(3)
    mp = wall_grid(4)
    if scan == "random":
        mp = np.stack([rng.uniform(-1, 1, 16), rng.uniform(-1, 1, 16),
                       np.zeros(16)]).astype(np.float32)
    m = torch.from_numpy(np.ascontiguousarray(mp)).to(dev())
    cols = np.stack(np.meshgrid(np.arange(X), np.arange(Y), indexing="ij"), -1).reshape(-1, 2)
    n = 0
    for t in np.linspace(2, T - 1, 24).astype(int):
        s = int(rng.integers(0, 16))
        G = torch.zeros(16, T, device=dev())
        G[s, int(t)] = 1.0
        out = torch.full((X, Y, Z), float("nan"), device=dev())
        volume_confocal_grad_volume(out, m, G, origin, SIZE, w, off)
        got = out.cpu().numpy().astype(np.float64)
        idx = np.concatenate([np.full((len(cols), 1), s), np.full((len(cols), 1), t), cols], 1)
        zi, al, d2 = O.r1_decisions(idx, mp, X, Y, Z, origin, SIZE, w, off)
        act = (d2 > 0) & (zi >= 0) & (zi <= Z - 2)
        tc = float(np.float32(np.float32(t) * np.float32(w)) + np.float32(off))
        wgt = (np.sqrt(d2[act].astype(np.float64)) / (tc * tc)) ** 4
        a = al[act].astype(np.float64)
        cx, cy, z = cols[act, 0], cols[act, 1], zi[act]
        want = np.zeros((X, Y, Z))
        np.add.at(want, (cx, cy, z), (1 - a) * wgt)
        np.add.at(want, (cx, cy, z + 1), a * wgt)
        touched = np.zeros((X, Y, Z), bool)
        touched[cx, cy, z] = touched[cx, cy, z + 1] = True
        assert not ((got != 0) & ~touched).any()
        # alpha may differ by the guard's width (see the comment above)
        assert np.abs(got - want).max() <= 2.6e-3 * want.max()
        n += int(act.sum())
    assert n > 0


@pytest.mark.parametrize("shape,n,T", [
    ((8, 8, 8), 2, 64),       # one quad
    ((6, 4, 70), 4, 100),     # four quads, a partial tile, 9 slabs
    ((32, 32, 32), 16, 256),  # one quad per range
    ((20, 20, 20), 24, 200),  # 144 quads: ranges of one and two
    ((18, 7, 24), 8, 150),    # odd Y: pairs
    ((16, 16, 160), 8, 300),  # deep: chunks of few columns
])
def test_small_splits(shape, n, T):
    from totrilib_amd.totri_cpp.render import (volume_confocal_forward,
                                               volume_confocal_grad_volume)
    X, Y, Z = shape
    w = 3.0 / T
    rng = np.random.default_rng(n + T)
    mp = wall_grid(n)
    vol = rng.random(shape).astype(np.float32)
    G = rng.random((n * n, T)).astype(np.float32)
    m = torch.from_numpy(np.ascontiguousarray(mp)).to(dev())
    out = torch.full((n * n, T), float("nan"), device=dev())
    volume_confocal_forward(torch.from_numpy(vol).to(dev()), m, out, ORIGIN, SIZE, w, 0.0)
    gv = torch.full(shape, float("nan"), device=dev())
    volume_confocal_grad_volume(gv, m, torch.from_numpy(G).to(dev()), ORIGIN, SIZE, w, 0.0)
    ref = O.r1_forward(vol, mp, T, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64)
    refv = O.a1_transpose(G, mp, X, Y, Z, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64)
    assert rel_l2(out.cpu().numpy(), ref) < TOL
    assert rel_l2(gv.cpu().numpy(), refv) < TOL


def test_more_columns_than_a_launch_has_waves():
    """2^26 columns: the pass over the volume's columns fits a launch."""
    from totrilib_amd.totri_cpp.render import (volume_confocal_forward,
                                               volume_confocal_grad_measurement_points)
    X, Y, Z, N, T, w = 8192, 8192, 2, 2, 16, 0.25
    rng = np.random.default_rng(2)
    cols = np.stack([rng.integers(0, X, 50), rng.integers(0, Y, 50)], 1).astype(np.int32)
    cols[0], cols[1] = (0, 0), (X - 1, Y - 1)
    mp = rng.uniform(-1, 1, (3, N)).astype(np.float32)
    mp[2] = 0
    vol = np.zeros((X, Y, Z), np.float32)
    vol[cols[:, 0], cols[:, 1]] = rng.random((50, Z))
    v = torch.from_numpy(vol).to(dev())
    m = torch.from_numpy(mp).to(dev())
    out = torch.full((N, T), float("nan"), device=dev())
    volume_confocal_forward(v, m, out, ORIGIN, SIZE, w, 0.0)
    ref = O.r1_forward(vol, mp, T, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, cols=cols)
    assert ref.any() and rel_l2(out.cpu().numpy(), ref) < TOL
    gp = torch.full((3, N), float("nan"), device=dev())
    volume_confocal_grad_measurement_points(gp, v, m, torch.ones(N, T, device=dev()), ORIGIN, SIZE,
                                            w, 0.0)
    assert gp.isfinite().all() and gp.any()


@pytest.mark.parametrize("scan", ["mirror", "pairs", "random"])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_upstream_on_empty_rows(bad, scan):
    """A NaN or an infinity times an empty voxel is NaN in the scan-point
    gradient: of its own scan point, and of no other."""
    from totrilib_amd.totri_cpp.render import volume_confocal_grad_measurement_points
    X, Y, Z, T, w = 32, 32, 70, 1024, 0.003  # X Y N T = 2^28
    rng = np.random.default_rng(8)
    mp = wall_grid(16)
    if scan != "mirror":
        mp = np.stack([rng.uniform(-1, 1, 256), rng.uniform(-1, 1, 256),
                       np.zeros(256)]).astype(np.float32)
    if scan == "pairs":
        mp[:, 128:] = mp[:, :128] * np.array([[-1], [1], [1]], np.float32)
    vol = np.zeros((X, Y, Z), np.float32)
    vol[::3, 1::2, 5] = rng.random(vol[::3, 1::2, 5].shape)
    G = rng.standard_normal((256, T)).astype(np.float32)
    i = 37
    # the last bin at which a sample of scan point i is active lies on empty rows
    ones = O.r1_forward(np.ones_like(vol), mp, T, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=i,
                        i1=i + 1)[0]
    lit = O.r1_forward(vol, mp, T, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=i, i1=i + 1)[0]
    t = int(np.flatnonzero(ones)[-1])
    assert not lit[t - 64:].any()
    G[i, t] = bad
    gp = torch.full((3, 256), 7.0, device=dev())
    volume_confocal_grad_measurement_points(
        gp, torch.from_numpy(vol).to(dev()), torch.from_numpy(np.ascontiguousarray(mp)).to(dev()),
        torch.from_numpy(G).to(dev()), ORIGIN, SIZE, w, 0.0)
    got = gp.cpu().numpy()
    ref = O.a6(vol, mp, G, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=i, i1=i + 1)
    assert np.isnan(ref[:, i]).all()
    assert np.isnan(got[:, i]).all()
    others = np.arange(256) != i
    assert np.isfinite(got[:, others]).all()
    pts = (0, 127, 200, 255)
    refp = sum(O.a6(vol, mp, G, ORIGIN, SIZE, w, 0.0, mode=O.PINNED64, i0=k, i1=k + 1) for k in pts)
    assert rel_l2(got[:, pts], refp[:, pts]) < TOL
