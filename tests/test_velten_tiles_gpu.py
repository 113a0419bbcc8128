"""Velten backprojections (A2, A3) bit for bit against the FP32 oracle at the
edges of their tiling: units of up to sixteen (scan, laser) pairs (laser tiles
of equal size, one to three kept in registers, or recomputed above), stages of
LDS rows with and without a remainder, workgroups of 256 and of 1024 lanes,
points inside the box (no short root) and width / offset pairs whose quotient
rounds on bin edges.  Sums run in the reference's order, so equality is exact."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

VS, VE = (-1.0, -1.0, 0.5), (1.0, 1.0, 2.5)


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def points(rng, B, n, inside=False):
    z = np.full((B, n, 1), 1.0 if inside else 0.0)
    return np.concatenate([rng.uniform(-1, 1, (B, n, 2)), z], 2).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 16, 17, 25, 33, 48, 49])
@pytest.mark.parametrize("T", [96, 1000])
def test_velten_exhaustive_laser_tiles(L, T):
    from totrilib_amd.reconstruct import BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(100 + L)
    B, S, res = 2, 7, (5, 6, 11)
    w, off = 8.0 / T, 0.25
    scan, laser = points(rng, B, S), points(rng, B, L, inside=L % 2 == 1)
    lorg = (laser - np.array([0, 0, 1.0])).astype(np.float32) if L % 3 == 0 else None
    tr = rng.random((B, T, S, L)).astype(np.float32)
    got = BackprojectionExhaustiveVelten.apply(
        t(tr), t(scan), t(laser), VolumeDef(VS, VE, res), BinDef(w, off, T), None,
        None if lorg is None else t(lorg)).cpu().numpy()
    ref = O.velten_exhaustive(tr, scan, laser, None, lorg, res, VS, VE, w, off, mode=O.FP32)
    assert np.count_nonzero(ref) > 300
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("res", [(64, 48, 65), (3, 5, 7)])     # 1024 and 256 lanes
@pytest.mark.parametrize("S,T", [(1, 64), (9, 512), (21, 1500), (5, 3000)])
def test_velten_stages(res, S, T):
    from totrilib_amd.reconstruct import BackprojectionConfocalVelten, BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(S + T)
    w, off = 0.0078125 * 512 / T, 0.0
    scan, laser = points(rng, 1, S), points(rng, 1, 2)
    tr = rng.random((1, T, S, 2)).astype(np.float32)
    vd, bd = VolumeDef(VS, VE, res), BinDef(w, off, T)
    got = BackprojectionConfocalVelten.apply(t(tr[..., 0]), t(scan), vd, bd).cpu().numpy()
    ref = O.velten_confocal(tr[..., 0], scan, None, res, VS, VE, w, off, mode=O.FP32)
    assert ref.any()
    assert np.array_equal(got.astype(np.float64), ref)
    got = BackprojectionExhaustiveVelten.apply(t(tr), t(scan), t(laser), vd, bd).cpu().numpy()
    ref = O.velten_exhaustive(tr, scan, laser, None, None, res, VS, VE, w, off, mode=O.FP32)
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("L", [9, 10, 11, 12, 16, 17, 36])
@pytest.mark.parametrize("T", [1600, 1900, 2200, 2500])   # 11, 9, 8 and 7 rows to a stage
def test_velten_exhaustive_few_rows_per_stage(L, T):
    """Laser points in several tiles where a stage holds few rows."""
    from totrilib_amd.reconstruct import BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(L + T)
    S, res = 5, (5, 6, 11)
    scan, laser = points(rng, 1, S), points(rng, 1, L)
    tr = rng.random((1, T, S, L)).astype(np.float32)
    got = BackprojectionExhaustiveVelten.apply(
        t(tr), t(scan), t(laser), VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T)).cpu().numpy()
    ref = O.velten_exhaustive(tr, scan, laser, None, None, res, VS, VE, 8.0 / T, 0.0, mode=O.FP32)
    assert ref.any()
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("res,T,L", [((56, 56, 56), 640, 9), ((56, 56, 56), 700, 16),
                                     ((48, 48, 48), 1024, 9)])
def test_velten_exhaustive_smaller_stages(res, T, L):
    """Volumes of several workgroups per CU, whose stages are smaller."""
    from totrilib_amd.reconstruct import BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(T)
    scan, laser = points(rng, 1, 3), points(rng, 1, L)
    tr = rng.random((1, T, 3, L)).astype(np.float32)
    got = BackprojectionExhaustiveVelten.apply(
        t(tr), t(scan), t(laser), VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T)).cpu().numpy()
    ref = O.velten_exhaustive(tr, scan, laser, None, None, res, VS, VE, 8.0 / T, 0.0, mode=O.FP32)
    assert ref.any()
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 6, 7, 8, 13, 18])
def test_velten_exhaustive_rows_from_global_memory(L):
    """Rows longer than a stage: tiles of all laser points up to six, of 5 to 8
    points above."""
    from totrilib_amd.reconstruct import BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(L)
    S, T, res = 11, 19000, (5, 6, 11)
    scan, laser = points(rng, 1, S), points(rng, 1, L)
    tr = rng.random((1, T, S, L)).astype(np.float32)
    got = BackprojectionExhaustiveVelten.apply(
        t(tr), t(scan), t(laser), VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T)).cpu().numpy()
    ref = O.velten_exhaustive(tr, scan, laser, None, None, res, VS, VE, 8.0 / T, 0.0, mode=O.FP32)
    assert ref.any()
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("far", [np.inf, 1e20, 1e15])
@pytest.mark.parametrize("S,T", [(19, 64), (8, 3000)])
def test_velten_confocal_far_origin(S, T, far):
    """Origins without a bound on the path length: those scan points add
    nothing, whatever their place in the walk's groups."""
    from totrilib_amd.reconstruct import BackprojectionConfocalVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(S)
    res = (3, 5, 7)
    scan = points(rng, 1, S)
    origin = (scan - np.array([0, 0, 0.5])).astype(np.float32)
    origin[0, ::3, 0] = far
    origin[0, 4, 1] = -far
    tr = rng.random((1, T, S)).astype(np.float32)
    got = BackprojectionConfocalVelten.apply(
        t(tr), t(scan), VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T), t(origin)).cpu().numpy()
    ref = O.velten_confocal(tr, scan, origin, res, VS, VE, 8.0 / T, 0.0, mode=O.FP32)
    assert ref.any()
    assert np.array_equal(got.astype(np.float64), ref)


@pytest.mark.gpu
@pytest.mark.parametrize("res", [(1, 9, 8), (7, 1, 9), (6, 5, 1), (1, 1, 1), (1, 300, 400)])
@pytest.mark.parametrize("L", [1, 3, 8, 20])
@pytest.mark.parametrize("T", [50, 19000])
def test_velten_single_slices(res, L, T):
    """A grid of one voxel along an axis has NaN coordinates there, and a NaN
    path length lies in bin 0 (the conversion of NaN to int): every voxel adds
    bin 0 of all pairs, in their order."""
    from totrilib_amd.reconstruct import BackprojectionConfocalVelten, BackprojectionExhaustiveVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(L)
    S = 13
    scan, laser = points(rng, 1, S), points(rng, 1, L)
    tr = rng.random((1, T, S, L)).astype(np.float32)
    vd, bd = VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T)
    got = BackprojectionExhaustiveVelten.apply(t(tr), t(scan), t(laser), vd, bd)
    assert (got == float(np.add.accumulate(tr[0, 0].reshape(-1))[-1])).all()
    got = BackprojectionConfocalVelten.apply(t(tr[..., 0]), t(scan), vd, bd)
    assert (got == float(np.add.accumulate(tr[0, 0, :, 0])[-1])).all()


@pytest.mark.gpu
@pytest.mark.parametrize("S,T", [(19, 64), (16, 3000)])
def test_velten_confocal_nan_origin(S, T):
    """A NaN path length lies in bin 0, whatever the scan point's place in the
    walk's groups.  (Whole numbers: sums are exact in any order.)"""
    from totrilib_amd.reconstruct import BackprojectionConfocalVelten
    from totrilib_amd.types import BinDef, VolumeDef
    rng = np.random.default_rng(S)
    res = (3, 5, 7)
    scan = points(rng, 1, S)
    origin = (scan - np.array([0, 0, 0.5])).astype(np.float32)
    lost = np.arange(1, S, 4)
    origin[0, lost, 1] = np.nan
    tr = rng.integers(1, 50, (1, T, S)).astype(np.float32)
    got = BackprojectionConfocalVelten.apply(
        t(tr), t(scan), VolumeDef(VS, VE, res), BinDef(8.0 / T, 0.0, T), t(origin)).cpu().numpy()
    kept = np.setdiff1d(np.arange(S), lost)
    ref = O.velten_confocal(tr[..., kept], scan[:, kept], origin[:, kept], res, VS, VE, 8.0 / T,
                            0.0, mode=O.FP32)
    assert np.array_equal(got.astype(np.float64), ref + tr[0, 0, lost].sum())
