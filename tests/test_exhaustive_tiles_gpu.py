"""Exhaustive render adjoint (A5) against the FP64-summed oracle at the edges of
its forms: laser tiles of 1 to 8 points and several, scan points with and
without a remainder, spans of at most 2 and 6 bins (masked reads) and of
dozens (running sums), histograms that cut voxels off at both ends, rows too
long for a stage, 256 and 1024 lanes, and a gradient with an infinity.

Tolerance 1e-6 relative L2, that of the existing adjoint test: the oracle's
weights are the same FP32 numbers to an ulp of frac, summed in double; here a
voxel sums a few hundred pairs in float (2^-24 each, random signs)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from tests.cases import rel_l2

VS, VE = (-1.0, -1.0, 0.5), (1.0, 1.0, 2.5)


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def adjoint(G, res, scan, laser, w, off):
    from totrilib_amd.totri_cpp.render import volume_render_exhaustive_grad_volume
    B = G.shape[0]
    out = torch.empty((B,) + res, device="cuda")
    empty = torch.empty(B, 3, 0, device="cuda")
    volume_render_exhaustive_grad_volume(t(G), t(scan), t(laser), empty, empty, out, VS, VE, w, off)
    return out.cpu().numpy()


def points(rng, B, n):
    return np.concatenate([rng.uniform(-1, 1, (B, 2, n)), np.zeros((B, 1, n))], 1).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 7, 8, 9, 17])
@pytest.mark.parametrize("T,w,off,D", [
    (40, 0.2, 0.0, 20),      # spans within 2 bins
    (150, 0.05, 0.0, 20),    # within 6 bins
    (60, 0.05, 3.0, 20),     # cut off at both ends
    (700, 0.0115, 0.0, 6),   # dozens of bins
    (200, 0.0115, 3.5, 6),   # dozens, cut off
])
def test_adjoint_tiles(L, T, w, off, D):
    rng = np.random.default_rng(L + T)
    B, S, res = 2, 9, (D, 5, 7)
    scan, laser = points(rng, B, S), points(rng, B, L)
    G = rng.standard_normal((B, T, S, L)).astype(np.float32)
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, off, mode=O.PINNED64)
    assert ref.any()
    assert rel_l2(adjoint(G, res, scan, laser, w, off), ref) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("res", [(64, 48, 65), (5, 6, 7)])     # 1024 and 256 lanes
@pytest.mark.parametrize("T", [64, 1100, 2600, 9000])
def test_adjoint_stages(res, T):
    rng = np.random.default_rng(T)
    w = 8.0 / T
    scan, laser = points(rng, 1, 3), points(rng, 1, 2)
    G = rng.standard_normal((1, T, 3, 2)).astype(np.float32)
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64)
    assert rel_l2(adjoint(G, res, scan, laser, w, 0.0), ref) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("T,D", [(150, 20), (700, 6)])
def test_adjoint_infinite_gradient(T, D):
    """An infinity reaches the voxels whose spans hold its bin, and no others."""
    rng = np.random.default_rng(T)
    res, w = (D, 5, 7), 8.0 / T
    scan, laser = points(rng, 1, 3), points(rng, 1, 2)
    G = rng.standard_normal((1, T, 3, 2)).astype(np.float32)
    G[0, T // 2, 1, 1] = np.inf
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64)
    got = adjoint(G, res, scan, laser, w, 0.0)
    fine = np.isfinite(ref)
    assert 0 < np.count_nonzero(~fine) < fine.size
    assert np.array_equal(np.isfinite(got), fine)
    assert rel_l2(got[fine], ref[fine]) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("big", [1e8, 1e10, 1e14, 1e20, 3e38])
@pytest.mark.parametrize("T,D", [(150, 20), (700, 6), (2600, 6), (9000, 6)])
def test_adjoint_large_gradient(T, D, big):
    """A large finite bin costs the voxels whose spans do not hold it no accuracy."""
    rng = np.random.default_rng(T)
    res, w = (D, 5, 7), 8.0 / T
    scan, laser = points(rng, 1, 3), points(rng, 1, 2)
    G = rng.standard_normal((1, T, 3, 2)).astype(np.float32)
    G[0, T // 2, 1, 1] = np.inf
    clear = np.isfinite(O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64))
    G[0, T // 2, 1, 1] = big
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64)
    got = adjoint(G, res, scan, laser, w, 0.0)
    assert 0 < np.count_nonzero(~clear) < clear.size
    assert rel_l2(got[clear], ref[clear]) < 1e-6
    assert rel_l2(got, ref) < 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("T", [700, 2600])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 48])      # bin widths past DivConst's range
def test_adjoint_marked_rows(T, scale):
    """Batches without, with a few and with many rows of large range."""
    from totrilib_amd.totri_cpp.render import volume_render_exhaustive_grad_volume
    rng = np.random.default_rng(T)
    res, w = (6, 5, 7), 8.0 / T * scale
    VS, VE = ((-scale, -scale, 0.5 * scale), (scale, scale, 2.5 * scale))
    scan, laser = (points(rng, 3, n) * np.float32(scale) for n in (9, 5))
    G = rng.standard_normal((3, T, 9, 5)).astype(np.float32)
    clear = np.ones((3,) + res, bool)
    for b, pairs in ((1, [(8, 4)]), (2, [(s, l) for s in range(9) for l in range(3)])):
        for s, l in pairs:
            G[b, T // 2, s, l] = np.inf
    clear = np.isfinite(O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64))
    G[np.isinf(G)] = 1e15
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64)
    out = torch.empty((3,) + res, device="cuda")
    empty = torch.empty(3, 3, 0, device="cuda")
    volume_render_exhaustive_grad_volume(t(G), t(scan), t(laser), empty, empty, out, VS, VE, w, 0.0)
    got = out.cpu().numpy()
    for b in range(3):
        assert clear[b].any()
        assert rel_l2(got[b][clear[b]], ref[b][clear[b]]) < 1e-6
        assert rel_l2(got[b], ref[b]) < 1e-6


@pytest.mark.gpu
def test_adjoint_rows_past_two_to_the_31():
    """Eight rows of 1.6e8 bins each, whose running sums lie more than 2^31
    floats apart.  Row l holds l + 1 everywhere, so each of its spans averages
    to l + 1 (1e-5: spans of 2e7 bins, positions in float to 16 bins)."""
    from totrilib_amd.totri_cpp.render import volume_render_exhaustive_grad_volume
    rng = np.random.default_rng(1)
    T, L, res = 160_000_000, 8, (2, 2, 2)
    scan, laser = points(rng, 1, 1), points(rng, 1, L)
    G = torch.arange(1, L + 1, device="cuda", dtype=torch.float32).expand(1, T, 1, L).contiguous()
    out = torch.empty((1,) + res, device="cuda")
    empty = torch.empty(1, 3, 0, device="cuda")
    volume_render_exhaustive_grad_volume(G, t(scan), t(laser), empty, empty, out, VS, VE, 8.0 / T,
                                         0.0)
    assert (out / 36 - 1).abs().max() < 1e-5
    del G
    torch.cuda.empty_cache()


def _sizes(B, T, S, L, res, w):
    from totrilib_amd import _lib
    lib = _lib.load()
    return (lib.totri_volume_render_exhaustive_grad_volume_workspace(B, T, S, L),
            lib.totri_volume_render_exhaustive_grad_volume_workspace_box(
                B, T, S, L, *res, _lib.f3(VS), _lib.f3(VE), w))


@pytest.mark.parametrize("B,T,S,L", [(1, 512, 256, 16), (2, 1000, 33, 1), (1, 2000, 1024, 1000)])
def test_adjoint_scratch_sizes(B, T, S, L):
    """Four bytes per bin and the points' headers; running sums only for spans
    that need them."""
    n = 4 * B * T * S * L
    least, short = _sizes(B, T, S, L, (64, 8, 8), 4.0 / 64 / 4.0)
    assert n <= least == short <= n + 16 * B * S * L + 16 * B * (S + L) + 1024
    least, long = _sizes(B, T, S, L, (16, 8, 8), 4.0 / 16 / 40.0)
    assert 3 * n <= long <= 3 * n + 64 * B * S * L + 16 * B * (S + L) + 2048


@pytest.mark.gpu
@pytest.mark.parametrize("T,D", [(150, 20), (700, 6), (2600, 6), (9000, 6), (9000, 70)])
def test_adjoint_least_scratch(T, D):
    """With the first query's bytes, long spans add the bins."""
    from totrilib_amd import _lib
    lib = _lib.load()
    rng = np.random.default_rng(T)
    res, w = (D, 5, 7), 8.0 / T
    scan, laser = points(rng, 2, 9), points(rng, 2, 5)
    G = rng.standard_normal((2, T, 9, 5)).astype(np.float32)
    n = lib.totri_volume_render_exhaustive_grad_volume_workspace(2, T, 9, 5)
    g, s, l = t(G), t(scan), t(laser)
    out = torch.empty((2,) + res, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    for size in (n - 1, n):
        buf = torch.full((n + 4096,), 0xff, dtype=torch.uint8, device="cuda")
        got = lib.totri_volume_render_exhaustive_grad_volume(
            g.data_ptr(), 2, T, 9, 5, s.data_ptr(), l.data_ptr(), out.data_ptr(), *res,
            _lib.f3(VS), _lib.f3(VE), w, 0.0, buf.data_ptr(), size, st)
        assert (got == 0) == (size == n)
        assert (buf[n:] == 0xff).all()
    ref = O.r2_adjoint(G, res, scan, laser, VS, VE, w, 0.0, mode=O.PINNED64)
    assert rel_l2(out.cpu().numpy(), ref) < 1e-6
