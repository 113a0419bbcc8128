// Backprojections for gfx950: Velten confocal (A2), Velten exhaustive (A3)
// and Arellano ellipsoid splatting (A4).
//
// Reference: src/reconstruct/backprojection_cuda.cu:10-322,
//            src/reconstruct/backprojection.cpp:7-49.
//
// Every discrete decision (the nearest bin of a path length, the voxel an
// ellipsoid hit falls into) follows the reference's FP32 formula with IEEE
// correctly rounded square roots and divisions, no contraction, and
// norm3df(d) restated as sqrt((dx*dx + dy*dy) + dz*dz).
//
// A2/A3 (gathers): one lane per voxel, flat over [D][H][W] so that volume
// writes are coalesced.  The transient is first transposed so that each scan
// point's (and laser point's) bins are contiguous; a workgroup then stages the
// rows of a group of scan points in LDS and every lane gathers its bin from
// there.  Sums run over scan (and laser) points in the reference's order.
//
// A4 (scatter): the positive bins of the transient are first listed in
// (scan, laser, bin) order (stream compaction) and the list is split into
// chunks.  A wave owns 64 volume columns (x, y) and one chunk; the columns'
// D voxels are accumulated in LDS slots owned by their lanes (row-major
// [D][64]), so the reference's global atomics become plain read-modify-
// writes; list entries are uniform across the wave.  Chunks write partial
// volumes that are summed in chunk order.
#include <math.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "compact.h"
#include "stage.h"

namespace totri_hip {
namespace {

// Blocks of a grid-stride loop over n elements (capped).
int grid1d(size_t n, int block = 256) {
  size_t b = (n + block - 1) / block;
  if (b > 65535 * 4) b = 65535 * 4;
  return (int)(b < 1 ? 1 : b);
}

// Blocks of a one-lane-per-element launch over n < 2^31 elements (uncapped).
unsigned blocks_for(size_t n, int block = 256) {
  const size_t b = (n + block - 1) / block;
  return (unsigned)(b < 1 ? 1 : b);
}

// out[b][c][ooff + r] = in[b][r][c] for a [B][R][C] array, out rows of
// stride ldo (tiled through LDS).
__global__ void transpose_kernel(const float* __restrict__ in, float* __restrict__ out,
                                 int R, int C, int ldo, int ooff) {
  __shared__ float tile[32][33];
  const int b = blockIdx.z;
  const float* src = in + (size_t)b * R * C;
  float* dst = out + (size_t)b * C * ldo + ooff;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  for (int k = threadIdx.y; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + threadIdx.x;
    if (r < R && c < C) tile[k][threadIdx.x] = src[(size_t)r * C + c];
  }
  __syncthreads();
  for (int k = threadIdx.y; k < 32; k += 8) {
    const int c = c0 + k, r = r0 + threadIdx.x;
    if (r < R && c < C) dst[(size_t)c * ldo + r] = tile[threadIdx.x][k];
  }
}

int launch_transpose(const float* in, float* out, int B, int R, int C, hipStream_t st) {
  return transpose_batched(in, out, B, R, C, st);
}

struct BoxGeom {
  int B, D, H, W, T;
  float sx, sy, sz, ex, ey, ez;
  float w, off;
};

// Nearest bin of a path length (backprojection_cuda.cu:187,279):
// floorf((dist - offset) / width + 0.5f).
__device__ __forceinline__ int nearest_bin(float dist, float w, float off) {
  float tf = (dist - off) / w;
  tf = tf + 0.5f;
  return (int)floorf(tf);
}

// ---------------------------------------------------------------------------
// A2: vol[b][z][y][x] = sum_s tr[b][t(s)][s],
// t = nearest_bin(2 |p_s - o_s| + 2 |p_s - q|)       (backprojection_cuda.cu:152-194)
//
// A cheap estimate of the bin's argument (hardware square root, one FMA with
// precomputed constants) decides wherever its distance to the next bin edge
// exceeds a bound on its error; the few samples nearer to an edge take the
// reference's formula.  That is the exact decision, with no correctly rounded
// root or division for most (voxel, scan point) pairs, and one gather a pair.
// (Correcting the estimate with two thresholds of a table per scan point
// needs no bound but three gathers, and the thresholds a kernel of their own:
// 0.38 ms at 64^3 voxels, 32 x 32 points, 512 bins, against 0.165 ms.)
// ---------------------------------------------------------------------------

// The exact bin of squared distance e for a scan point whose origin term is
// dso2 = 2 |p_s - o_s| (0 without an origin): backprojection_cuda.cu:177-187.
__device__ __forceinline__ int velten_bin(float e, float dso2, float w, float off) {
  const float dsv = sqrt_rn(e);
  const float dist = dso2 + 2.f * dsv;
  return nearest_bin(dist, w, off);
}

// Workspace of A2: a header of 8 floats per scan point,
//   {x, y, z, c, dso2, half, 0, 0}: the estimate is fma(sqrt(e), 2/w, c),
//   c = ((dso2 - off) * (1/w)) + 0.5, and decides where its fraction lies
//   within `half` of 1/2; c is NaN where no bound holds (every pair of that
//   point takes the formula); x is NaN where every path length is (the formula
//   puts those into bin 0, DivConst does not: a NaN squared distance keeps to the
//   formula's own division),
// then one row of nv floats per scan point: bin t at t, a zero at T (nv = T + 1
// rounded up to a multiple of 4).
constexpr int kVeltenHead = 8;

__host__ __device__ __forceinline__ int velten_row(int T) { return (T + 4) & ~3; }

// Estimate error: the exact chain rounds five times (root, sum, difference,
// quotient, + 0.5) and the estimate about eight times (hardware root within
// 1 ulp, 1/w, 2/w, the constant's three roundings, the FMA), each a relative
// error of at most 2^-24 (2^-23 for the root) of a term no larger than M bins,
// M = (2 d_max + |dso2| + |off|) / w + 1 with d_max the largest distance from
// the scan point to the box's corners.  The two differ by under 16 * 2^-24 * M
// bins; the guard takes 17, and M < 2^16 keeps it below 1/14 of a bin.
constexpr float kVeltenMaxBins = 65536.f;
constexpr float kVeltenGuard = 17.f * 0x1p-24f;

// One thread per scan point: its header and the zero slot of its row.
__global__ __launch_bounds__(256) void velten_head_kernel(
    const float* __restrict__ scan, const float* __restrict__ orig, BoxGeom g, int S, int So,
    float rw, float* __restrict__ head, float* __restrict__ rows) {
  const int nv = velten_row(g.T);
  const size_t bs = (size_t)blockIdx.x * blockDim.x + threadIdx.x;  // b * S + s
  if (bs >= (size_t)g.B * S) return;
  const int b = (int)(bs / S), s = (int)(bs - (size_t)b * S);
  const float* p = scan + bs * 3;
  const float px = p[0], py = p[1], pz = p[2];
  float dso = 0.f;
  if (So > 0) {
    const float* o = orig + ((size_t)b * So + s) * 3;
    dso = dist3(px, py, pz, o[0], o[1], o[2]);                               // :178-183
  }
  const float dso2 = 2.f * dso;
  // the largest distance to the box is at a corner
  float dmax = 0.f;
  for (int c = 0; c < 8; ++c)
    dmax = fmaxf(dmax, dist3(px, py, pz, (c & 1) ? g.ex : g.sx, (c & 2) ? g.ey : g.sy,
                             (c & 4) ? g.ez : g.sz));
  const float m = (2.f * dmax + fabsf(dso2) + fabsf(g.off)) / g.w + 1.f;
  const bool est = g.w > 0.f && m < kVeltenMaxBins;  // false for NaN or inf
  float4* h = (float4*)(head + bs * kVeltenHead);
  h[0] = make_float4(isnan(dso2 - g.off) ? __builtin_nanf("") : px, py, pz,
                     est ? (dso2 - g.off) * rw + 0.5f : __builtin_nanf(""));
  h[1] = make_float4(dso2, est ? 0.5f - kVeltenGuard * m : 0.f, 0.f, 0.f);
  rows[bs * nv + g.T] = 0.f;
}

__device__ __forceinline__ float velten_sqdist(float px, float py, float pz, float qx, float qy,
                                               float qz) {
  const float dx = px - qx, dy = py - qy, dz = pz - qz;
  float e = dx * dx;
  e = e + dy * dy;
  e = e + dz * dz;
  return e;
}

// Whether an estimate r lies too near a bin edge to decide (also NaN, inf).
__device__ __forceinline__ bool velten_near(float r, float half) {
  return !(fabsf(__builtin_amdgcn_fractf(r) - 0.5f) <= half);
}

// Slot of bin t: bins outside [0, T) read the zero at T.
__device__ __forceinline__ unsigned velten_slot(int t, int T) {
  return min((unsigned)t, (unsigned)T);
}

// One lane per voxel, flat over [D][H][W].  The rows of R scan points at a
// time are staged in LDS (STAGED), or read from global memory (rows too long
// for the stage).  The headers are uniform and come through the scalar cache.
// Sums run over scan points in order, as the reference's loop.
template <bool STAGED, int NTH>
__global__ __launch_bounds__(NTH) void velten_confocal_kernel(
    const float* __restrict__ head, const float* __restrict__ rows, float* __restrict__ vol,
    BoxGeom g, int S, int R, int cap, float k2, DivConst dw) {
  constexpr int UN = 8;  // scan points at a time
  extern __shared__ float4 lds4[];
  const int T = g.T;
  const int nv = velten_row(T);
  const int b = blockIdx.y;
  const int nvox = g.D * g.H * g.W;
  const int v = blockIdx.x * NTH + threadIdx.x;
  const bool ok = v < nvox;
  const int vv = ok ? v : 0;
  const int x = vv % g.W;
  const int y = (vv / g.W) % g.H;
  const int z = vv / (g.W * g.H);
  const float qx = inclusive_coord(x, g.W, g.sx, g.ex);
  const float qy = inclusive_coord(y, g.H, g.sy, g.ey);
  const float qz = inclusive_coord(z, g.D, g.sz, g.ez);
  const size_t bS = (size_t)b * S;
  float* stage = (float*)lds4;
  RowStage<NTH> next;
  auto load = [&](int s0) { next.load(rows + (bS + s0) * nv, min(R, S - s0) * nv / 4); };
  if (STAGED) {
    load(0);
    next.store(stage, min(R, S) * nv / 4);
    if (R < S) load(R);
    __syncthreads();
  }
  float value = 0.f;
  int cur = 0;
  for (int s0 = 0; s0 < S; s0 += R) {
    const int ns = min(R, S - s0);
    const float* base = STAGED ? stage + cur * cap : rows + (bS + s0) * nv;
    if (STAGED && s0 + R < S) {
      next.store(stage + (cur ^ 1) * cap, min(R, S - s0 - R) * nv / 4);
      if (s0 + 2 * R < S) load(s0 + 2 * R);
    }
    // UN points at a time: their decisions and gathers overlap, their values
    // are added in point order.  (No short-circuit in the guard test: a branch
    // per point serialises the scalar loads, 0.35 ms.)
    const float* h = head + (bS + s0) * kVeltenHead;
    int k = 0;
    for (; k + UN <= ns; k += UN, h += UN * kVeltenHead) {
      float px[UN], py[UN], pz[UN], c[UN], dso2[UN], half[UN];
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        px[u] = h[u * kVeltenHead];
        py[u] = h[u * kVeltenHead + 1];
        pz[u] = h[u * kVeltenHead + 2];
        c[u] = h[u * kVeltenHead + 3];
        dso2[u] = h[u * kVeltenHead + 4];
        half[u] = h[u * kVeltenHead + 5];
      }
      float e[UN], a[UN];
      int t[UN];
      bool near = false;
#pragma unroll
      for (int u = 0; u < UN; ++u) {
        e[u] = velten_sqdist(px[u], py[u], pz[u], qx, qy, qz);
        const float r = __builtin_fmaf(sqrt_fast(e[u]), k2, c[u]);
        t[u] = floor_to_int(r);
        near |= velten_near(r, half[u]);
      }
      if (near) {
#pragma unroll
        for (int u = 0; u < UN; ++u)
          if (velten_near(__builtin_fmaf(sqrt_fast(e[u]), k2, c[u]), half[u]))
            t[u] = sqrt_mid_range(e[u]) && dw.ok
                       ? floor_to_int(div_const(dso2[u] + 2.f * sqrt_rn_mid(e[u]) - g.off, dw) +
                                      0.5f)
                       : velten_bin(e[u], dso2[u], g.w, g.off);              // :177,185-187
      }
#pragma unroll
      for (int u = 0; u < UN; ++u) a[u] = base[(k + u) * nv + velten_slot(t[u], T)];
#pragma unroll
      for (int u = 0; u < UN; ++u) value += a[u];                            // :188-190
    }
    for (; k < ns; ++k, h += kVeltenHead) {
      const float e = velten_sqdist(h[0], h[1], h[2], qx, qy, qz);
      const int t = velten_bin(e, h[4], g.w, g.off);
      value += base[k * nv + velten_slot(t, T)];
    }
    if (STAGED) {
      __syncthreads();  // these rows are no longer read, the next are written
      cur ^= 1;
    }
  }
  if (ok) vol[(size_t)b * nvox + v] = value;                                 // :192
}

// ---------------------------------------------------------------------------
// A3: vol = sum_{s,l} tr[b][t(s,l)][s][l],
// t = nearest_bin(|p_s - o_s| + |p_s - q| + |p_l - q| + |p_l - o_l|)
// (backprojection_cuda.cu:228-287)
//
// The path length D is computed as the reference does (correctly rounded
// roots, sums in its order).  Its two roots belong to the voxel and one
// point each, so a lane computes |p_s - q| once per scan point, and keeps the
// distances to up to sixteen laser points in registers for the whole call.
// A pair is then two sums, a difference, the correctly rounded division by
// the bin width as four multiply-adds (DivConst), + 0.5, floor and one
// gather: about 13 vector instructions, which set its time.  64^3 voxels,
// 256 x 16 points, 512 bins: 0.60 ms, against 1.76 ms with two roots and a
// table correction (three gathers) per pair.
// ---------------------------------------------------------------------------

// Workspace of A3: headers of 8 floats per scan point, then per laser point,
//   {x, y, z, |p - o|, reach, mid, 0, 0}: reach bounds |p - o| + |p - q| over
//   the box (+inf for NaN), mid is 1 where every squared distance to the box
//   lies in [2^-64, 2^64] (the short correctly rounded root serves),
// then one row per pair r = s * L + l as in A2 (velten_row).

// Thread i of batch b: header i (scan points, then laser points), and the
// zero slot of row i.
__global__ __launch_bounds__(256) void velten_ex_head_kernel(
    const float* __restrict__ scan, const float* __restrict__ laser,
    const float* __restrict__ sorig, const float* __restrict__ lorig, BoxGeom g, int S, int L,
    int So, int Lo, float* __restrict__ head, float* __restrict__ rows) {
  const int nv = velten_row(g.T);
  const int b = blockIdx.y;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (size_t)S * L) rows[((size_t)b * S * L + i) * nv + g.T] = 0.f;
  if (i >= (size_t)S + L) return;
  const bool is_scan = i < (size_t)S;
  const size_t k = is_scan ? (size_t)b * S + i : (size_t)b * L + (i - S);
  const float* p = (is_scan ? scan : laser) + k * 3;
  const float px = p[0], py = p[1], pz = p[2];
  float o = 0.f;
  if ((is_scan ? So : Lo) > 0) {
    const float* q = (is_scan ? sorig : lorig) + k * 3;
    o = dist3(px, py, pz, q[0], q[1], q[2]);                                 // :256-261,269-274
  }
  float d = 0.f;
  bool nan = !(px == px) || !(py == py) || !(pz == pz);
  for (int c = 0; c < 8; ++c)
    d = fmaxf(d, dist3(px, py, pz, (c & 1) ? g.ex : g.sx, (c & 2) ? g.ey : g.sy,
                       (c & 4) ? g.ez : g.sz));
  const float reach = o + d;
  nan = nan || !(reach == reach);
  // at least 2^-20 from the box and at most 2^30 from its far corners
  const float lo = box_sqdist(px, py, pz, g.sx, g.sy, g.sz, g.ex, g.ey, g.ez);
  const bool mid = !nan && lo >= 0x1p-40f && d <= 0x1p30f;
  float4* h = (float4*)(head + ((size_t)b * (S + L) + i) * kVeltenHead);
  h[0] = make_float4(px, py, pz, o);
  h[1] = make_float4(nan ? INFINITY : reach, mid ? 1.f : 0.f, 0.f, 0.f);
}

// |p - q| of N points with headers at h (uniform), every stride-th float: one
// uniform test for all, so that the header loads are in flight together.
template <int N, typename At>
__device__ __forceinline__ void ex_head_dists(At at, float qx, float qy, float qz, float (&d)[N]) {
  float mid = 1.f;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    d[j] = velten_sqdist(at(j)[0], at(j)[1], at(j)[2], qx, qy, qz);
    mid = fminf(mid, at(j)[5]);
  }
  if (mid != 0.f) {
#pragma unroll
    for (int j = 0; j < N; ++j) d[j] = sqrt_rn_mid(d[j]);                    // :255,268
  } else {
#pragma unroll
    for (int j = 0; j < N; ++j) d[j] = sqrt_rn(d[j]);
  }
}

// A unit of the exhaustive walk: SG scan points and a tile of KT laser points,
// up to sixteen pairs whose decisions and gathers overlap (eight: 0.79 ms at
// the size above), or up to eight where the stage does not hold sixteen rows.  Several scan points only where
// one tile holds all laser points (KT = L).
__host__ __device__ constexpr int ex_scan_group(int KT, int pairs) {
  return KT <= 6 ? (pairs / KT > 1 ? pairs / KT : 1) : 1;
}

// One lane per voxel, flat over [D][H][W].  The rows of U consecutive units
// are staged in LDS (STAGED), or read from global memory (long rows).  NTL:
// tiles whose distances stay in registers (L <= NTL * KT), or 0 (computed per
// unit).  Sums run over pairs in the reference's order (scan point outer,
// laser point inner).
template <int KT, int NTL, int SG, bool STAGED, int NTH>
__global__ __launch_bounds__(NTH) void velten_exhaustive_kernel(
    const float* __restrict__ head, const float* __restrict__ rows, float* __restrict__ vol,
    BoxGeom g, int S, int L, int U, int cap, DivConst dw) {
  extern __shared__ float4 lds4[];
  const int T = g.T;
  const int nv = velten_row(T);
  const int b = blockIdx.y;
  const int nvox = g.D * g.H * g.W;
  const int v = blockIdx.x * NTH + threadIdx.x;
  const bool ok = v < nvox;
  const int vv = ok ? v : 0;
  const int x = vv % g.W;
  const int y = (vv / g.W) % g.H;
  const int z = vv / (g.W * g.H);
  const float qx = inclusive_coord(x, g.W, g.sx, g.ex);
  const float qy = inclusive_coord(y, g.H, g.sy, g.ey);
  const float qz = inclusive_coord(z, g.D, g.sz, g.ez);
  // A grid of one voxel along an axis has no coordinate there (0 / 0): its path
  // lengths are NaN, which the formula puts into bin 0.
  const float reach0 = isnan(qx + qy + qz) ? INFINITY : fabsf(g.off);
  const float* hs = head + (size_t)b * (S + L) * kVeltenHead;
  const float* hl = hs + (size_t)S * kVeltenHead;
  const float* rb = rows + (size_t)b * S * L * nv;
  const int NT = (L + KT - 1) / KT;  // 1 where SG > 1
  const int n_units = (S + SG - 1) / SG * NT;
  // first row of unit u <= n_units
  auto unit_row = [&](int u) { return min(u / NT * SG, S) * L + u % NT * KT; };

  float dl[NTL > 0 ? NTL : 1][KT];
  float reach[NTL > 0 ? NTL : 1];
  auto laser_tile = [&](int k, float (&d)[KT], float& rch) {
    rch = 0.f;
    auto at = [&](int j) { return hl + min(k * KT + j, L - 1) * kVeltenHead; };
    ex_head_dists<KT>(at, qx, qy, qz, d);
#pragma unroll
    for (int j = 0; j < KT; ++j) rch = fmaxf(rch, at(j)[4]);
  };
#pragma unroll
  for (int k = 0; k < NTL; ++k) laser_tile(k, dl[k], reach[k]);

  float* stage = (float*)lds4;
  RowStage<NTH> next;
  auto unit_n4 = [&](int u0) { return (unit_row(min(u0 + U, n_units)) - unit_row(u0)) * nv / 4; };
  auto load = [&](int u0) { next.load(rb + (size_t)unit_row(u0) * nv, unit_n4(u0)); };
  if (STAGED) {
    load(0);
    next.store(stage, unit_n4(0));
    if (U < n_units) load(U);
    __syncthreads();
  }

  float value = 0.f, as[SG], rs = 0.f;
  // One unit: scan points s .. s + SG - 1 (as: |p - o| + |p - q| of each, rs:
  // their largest reach), tile k, its rows at base.
  auto unit = [&](const float* base, int s, int k, const float (&d)[KT], float rch) {
    const int ns = min(SG, S - s), nl = min(KT, L - k * KT);
    const float* h = hl + k * KT * kVeltenHead;
    float lo[KT];
#pragma unroll
    for (int j = 0; j < KT; ++j) lo[j] = h[min(j, nl - 1) * kVeltenHead + 3];
    float dist[SG][KT];
#pragma unroll
    for (int i = 0; i < SG; ++i)
#pragma unroll
      for (int j = 0; j < KT; ++j) {
        dist[i][j] = as[i] + d[j];                                           // :276-277
        dist[i][j] = dist[i][j] + lo[j];
      }
    // false for NaN or inf; uniform
    if (dw.ok && (rs + rch + reach0) * dw.hi < kVeltenMaxBins) {
      unsigned at[SG][KT];
#pragma unroll
      for (int i = 0; i < SG; ++i)
#pragma unroll
        for (int j = 0; j < KT; ++j)
          at[i][j] = velten_slot(floor_to_int(div_const(dist[i][j] - g.off, dw) + 0.5f), T);  // :279
      if (ns == SG && nl == KT) {
        float a[SG][KT];
        const float* row = base;
#pragma unroll
        for (int i = 0; i < SG; ++i)
#pragma unroll
          for (int j = 0; j < KT; ++j, row += nv) a[i][j] = row[at[i][j]];
#pragma unroll
        for (int i = 0; i < SG; ++i)
#pragma unroll
          for (int j = 0; j < KT; ++j) value += a[i][j];                     // :280-282
      } else {
#pragma unroll
        for (int i = 0; i < SG; ++i)
#pragma unroll
          for (int j = 0; j < KT; ++j)
            if (i < ns && j < nl) value += base[(i * nl + j) * nv + at[i][j]];
      }
    } else {
#pragma unroll
      for (int i = 0; i < SG; ++i)
#pragma unroll
        for (int j = 0; j < KT; ++j)
          if (i < ns && j < nl)
            value += base[(i * nl + j) * nv +
                          velten_slot(nearest_bin(dist[i][j], g.w, g.off), T)];
    }
  };

  int s = 0, k = 0;  // the next unit's first scan point and tile
  int cur = 0;
  for (int u0 = 0; u0 < n_units; u0 += U) {
    const int ue = min(u0 + U, n_units);
    const float* base = STAGED ? stage + cur * cap : rb + (size_t)unit_row(u0) * nv;
    if (STAGED && ue < n_units) {
      next.store(stage + (cur ^ 1) * cap, unit_n4(ue));
      if (ue + U < n_units) load(ue + U);
    }
    for (int u = u0; u < ue; ++u) {
      if (k == 0) {
        rs = 0.f;
        auto at = [&](int i) { return hs + (size_t)min(s + i, S - 1) * kVeltenHead; };
        ex_head_dists<SG>(at, qx, qy, qz, as);
#pragma unroll
        for (int i = 0; i < SG; ++i) {
          as[i] = at(i)[3] + as[i];                                          // :276-277
          rs = fmaxf(rs, at(i)[4]);
        }
      }
      if constexpr (NTL == 0) {
        laser_tile(k, dl[0], reach[0]);
        unit(base, s, k, dl[0], reach[0]);
      } else if constexpr (NTL == 1) {
        unit(base, s, 0, dl[0], reach[0]);
      } else {
#pragma unroll
        for (int c = 0; c < NTL; ++c)
          if (k == c) unit(base, s, c, dl[c], reach[c]);
      }
      base += (size_t)(min(SG, S - s) * min(KT, L - k * KT)) * nv;
      if (++k == NT) {
        k = 0;
        s += SG;
      }
    }
    if (STAGED) {
      __syncthreads();  // these rows are no longer read, the next are written
      cur ^= 1;
    }
  }
  if (ok) vol[(size_t)b * nvox + v] = value;                                 // :285
}

// ---------------------------------------------------------------------------
// A4: Arellano ellipsoid backprojection (backprojection_cuda.cu:10-115).
// ---------------------------------------------------------------------------
// Geometry of one scan/laser pair (backprojection_cuda.cu:51-74), shared by
// all of the pair's bins.
struct EllPair {
  float sd, ld, len, nx, ny, nz, cx, cy, cz;
};

__device__ __forceinline__ EllPair ell_pair(const float* sb, const float* lb,
                                            const float* sob, const float* lob, int S,
                                            int L, int So, int Lo, int s, int l) {
  EllPair e;
  const float spx = sb[s], spy = sb[S + s], spz = sb[2 * S + s];
  const float lpx = lb[l], lpy = lb[L + l], lpz = lb[2 * L + l];
  e.sd = So > 0 ? dist3(spx, spy, spz, sob[s], sob[So + s], sob[2 * So + s]) : 0.f;
  e.ld = Lo > 0 ? dist3(lpx, lpy, lpz, lob[l], lob[Lo + l], lob[2 * Lo + l]) : 0.f;
  e.cx = 0.5f * (spx + lpx);
  e.cy = 0.5f * (spy + lpy);
  e.cz = 0.5f * (spz + lpz);
  float nx = spx - lpx, ny = spy - lpy, nz = spz - lpz;                      // :62-66
  float ls = nx * nx;
  ls = ls + ny * ny;
  ls = ls + nz * nz;
  e.len = sqrt_rn(ls);                                                       // :67
  if (e.len > 1.e-6f) {                                                      // :68-70
    const float inv = 1.f / e.len;
    nx = inv * nx;
    ny = inv * ny;
    nz = inv * nz;
  }
  e.nx = nx;
  e.ny = ny;
  e.nz = nz;
  return e;
}

// The value lane `l` (uniform) holds.
__device__ __forceinline__ float readlane_f(float v, int l) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), l));
}

// One wave: columns tile*64 .. tile*64+63 of batch b, list chunk `chunk` of
// n_chunks.  dst is the chunk's partial volume [B][D][H][W] (written).
//
// Bound by the VALU issue of the per-column formula and the latency of its
// chain (the column accumulators in LDS leave two waves per SIMD at 64 rows).
// What depends on the bin alone -- its index split, value, radii, one root, one
// quotient and its pair's geometry -- is computed for 64 list entries at once, a
// lane each, and handed out by readlane; entries whose ellipsoid misses the
// wave's columns are left out there; two entries of one scan/laser pair then
// go together, so their chains overlap.  Roots and quotients of values in the
// middle of the range take the short correctly rounded forms; other values
// send the entry through the full ones (same results).  16^2 scan and 4^2
// laser points, 512 bins, 5 % positive, 64^3 voxels: 2.04 -> 0.87 ms (1.27
// without leaving entries out).
template <bool IN_LDS>
__global__ __launch_bounds__(64) void arellano_kernel(
    const float* __restrict__ trT,     // [B][S][L][T]
    const int* __restrict__ list,      // [B][S*L*T] positive bins, in order
    const int* __restrict__ totals,    // [B]
    const float* __restrict__ scan,    // [B][3][S]
    const float* __restrict__ laser,   // [B][3][L]
    const float* __restrict__ sorig,   // [B][3][So]
    const float* __restrict__ lorig,   // [B][3][Lo]
    float* __restrict__ dst,           // [n_chunks][B][D][H][W]
    BoxGeom g, int S, int L, int So, int Lo, int n_chunks) {
  extern __shared__ float colacc[];    // [D][64] when IN_LDS
  const int lane = threadIdx.x;
  const int chunk = blockIdx.y;
  const int b = blockIdx.z;
  const int ncol = g.H * g.W;
  const int v = blockIdx.x * 64 + lane;
  const bool ok = v < ncol;
  const int vv = ok ? v : 0;
  const int xi = vv % g.W, yi = vv / g.W;                                    // :27-28
  const float xf = inclusive_coord(xi, g.W, g.sx, g.ex);                     // :29-30
  const float yf = inclusive_coord(yi, g.H, g.sy, g.ey);                     // :31-32
  float* gcol = dst + ((size_t)chunk * g.B + b) * g.D * ncol + vv;           // stride ncol
  if (IN_LDS) {
    for (int z = 0; z < g.D; ++z) colacc[z * 64 + lane] = 0.f;
  } else if (ok) {
    for (int z = 0; z < g.D; ++z) gcol[(size_t)z * ncol] = 0.f;
  }
  const int n_elem = S * L * g.T;
  const int total = totals[b];
  const int per = (total + n_chunks - 1) / n_chunks;
  const int k0 = chunk * per, k1 = min(total, k0 + per);
  const int* lb_list = list + (size_t)b * n_elem;
  const float* tb = trT + (size_t)b * n_elem;
  const float* sb = scan + (size_t)b * 3 * S;
  const float* lb = laser + (size_t)b * 3 * L;
  const float* sob = sorig + (size_t)b * 3 * So;
  const float* lob = lorig + (size_t)b * 3 * Lo;
  const float depth = (float)g.D;
  // The box of this wave's columns, a row longer at either end (a hit's row is
  // rounded to the nearest, and row 0 takes what lies up to a row before it).
  float bx0 = ok ? xf : INFINITY, bx1 = ok ? xf : -INFINITY;
  float by0 = ok ? yf : INFINITY, by1 = ok ? yf : -INFINITY;
  for (int m = 1; m < 64; m <<= 1) {
    bx0 = fminf(bx0, __shfl_xor(bx0, m));
    bx1 = fmaxf(bx1, __shfl_xor(bx1, m));
    by0 = fminf(by0, __shfl_xor(by0, m));
    by1 = fmaxf(by1, __shfl_xor(by1, m));
  }
  const float row_z = 2.f * fabsf(g.ez - g.sz) / depth;
  const float bz0 = fminf(g.sz, g.ez) - row_z, bz1 = fmaxf(g.sz, g.ez) + row_z;
  const float box_far = fmaxf(fmaxf(fmaxf(fabsf(bx0), fabsf(bx1)), fmaxf(fabsf(by0), fabsf(by1))),
                              fmaxf(fabsf(bz0), fabsf(bz1)));
  // Smallest and largest distance of (px, py, pz) to the box, added; the largest
  // coordinate.
  auto box_reach = [&](float px, float py, float pz, float* lo, float* hi, float* far) {
    const float ax = fmaxf(fmaxf(bx0 - px, px - bx1), 0.f), cx = fmaxf(px - bx0, bx1 - px);
    const float ay = fmaxf(fmaxf(by0 - py, py - by1), 0.f), cy = fmaxf(py - by0, by1 - py);
    const float az = fmaxf(fmaxf(bz0 - pz, pz - bz1), 0.f), cz = fmaxf(pz - bz0, bz1 - pz);
    *lo += sqrt_fast(ax * ax + ay * ay + az * az);
    *hi += sqrt_fast(cx * cx + cy * cy + cz * cz);
    *far = fmaxf(fmaxf(*far, fabsf(px)), fmaxf(fabsf(py), fabsf(pz)));
  };
  float nx = 0.f, ny = 0.f, nz = 0.f;
  float rsx = 0.f, rsy = 0.f, rsz = 0.f, rez = 0.f, dps = 0.f, dpe = 0.f;

  // The row of one entry in this lane's column, -1 for none; k1m = r1/r0 - 1
  // and r1q = r1^2 are the entry's.  MID: *out tells that a root or quotient
  // leaves the range of the short forms.
  auto row_of = [&](float k1m, float r1q, auto mid, bool* out) {
    constexpr bool MID = decltype(mid)::value;
    const float ks = k1m * dps;                                              // :87
    const float stx = rsx + ks * nx, sty = rsy + ks * ny, stz = rsz + ks * nz;
    const float ke = k1m * dpe;                                              // :88
    const float etx = rsx + ke * nx, ety = rsy + ke * ny, etz = rez + ke * nz;
    float dx = etx - stx, dy = ety - sty, dz = etz - stz;                    // :89
    float rl = dx * dx;
    rl = rl + dy * dy;
    rl = rl + dz * dz;
    const float rlen = MID ? sqrt_rn_mid(rl) : sqrt_rn(rl);                  // :90
    const float ir = MID ? recip_rn_mid(rlen) : 1.f / rlen;                  // :91
    dx = ir * dx;
    dy = ir * dy;
    dz = ir * dz;
    float v0 = dx * stx;                                                     // :93
    v0 = v0 + dy * sty;
    v0 = v0 + dz * stz;
    float ss = stx * stx;
    ss = ss + sty * sty;
    ss = ss + stz * stz;
    float v1 = v0 * v0 - (ss - r1q);                                         // :94
    const bool hit = (v1 > 0.f) & ok;                                        // :95
    if (MID) {
      const float other = hit ? v1 : rl;
      *out = !(fminf(rl, other) >= 0x1p-64f && fmaxf(rl, other) <= 0x1p64f);
    }
    v1 = MID ? sqrt_rn_mid(v1) : sqrt_rn(v1);
    float d = -v0 - v1;
    d = d < 0.f ? -v0 + v1 : d;                                              // :97-100
    float bf = MID ? div_recip_mid(d, rlen, ir) : d / rlen;
    bf = bf * depth;
    bf = bf + 0.5f;
    const int row = (int)bf;                                                 // :101-102
    return hit & (row >= 0) & (row < g.D) ? row : -1;
  };

  for (int base = k0; base < k1; base += 64) {
    const int n = min(64, k1 - base);
    // lane j: entry base + j
    const int idx = lb_list[base + min(lane, n - 1)];
    const float value = tb[idx];                                             // > 0 (:77)
    const int pair = idx / g.T;                                              // s * L + l
    const int s = pair / L;
    const EllPair e = ell_pair(sb, lb, sob, lob, S, L, So, Lo, s, pair - s * L);
    float tc = (float)(idx - pair * g.T) * g.w;                              // :79-80
    tc = tc + g.off;
    tc = tc - e.sd;
    tc = tc - e.ld;
    const float r0 = tc / 2.f;                                               // :83
    float r1s = r0 * r0;
    r1s = r1s - (e.len * e.len) / 4.f;                                       // :84
    const float r1 = sqrt_rn(r1s);
    const float k1m = r1 / r0 - 1.f;                                         // :85
    const float r1q = tc > e.len ? r1 * r1 : -INFINITY;                      // :81: no hit
    // An ellipsoid that stays clear of the box hits no column of it.  Its points
    // have distance sums tc, which the formula's roundings move.  (u = 2^-24; hi
    // is the box's largest sum, and r1^2 >= 10^-3 hi^2.)  r1^2 is the rest of
    // r0^2 - len^2 / 4: 3 u r0^2 / r1^2 < 2e-4 of it.  A line that passes the
    // sphere outside counts as a hit within about 8 u hi^2 of r1^2: 5e-4 of it.
    // Both scale the ellipsoid by under 4e-4, the sums of its points by 8e-4.  Where
    // a line touches the sphere the root carries that error over as up to 7e-4 hi
    // along the column, 1.4e-3 hi in the sums: 4e-3 hi holds both.  The pair's
    // centre is rounded to u of the coordinates, in three axes, which moves a sum
    // by under 4 u of the largest coordinate; 1e-6 of it is left.
    float lo = 0.f, hi = 0.f, far = box_far;
    const int l = pair - s * L;
    box_reach(sb[s], sb[S + s], sb[2 * S + s], &lo, &hi, &far);
    box_reach(lb[l], lb[L + l], lb[2 * L + l], &lo, &hi, &far);
    const float slack = 4e-3f * hi + 1e-6f * far;
    const bool clear = !(tc > e.len) || (r1q >= 1e-3f * hi * hi &&
                                         (tc < lo - slack || tc > hi + slack));
    unsigned long long todo = __ballot(lane < n && !clear);
    auto entries = [&](const int* j, auto count) {
      constexpr int U = decltype(count)::value;
      int row[U];
      bool out = false;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        bool o;
        row[u] = row_of(readlane_f(k1m, j[u]), readlane_f(r1q, j[u]), std::true_type{}, &o);
        out |= o;
      }
      if (__ballot(out) != 0) {
        for (int u = 0; u < U; ++u)
          row[u] = row_of(readlane_f(k1m, j[u]), readlane_f(r1q, j[u]), std::false_type{},
                          nullptr);
      }
      // :103-109: the interpolation weight is int - int = 0, so only the row
      // itself receives the value.
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float add = readlane_f(value, j[u]);
        if (row[u] >= 0) {
          if (IN_LDS)
            colacc[row[u] * 64 + lane] += add;
          else
            gcol[(size_t)row[u] * ncol] += add;
        }
      }
    };
    int cur = -1;
    while (todo != 0) {
      int j[2];
      j[0] = (int)__builtin_ctzll(todo);
      todo &= todo - 1;
      const int p = __builtin_amdgcn_readlane(pair, j[0]);
      if (p != cur) {
        cur = p;
        nx = readlane_f(e.nx, j[0]);
        ny = readlane_f(e.ny, j[0]);
        nz = readlane_f(e.nz, j[0]);
        const float cz = readlane_f(e.cz, j[0]);
        rsx = xf - readlane_f(e.cx, j[0]);                                   // :72, :74
        rsy = yf - readlane_f(e.cy, j[0]);
        rsz = g.sz - cz;
        rez = g.ez - cz;
        dps = rsx * nx;
        dps = dps + rsy * ny;
        dpe = dps + rez * nz;
        dps = dps + rsz * nz;
      }
      j[1] = todo != 0 ? (int)__builtin_ctzll(todo) : 63;
      if (todo != 0 && __builtin_amdgcn_readlane(pair, j[1]) == p) {
        todo &= todo - 1;
        entries(j, std::integral_constant<int, 2>{});
      } else {
        entries(j, std::integral_constant<int, 1>{});
      }
    }
  }
  if (IN_LDS && ok)
    for (int z = 0; z < g.D; ++z) gcol[(size_t)z * ncol] = colacc[z * 64 + lane];
}

__global__ void zero_kernel(float* __restrict__ out, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x)
    out[e] = 0.f;
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// out[e] = sum over parts p of part[p * n + e], in part order.
__global__ void sum_parts_kernel(const float* __restrict__ part, int n_parts, size_t n,
                                 float* __restrict__ out) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x) {
    float v = part[e];
    for (int p = 1; p < n_parts; ++p) v += part[(size_t)p * n + e];
    out[e] = v;
  }
}

BoxGeom box_geom(int64_t B, int64_t D, int64_t H, int64_t W, int64_t T,
                 const float* vs, const float* ve, float w, float off) {
  BoxGeom g;
  g.B = (int)B;
  g.D = (int)D;
  g.H = (int)H;
  g.W = (int)W;
  g.T = (int)T;
  g.sx = vs[0];
  g.sy = vs[1];
  g.sz = vs[2];
  g.ex = ve[0];
  g.ey = ve[1];
  g.ez = ve[2];
  g.w = w;
  g.off = off;
  return g;
}

int check_dims(std::initializer_list<int64_t> dims, int64_t elems_limit_a, int64_t elems_limit_b) {
  for (int64_t d : dims)
    TOTRI_CHECK_ARG(d >= 0 && d < (1ll << 31), "dimension out of range");
  TOTRI_CHECK_ARG(elems_limit_a < (1ll << 31) && elems_limit_b < (1ll << 31),
                  "tensor has more than 2^31 elements");
  return TOTRI_OK;
}

}  // namespace

int transpose_strided(const float* in, float* out, int B, int R, int C, int ldo, int ooff,
                      hipStream_t st) {
  dim3 grid((C + 31) / 32, (R + 31) / 32, B);
  hipLaunchKernelGGL(transpose_kernel, grid, dim3(32, 8), 0, st, in, out, R, C, ldo, ooff);
  return check_launch("transpose_kernel");
}

int transpose_batched(const float* in, float* out, int B, int R, int C, hipStream_t st) {
  return transpose_strided(in, out, B, R, C, R, 0, st);
}

}  // namespace totri_hip

using namespace totri_hip;

namespace totri_hip {
namespace {

// Scratch that A2 asks for, per scan point: room for two floats per bin,
// which bounds what the allocation-free entry point takes.  Its headers and
// rows need about half of it.
size_t velten_bytes(int64_t B, int64_t T, int64_t S) {
  const size_t len = 4 + (((size_t)T + 5) & ~(size_t)3) + (((size_t)T + 6) & ~(size_t)3);
  return align256((size_t)B * S * len * sizeof(float));
}

}  // namespace
}  // namespace totri_hip

extern "C" size_t totri_backprojection_confocal_velten_workspace(int64_t B, int64_t T,
                                                                 int64_t S) {
  if (B <= 0 || T < 0 || S <= 0) return 0;
  return totri_hip::velten_bytes(B, T, S);
}

namespace totri_hip {
namespace {

// A2 with its scratch (a header and a row of the transient per scan point)
// supplied by the caller: the workspace of the entry point below, or the
// library's own array for the allocation-free variant.
int velten_confocal(const float* transient, int64_t B, int64_t T, int64_t S,
                    const float* scan_points, const float* scan_origin, int64_t So,
                    float* volume, int64_t D, int64_t H, int64_t W,
                    const float volume_start[3], const float volume_end[3], float bin_width,
                    float bin_offset, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_dims({B, T, S, So, D, H, W}, B * T * S, B * D * H * W);
  if (rc) return rc;
  TOTRI_CHECK_ARG(So == 0 || So == S, "scan_origin must have 0 or S points");
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  TOTRI_CHECK_ARG(T < (1 << 30), "T=%lld too large", (long long)T);
  hipStream_t st = (hipStream_t)stream;
  const size_t nvox = (size_t)D * H * W;
  if (B == 0 || nvox == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume != nullptr, "null volume");
  const BoxGeom g = box_geom(B, D, H, W, T, volume_start, volume_end, bin_width, bin_offset);
  if (T == 0 || S == 0) {  // no bins or no scan points: a zero volume
    hipLaunchKernelGGL(zero_kernel, dim3(grid1d(B * nvox)), dim3(256), 0, st, volume,
                       (size_t)B * nvox);
    return check_launch("zero_kernel");
  }
  TOTRI_CHECK_ARG(transient && scan_points, "null input");
  TOTRI_CHECK_ARG(So == 0 || scan_origin, "null scan_origin");
  const size_t need = velten_bytes(B, T, S);
  if (workspace_bytes < need)
    return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", need,
                workspace_bytes);
  TOTRI_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace & 15) == 0,
                  "workspace must be a non-null, 16-byte aligned device pointer");
  // headers, then rows: 8 + nv floats per scan point, of the 4 + nv + nt
  // (nt >= 4) asked for
  float* head = (float*)workspace;
  float* rows = head + (size_t)B * S * kVeltenHead;
  const int nv = velten_row((int)T);
  rc = transpose_strided(transient, rows, (int)B, (int)T, (int)S, nv, 0, st);
  if (rc) return rc;
  const float rw = 1.f / bin_width;
  hipLaunchKernelGGL(velten_head_kernel, dim3((unsigned)((B * S + 255) / 256)), dim3(256), 0, st,
                     scan_points, scan_origin, g, (int)S, (int)So, rw, head, rows);
  rc = check_launch("velten_head_kernel");
  if (rc) return rc;
  // Scan points per LDS stage: whole groups of eight.  Where fewer rows fit (T
  // above 2,300 bins, or 840 to 1,280 for volumes of several workgroups per CU) the
  // stage's barriers would come every few points: the rows are then read from
  // global memory, through the caches.
  const StagePlan sp = stage_plan(B, (int64_t)nvox);
  const int R = (sp.cap / nv) & ~7;
  const float k2 = 2.f * rw;
  const bool wide = sp.threads == 1024;
  auto kernel = R == 0 ? velten_confocal_kernel<false, 256>
                : wide ? velten_confocal_kernel<true, 1024>
                       : velten_confocal_kernel<true, 256>;
  const int threads = R > 0 ? sp.threads : 256;
  rc = allow_stage(kernel);
  if (rc) return rc;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(nvox, threads), (unsigned)B), dim3(threads),
                     R > 0 ? 2 * (size_t)sp.cap * sizeof(float) : 0, st, head, rows, volume, g,
                     (int)S, R > 0 ? R : (int)S, sp.cap, k2, make_div_const(g.w));
  return check_launch("velten_confocal_kernel");
}

// Scratch of the allocation-free A2.
// Every device that runs the library holds its own copy of this array, at
// its own address, until the process ends.  Host code never passes the
// array's name to a kernel (on the host it only stands for the symbol): it
// uses the device address that hipGetSymbolAddress returns, kept per device.
constexpr size_t kNoAllocScratchBytes = size_t(64) << 20;
__device__ __align__(256) float scratch[kNoAllocScratchBytes / sizeof(float)];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices];  // per device, resolved on its first call

// The current device's address of `scratch`, resolved once per device with
// that device current.
int scratch_address(void** out) {
  int dev = 0;
  TOTRI_CHECK_HIP(hipGetDevice(&dev));
  TOTRI_CHECK_ARG(dev >= 0 && dev < kMaxDevices, "device %d beyond the %d supported", dev,
                  kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(TOTRI_EHIP, "hipGetSymbolAddress(scratch) on device %d failed: %s", dev,
                  hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return TOTRI_OK;
}

}  // namespace
}  // namespace totri_hip

extern "C" int totri_backprojection_confocal_velten_forward(
    const float* transient, int64_t B, int64_t T, int64_t S, const float* scan_points,
    const float* scan_origin, int64_t So, float* volume, int64_t D, int64_t H, int64_t W,
    const float volume_start[3], const float volume_end[3], float bin_width,
    float bin_offset, void* workspace, size_t workspace_bytes, void* stream) {
  return totri_hip::velten_confocal(transient, B, T, S, scan_points, scan_origin, So, volume, D,
                                    H, W, volume_start, volume_end, bin_width, bin_offset,
                                    workspace, workspace_bytes, stream);
}

extern "C" size_t totri_backprojection_confocal_velten_noalloc_max_bytes(void) {
  return totri_hip::kNoAllocScratchBytes;
}

extern "C" int totri_backprojection_confocal_velten_forward_noalloc(
    const float* transient, int64_t B, int64_t T, int64_t S, const float* scan_points,
    const float* scan_origin, int64_t So, float* volume, int64_t D, int64_t H, int64_t W,
    const float volume_start[3], const float volume_end[3], float bin_width,
    float bin_offset, void* stream) {
  using namespace totri_hip;
  TOTRI_CHECK_ARG(B >= 0 && T >= 0 && S >= 0, "negative dimension");
  const size_t need = totri_backprojection_confocal_velten_workspace(B, T, S);
  if (need > kNoAllocScratchBytes)
    return fail(TOTRI_EINVAL,
                "transient of %zu bytes (B=%lld T=%lld S=%lld) exceeds the %zu-byte scratch of "
                "the allocation-free backprojection; use "
                "totri_backprojection_confocal_velten_forward with a workspace",
                need, (long long)B, (long long)T, (long long)S, kNoAllocScratchBytes);
  void* ws = nullptr;
  int rc = scratch_address(&ws);
  if (rc) return rc;
  return velten_confocal(transient, B, T, S, scan_points, scan_origin, So, volume, D, H, W,
                         volume_start, volume_end, bin_width, bin_offset, ws,
                         kNoAllocScratchBytes, stream);
}

namespace totri_hip {
namespace {

// Workspace of A3: the point headers, then the pair rows [B][S*L][nv].
struct ExLayout {
  size_t rows_off, end;
};

ExLayout ex_layout(int64_t B, int64_t T, int64_t S, int64_t L) {
  ExLayout l;
  l.rows_off = align256((size_t)B * (S + L) * kVeltenHead * sizeof(float));
  l.end = l.rows_off + align256((size_t)B * S * L * velten_row((int)T) * sizeof(float));
  return l;
}

template <int KT, int NTL, int SG>
int launch_velten_ex(const float* head, const float* rows, float* volume, const BoxGeom& g,
                     int64_t S, int64_t L, const StagePlan& sp, hipStream_t st) {
  const int nv = velten_row(g.T);
  const int64_t NT = (L + KT - 1) / KT;
  // Units per LDS stage: whole scan points, else one tile of a scan point.
  int64_t U = 1;
  if (SG * L * nv <= sp.cap)
    U = std::min<int64_t>((S + SG - 1) / SG, sp.cap / (SG * L * nv)) * NT;
  auto kernel = sp.threads == 1024 ? velten_exhaustive_kernel<KT, NTL, SG, true, 1024>
                                   : velten_exhaustive_kernel<KT, NTL, SG, true, 256>;
  const int rc = allow_stage(kernel);
  if (rc) return rc;
  hipLaunchKernelGGL(kernel, dim3(blocks_for((size_t)g.D * g.H * g.W, sp.threads), (unsigned)g.B),
                     dim3(sp.threads), 2 * (size_t)sp.cap * sizeof(float), st, head, rows, volume,
                     g, (int)S, (int)L, (int)U, sp.cap, make_div_const(g.w));
  return check_launch("velten_exhaustive_kernel");
}

// The tile size for L laser points, tiles of at most 16 points and `most`
// rows: tiles of equal size, rounded up to one that is compiled.  A tile
// that is not full masks its last points.  Tiles of up to six points belong to
// calls whose laser points make exactly one (their units take several scan
// points); several tiles have seven points or more, also where that masks more
// of the last.  Where a stage holds fewer than eight rows for them, rows from
// global memory are faster (56^3 voxels, 64 x 9 pairs, 900 bins: 0.33 ms with
// tiles of seven staged rows).
int velten_ex_tile(int64_t L, int64_t most) {
  static const int sizes[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16};
  int top = 0;
  for (int k : sizes)
    if (k <= most) top = k;
  if (top == 0 || (L > top && top < 8)) return 0;
  const int64_t nt = (L + top - 1) / top;
  int64_t kt = (L + nt - 1) / nt;
  if (nt > 1 && kt < 7) kt = 7;  // top >= 8 here
  for (int k : sizes)
    if (k >= kt) return k;
  return 0;
}

int velten_ex(const float* head, const float* rows, float* volume, const BoxGeom& g, int64_t S,
              int64_t L, hipStream_t st) {
  const size_t nvox = (size_t)g.D * g.H * g.W;
  const StagePlan sp = stage_plan(g.B, (int64_t)nvox);
  const int64_t fit = sp.cap / velten_row(g.T);
  int kt = velten_ex_tile(L, fit);
  const int pairs = ex_scan_group(kt > 0 ? kt : 1, 16) * (int64_t)kt <= fit ? 16 : 8;
  if (kt > 0 && ex_scan_group(kt, pairs) * (int64_t)kt > fit) kt = 0;
  if (kt == 0) {  // rows longer than the stage: read from global memory
    // up to six laser points: one tile, eight pairs a unit; else tiles of 5 to
    // 8 points, the size that masks fewest
    kt = (int)L;
    if (L > 6) {
      kt = 8;
      for (int k = 7; k >= 5; --k)
        if ((L + k - 1) / k * k < (L + kt - 1) / kt * kt) kt = k;
    }
    const int64_t sg = L > 6 ? 1 : ex_scan_group(kt, 8);
    const int64_t units = (S + sg - 1) / sg * ((L + kt - 1) / kt);
#define TOTRI_EXG(KT, NTL, SG) \
  if (kt == KT && (L <= 6) == (NTL == 1)) kernel = velten_exhaustive_kernel<KT, NTL, SG, false, 256>;
    auto kernel = velten_exhaustive_kernel<8, 0, 1, false, 256>;
    TOTRI_EXG(1, 1, ex_scan_group(1, 8)) TOTRI_EXG(2, 1, ex_scan_group(2, 8))
    TOTRI_EXG(3, 1, ex_scan_group(3, 8)) TOTRI_EXG(4, 1, ex_scan_group(4, 8))
    TOTRI_EXG(5, 1, 1) TOTRI_EXG(6, 1, 1)
    TOTRI_EXG(5, 0, 1) TOTRI_EXG(6, 0, 1) TOTRI_EXG(7, 0, 1)
#undef TOTRI_EXG
    hipLaunchKernelGGL(kernel, dim3(blocks_for(nvox), (unsigned)g.B), dim3(256), 0, st, head,
                       rows, volume, g, (int)S, (int)L, (int)units, 0, make_div_const(g.w));
    return check_launch("velten_exhaustive_kernel");
  }
  const int64_t nt = (L + kt - 1) / kt;
#define TOTRI_EX(KT, NTL) \
  if (kt == KT && (nt > 3 ? 0 : nt) == NTL) \
    return launch_velten_ex<KT, NTL, 1>(head, rows, volume, g, S, L, sp, st);
#define TOTRI_EX4(KT) TOTRI_EX(KT, 1) TOTRI_EX(KT, 2) TOTRI_EX(KT, 3) TOTRI_EX(KT, 0)
#define TOTRI_EX1(KT) \
  if (kt == KT && nt == 1) \
    return pairs == 16 ? launch_velten_ex<KT, 1, ex_scan_group(KT, 16)>(head, rows, volume, g, S, L, sp, st) \
                       : launch_velten_ex<KT, 1, ex_scan_group(KT, 8)>(head, rows, volume, g, S, L, sp, st);
  TOTRI_EX1(1) TOTRI_EX1(2) TOTRI_EX1(3) TOTRI_EX1(4) TOTRI_EX1(5) TOTRI_EX1(6)
  TOTRI_EX4(7) TOTRI_EX4(8) TOTRI_EX4(10) TOTRI_EX4(12) TOTRI_EX4(14) TOTRI_EX4(16)
#undef TOTRI_EX1
#undef TOTRI_EX4
#undef TOTRI_EX
  return fail(TOTRI_EINVAL, "no kernel for %lld tiles of %d laser points", (long long)nt, kt);
}

}  // namespace
}  // namespace totri_hip

extern "C" size_t totri_backprojection_exhaustive_velten_workspace(int64_t B, int64_t T,
                                                                   int64_t S, int64_t L) {
  if (B <= 0 || T < 0 || S <= 0 || L <= 0) return 0;
  return totri_hip::ex_layout(B, T, S, L).end;
}

extern "C" int totri_backprojection_exhaustive_velten_forward(
    const float* transient, int64_t B, int64_t T, int64_t S, int64_t L,
    const float* scan_points, const float* laser_points, const float* scan_origin,
    int64_t So, const float* laser_origin, int64_t Lo, float* volume, int64_t D, int64_t H,
    int64_t W, const float volume_start[3], const float volume_end[3], float bin_width,
    float bin_offset, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_dims({B, T, S, L, So, Lo, D, H, W}, B * T * S * L, B * D * H * W);
  if (rc) return rc;
  TOTRI_CHECK_ARG(So == 0 || So == S, "scan_origin must have 0 or S points");
  TOTRI_CHECK_ARG(Lo == 0 || Lo == L, "laser_origin must have 0 or L points");
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  TOTRI_CHECK_ARG(T < (1 << 30), "T=%lld too large", (long long)T);
  hipStream_t st = (hipStream_t)stream;
  const size_t nvox = (size_t)D * H * W;
  if (B == 0 || nvox == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume != nullptr, "null volume");
  const BoxGeom g = box_geom(B, D, H, W, T, volume_start, volume_end, bin_width, bin_offset);
  if (T == 0 || S == 0 || L == 0) {  // no bins or no pairs: a zero volume
    hipLaunchKernelGGL(zero_kernel, dim3(grid1d(B * nvox)), dim3(256), 0, st, volume,
                       (size_t)B * nvox);
    return check_launch("zero_kernel");
  }
  TOTRI_CHECK_ARG(transient && scan_points && laser_points, "null input");
  TOTRI_CHECK_ARG((So == 0 || scan_origin) && (Lo == 0 || laser_origin), "null origin");
  const ExLayout lay = ex_layout(B, T, S, L);
  if (workspace_bytes < lay.end)
    return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", lay.end,
                workspace_bytes);
  TOTRI_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace & 15) == 0,
                  "workspace must be a non-null, 16-byte aligned device pointer");
  float* head = (float*)workspace;
  float* rows = (float*)((char*)workspace + lay.rows_off);
  const int nv = velten_row((int)T);
  rc = transpose_strided(transient, rows, (int)B, (int)T, (int)(S * L), nv, 0, st);
  if (rc) return rc;
  const int64_t n_head = std::max<int64_t>(S * L, S + L);
  hipLaunchKernelGGL(velten_ex_head_kernel, dim3((unsigned)((n_head + 255) / 256), (unsigned)B),
                     dim3(256), 0, st, scan_points, laser_points, scan_origin, laser_origin, g,
                     (int)S, (int)L, (int)So, (int)Lo, head, rows);
  rc = check_launch("velten_ex_head_kernel");
  if (rc) return rc;
  return velten_ex(head, rows, volume, g, S, L, st);
}

namespace totri_hip {
namespace {

// Arellano plan: chunks of the positive-bin list per column tile, enough
// waves to fill the device, partial volumes capped at 1 GiB.  Workspace:
// transposed transient | compaction | partial volumes (when chunks > 1).
struct ArellanoPlan {
  int chunks;
  size_t tr_bytes;
  CompactLayout cl;
  size_t part_off, ws;
};

ArellanoPlan plan_arellano(int64_t B, int64_t T, int64_t S, int64_t L, int64_t D, int64_t H,
                           int64_t W) {
  ArellanoPlan p;
  const int64_t n = T * S * L;
  const int64_t V = D * H * W;
  const int64_t tiles = ((H * W + 63) / 64) * (B > 0 ? B : 1);
  const int64_t target = 8 * (int64_t)device_cu_count();
  int64_t C = tiles > 0 ? (target + tiles - 1) / tiles : 1;
  if (C > 64) C = 64;
  const int64_t cap = (int64_t)1 << 28;  // floats of partial volumes
  if (B * V > 0 && C * B * V > cap) C = cap / (B * V);
  if (C < 1) C = 1;
  p.chunks = (int)C;
  p.tr_bytes = align256((size_t)B * n * sizeof(float));
  p.cl = compact_layout(B, n, p.tr_bytes);
  p.part_off = p.cl.end;
  p.ws = p.part_off + (C > 1 ? align256((size_t)C * B * V * sizeof(float)) : 0);
  return p;
}

}  // namespace
}  // namespace totri_hip

extern "C" size_t totri_backprojection_exhaustive_arellano_workspace(
    int64_t B, int64_t T, int64_t S, int64_t L, int64_t D, int64_t H, int64_t W) {
  if (B <= 0 || T <= 0 || S <= 0 || L <= 0 || D <= 0 || H <= 0 || W <= 0) return 0;
  return plan_arellano(B, T, S, L, D, H, W).ws;
}

extern "C" int totri_backprojection_exhaustive_arellano_forward(
    const float* transient, int64_t B, int64_t T, int64_t S, int64_t L,
    const float* scan_points, const float* laser_points, const float* scan_origin,
    int64_t So, const float* laser_origin, int64_t Lo, float* volume, int64_t D, int64_t H,
    int64_t W, const float volume_start[3], const float volume_end[3], float bin_width,
    float bin_offset, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_dims({B, T, S, L, So, Lo, D, H, W}, B * T * S * L, B * D * H * W);
  if (rc) return rc;
  TOTRI_CHECK_ARG(So == 0 || So == S, "scan_origin must have 0 or S points");
  TOTRI_CHECK_ARG(Lo == 0 || Lo == L, "laser_origin must have 0 or L points");
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  hipStream_t st = (hipStream_t)stream;
  const size_t ncol = (size_t)H * W;
  const size_t nv = (size_t)B * D * ncol;
  if (nv == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume != nullptr, "null volume");
  if (T == 0 || S == 0 || L == 0) {
    // nothing to backproject: the written volume is zero
    hipLaunchKernelGGL(zero_kernel, dim3(grid1d(nv)), dim3(256), 0, st, volume, nv);
    return check_launch("zero_kernel");
  }
  TOTRI_CHECK_ARG(transient && scan_points && laser_points, "null input");
  TOTRI_CHECK_ARG((So == 0 || scan_origin) && (Lo == 0 || laser_origin), "null origin");
  const ArellanoPlan p = plan_arellano(B, T, S, L, D, H, W);
  if (workspace_bytes < p.ws)
    return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", p.ws,
                workspace_bytes);
  TOTRI_CHECK_ARG(workspace != nullptr, "null workspace");
  const BoxGeom g = box_geom(B, D, H, W, T, volume_start, volume_end, bin_width, bin_offset);
  float* trT = (float*)workspace;
  rc = launch_transpose(transient, trT, (int)B, (int)T, (int)(S * L), st);
  if (rc) return rc;
  rc = launch_compact(trT, (int)B, (int)(T * S * L), p.cl, workspace, Positive(), st);
  if (rc) return rc;
  const int* totals = (const int*)((char*)workspace + p.cl.totals_off);
  const int* list = (const int*)((char*)workspace + p.cl.list_off);
  float* dst = p.chunks > 1 ? (float*)((char*)workspace + p.part_off) : volume;
  const dim3 grid((unsigned)((ncol + 63) / 64), (unsigned)p.chunks, (unsigned)B);
  if (D <= 256) {
    hipLaunchKernelGGL(arellano_kernel<true>, grid, dim3(64), (size_t)D * 64 * sizeof(float),
                       st, trT, list, totals, scan_points, laser_points, scan_origin,
                       laser_origin, dst, g, (int)S, (int)L, (int)So, (int)Lo, p.chunks);
  } else {
    hipLaunchKernelGGL(arellano_kernel<false>, grid, dim3(64), 0, st, trT, list, totals,
                       scan_points, laser_points, scan_origin, laser_origin, dst, g, (int)S,
                       (int)L, (int)So, (int)Lo, p.chunks);
  }
  rc = check_launch("arellano_kernel");
  if (rc || p.chunks == 1) return rc;
  hipLaunchKernelGGL(sum_parts_kernel, dim3(grid1d(nv)), dim3(256), 0, st, dst, p.chunks, nv,
                     volume);
  return check_launch("sum_parts_kernel");
}
