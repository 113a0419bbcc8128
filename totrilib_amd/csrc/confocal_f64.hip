// Double-precision forms of the confocal render (R1), its adjoint (A1, exact
// transpose and the reference's window form) and the confocal Velten
// backprojection (A2), for float64 tensors: the reference dispatches these
// kernels on float and double (AT_DISPATCH_FLOATING_TYPES,
// src/render/volume_cuda.cu:85,175, src/reconstruct/backprojection_cuda.cu:215).
//
// With scalar_t = double the reference keeps some float steps, restated here:
//   - geometry arguments are float; the bin radius t * w + off is a float
//     expression, widened (volume_cuda.cu:23,137);
//   - floorf(z_hat) and ceilf(tf) narrow their double argument to float
//     (:48,:132-134,:146);
//   - A2 converts the points to float3 and measures float distances; the bin
//     arithmetic and the sum are double (backprojection_cuda.cu:167-190).
// pow(x, 2) and pow(x, 4) are written as products.
//
// Each output's sum is the reference's sequence of double operations (columns,
// scan points and bins in order); FP64 is the accuracy form, the FP32 kernels
// are the fast path.
#include <math.h>

#include "common.h"

namespace totri_hip {
namespace {

__device__ __forceinline__ double cell_centre_d(int i, float o, float sz, int n) {
  double a = ((double)i + 0.5) * (double)sz;  // volume_cuda.cu:35
  a = a / (double)n;
  return (double)o + a;
}

// Correctly rounded square root without the library form's scaling and special
// values: one Newton step on the hardware's reciprocal root, then two residual
// steps, of which the last decides the rounding (Markstein).  For positive x in
// [2^-500, 2^500], which every active sample's d2 is: its terms are a square
// of a float radius and a difference from it, so a positive one is at least
// 2^-460 and at most 2^256.  Other x give NaN.
__device__ __forceinline__ double sqrt_mid_f64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}

// x is positive and finite.
__device__ __forceinline__ bool positive_f64(double x) {
  return __builtin_amdgcn_class(x, 0x180);
}

struct SampleD {
  bool active;
  int zi;
  double alpha, f2;
};

// One R1 sample (volume_cuda.cu:40-58 with scalar_t = double).
__device__ __forceinline__ SampleD sample_d(double tc, double wx, double wy, double wz,
                                            double x, double y, double o, double s, int Z) {
  SampleD r;
  r.active = false;
  r.zi = 0;
  r.alpha = 0.0;
  r.f2 = 0.0;
  const double t2 = tc * tc;
  const double dx = wx - x, dy = wy - y;
  double d2 = t2 - dx * dx;
  d2 = d2 - dy * dy;
  if (!(d2 > 0.0)) return r;
  const double depth = sqrt(d2);
  const double z = wz + depth;
  double zh = (z - o) * s;
  zh = zh - 0.5;
  const int zi = (int)floorf((float)zh);  // floorf narrows to float
  if (!(zi >= 0 && zi + 1 < Z)) return r;
  r.active = true;
  r.zi = zi;
  r.alpha = zh - (double)zi;
  const double q = -depth / t2;
  const double q2 = q * q;
  r.f2 = q2 * q2;
  return r;
}

struct GeomD {
  int X, Y, Z, N, T;
  float ox, oy, oz, sx, sy, sz, w, off;
};

// R1: one thread per (scan point, bin); columns in order (volume_cuda.cu:33-63).
// The form for transients of few bins: r1_tiles_f64_kernel takes the others.
__global__ __launch_bounds__(256) void r1_f64_kernel(const double* __restrict__ vol,
                                                     const double* __restrict__ mp,
                                                     double* __restrict__ tr, GeomD g) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)g.N * g.T) return;
  const int i = (int)(e / g.T), ti = (int)(e - (long long)i * g.T);
  const double wx = mp[i], wy = mp[g.N + i], wz = mp[2 * g.N + i];
  const double o = (double)g.oz;
  const double s = (double)g.Z / (double)g.sz;
  const double tc = (double)bin_distance(ti, g.w, g.off);
  double value = 0.0;
  for (int xi = 0; xi < g.X; ++xi) {
    const double x = cell_centre_d(xi, g.ox, g.sx, g.X);
    for (int yi = 0; yi < g.Y; ++yi) {
      const double y = cell_centre_d(yi, g.oy, g.sy, g.Y);
      const SampleD sm = sample_d(tc, wx, wy, wz, x, y, o, s, g.Z);
      if (!sm.active) continue;
      const double* col = vol + ((size_t)xi * g.Y + yi) * g.Z;
      const double f1 = (1.0 - sm.alpha) * col[sm.zi] + sm.alpha * col[sm.zi + 1];
      value = value + f1 * sm.f2;
    }
  }
  tr[e] = value;
}

// The same sums, 64 bins of one scan point to a workgroup: three producer waves
// take eight columns each, leave the samples' terms in LDS, and a fourth wave,
// a lane per bin, adds the previous round's in column order (a lane that walks
// its own columns waits for every sample's chain: 32^3 voxels, 256 points, 256
// bins are one wave per SIMD).  An inactive sample's term is +0, which leaves
// a sum that began at +0 unchanged.  Where bins and rows rise together (w > 0,
// off >= 0, size_z > 0) the rows of a column's first and last bin tell whether
// any bin between is active; columns with none leave zeros.  The bin's square
// is the lane's own, so depth / t2 is a division by a constant (see DivConst).
// Bound by the double-precision issue rate of the square roots and quotients.
// 32^3 voxels, 256 points, 256 bins: 287 -> 105 us (four waves, so that
// a workgroup loads the SIMDs evenly; with five, 178).
constexpr int kProdR1F64 = 3, kColsR1F64 = 8;
// Of fewer bins a tile has too many idle lanes: 32^2 x 16 voxels take 420 us
// with 4,096 points of 8 bins (r1_f64_kernel: 276), and with 16 bins the gain
// (275 -> 128 us, 1,024 points) is gone once r1_f64_kernel fills the chip.
constexpr int kMinBinsF64 = 32;

__global__ __launch_bounds__(64 * (kProdR1F64 + 1)) void r1_tiles_f64_kernel(
    const double* __restrict__ vol, const double* __restrict__ mp, double* __restrict__ tr,
    GeomD g, int n_tiles, int rising) {
  constexpr int P = kProdR1F64, U = kColsR1F64, H = 4;
  __shared__ double terms[2][P][U][64];
  __shared__ double2 lateral[P][64];  // squared x and y offsets of a wave's next columns
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double o = (double)g.oz;
  const double s = (double)g.Z / (double)g.sz;
  const int n_cols = g.X * g.Y;
  const int rounds = (n_cols + P * U - 1) / (P * U);
  const long long n_blocks = (long long)g.N * n_tiles;
  for (long long blk = blockIdx.x; blk < n_blocks; blk += gridDim.x) {
    // Neighbouring workgroups (on different XCDs) take the same bins: the near
    // bins are active in fewer columns.
    const int i = (int)(blk % g.N);
    const int tile = (int)(blk / g.N) * 64;
    const double wx = mp[i], wy = mp[g.N + i], wz = mp[2 * g.N + i];
    const int ti = min(tile + lane, g.T - 1);
    auto bin_square = [&](int t) {
      const double tc = (double)bin_distance(t, g.w, g.off);
      return tc * tc;
    };
    auto row_of = [&](double d2, double* depth, double* zh) {
      *depth = sqrt_mid_f64(d2);
      const double z = wz + *depth;
      *zh = (z - o) * s;
      *zh = *zh - 0.5;
      return (int)floorf((float)*zh);  // floorf narrows to float
    };
    const double t2 = bin_square(ti);
    const double t2a = bin_square(tile), t2b = bin_square(min(tile + 63, g.T - 1));
    const double hi = 1.0 / t2;
    const double lo = __builtin_fma(-hi, t2, 1.0) * hi;
    double value = 0.0;
    unsigned long long some = 0;  // bit: lateral[wave][bit]'s column has an active bin
    for (int r = 0; r <= rounds; ++r) {
      if (wave < P && r < rounds) {
        if (r % 8 == 0) {
          const int c = (r + (lane >> 3)) * (P * U) + wave * U + (lane & 7);
          const int cc = min(c, n_cols - 1);
          const int xi = cc / g.Y, yi = cc - xi * g.Y;
          const double dx = wx - cell_centre_d(xi, g.ox, g.sx, g.X);
          const double dy = wy - cell_centre_d(yi, g.oy, g.sy, g.Y);
          const double dx2 = dx * dx, dy2 = dy * dy;
          lateral[wave][lane] = make_double2(dx2, dy2);
          bool a = c < n_cols && g.Z > 1;
          if (rising) {
            double d2a = t2a - dx2, d2b = t2b - dx2, depth, zh;
            d2a = d2a - dy2;
            d2b = d2b - dy2;
            const bool past = positive_f64(d2a) && row_of(d2a, &depth, &zh) >= g.Z - 1;
            const bool before = !(d2b > 0.0) ||
                                (positive_f64(d2b) && row_of(d2b, &depth, &zh) < 0);
            a = a && !past && !before;
          }
          some = __ballot(a);
        }
        const int k = (r & 7) * U;
        const int c0 = r * (P * U) + wave * U;
#pragma unroll
        for (int h = 0; h < U; h += H) {
          double(*out)[64] = &terms[r & 1][wave][h];
          if (((some >> (k + h)) & ((1u << H) - 1u)) == 0) {
#pragma unroll
            for (int u = 0; u < H; ++u) out[u][lane] = 0.0;
            continue;
          }
          double depth[H], alpha[H], v0[H], v1[H];
          bool act[H];
#pragma unroll
          for (int u = 0; u < H; ++u) {
            const double2 l = lateral[wave][k + h + u];
            double d2 = t2 - l.x;
            d2 = d2 - l.y;
            double zh;
            const int zu = row_of(d2, &depth[u], &zh);
            // no short circuits: a branch per sample would serialise the chains
            act[u] = positive_f64(d2) & (zu >= 0) & (zu < g.Z - 1) & (c0 + h + u < n_cols);
            const unsigned zi = act[u] ? zu : 0;
            alpha[u] = zh - (double)zu;
            const double* p = vol + (size_t)min(c0 + h + u, n_cols - 1) * g.Z;
            v0[u] = p[zi];
            v1[u] = p[zi + 1];
          }
#pragma unroll
          for (int u = 0; u < H; ++u) {
            double q = __builtin_fma(depth[u], hi, depth[u] * lo);
            q = __builtin_fma(__builtin_fma(-q, t2, depth[u]), hi, q);
            q = q * q;
            const double f2 = q * q;
            const double f1 = (1.0 - alpha[u]) * v0[u] + alpha[u] * v1[u];
            out[u][lane] = act[u] ? f1 * f2 : 0.0;
          }
        }
      } else if (wave == P && r > 0) {
#pragma unroll
        for (int p = 0; p < P; ++p)
#pragma unroll
          for (int u = 0; u < U; ++u) value = value + terms[(r - 1) & 1][p][u][lane];
      }
      __syncthreads();
    }
    if (wave == P && tile + lane < g.T) tr[(size_t)i * g.T + tile + lane] = value;
  }
}

// A1 as the exact transpose of r1_f64_kernel: one thread per voxel; over scan
// points and bins in order, a sample flooring to z adds (1 - alpha) f2 G and
// one flooring to z - 1 adds alpha f2 G.  The general form: a1_rows_f64_kernel
// takes the calls with w > 0, off >= 0 and size_z > 0.
__global__ __launch_bounds__(256) void a1_f64_kernel(double* __restrict__ vol,
                                                     const double* __restrict__ mp,
                                                     const double* __restrict__ G, GeomD g) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)g.X * g.Y * g.Z) return;
  const int z = (int)(e % g.Z);
  const int col = (int)(e / g.Z);
  const int xi = col / g.Y, yi = col - (col / g.Y) * g.Y;
  const double x = cell_centre_d(xi, g.ox, g.sx, g.X);
  const double y = cell_centre_d(yi, g.oy, g.sy, g.Y);
  const double o = (double)g.oz;
  const double s = (double)g.Z / (double)g.sz;
  const bool windowed = g.w > 0.f && g.off >= 0.f && g.sz > 0.f;
  double value = 0.0;
  for (int i = 0; i < g.N; ++i) {
    const double wx = mp[i], wy = mp[g.N + i], wz = mp[2 * g.N + i];
    int t0 = 0, t1 = g.T - 1;
    if (windowed) {
      const double dx = wx - x, dy = wy - y;
      const double rho2 = dx * dx + dy * dy;
      const double dlo = fmax(((double)z - 3.0 + 0.5) / s + o - wz, 0.0);
      const double dhi = ((double)z + 3.0 + 0.5) / s + o - wz;
      if (!(dhi > 0.0)) continue;
      const double rlo = sqrt(rho2 + dlo * dlo) * (1.0 - 1e-6);
      const double rhi = sqrt(rho2 + dhi * dhi) * (1.0 + 1e-6);
      const double ta = floor((rlo - (double)g.off) / (double)g.w) - 2.0;
      const double tb = ceil((rhi - (double)g.off) / (double)g.w) + 2.0;
      t0 = ta < 0.0 ? 0 : (ta > (double)g.T ? g.T : (int)ta);
      t1 = tb > (double)(g.T - 1) ? g.T - 1 : (tb < -1.0 ? -1 : (int)tb);
    }
    const double* gi = G + (size_t)i * g.T;
    for (int ti = t0; ti <= t1; ++ti) {
      const double tc = (double)bin_distance(ti, g.w, g.off);
      const SampleD sm = sample_d(tc, wx, wy, wz, x, y, o, s, g.Z);
      if (!sm.active) continue;
      if (sm.zi == z) {
        value += (1.0 - sm.alpha) * (sm.f2 * gi[ti]);
      } else if (sm.zi + 1 == z) {
        value += sm.alpha * (sm.f2 * gi[ti]);
      }
    }
  }
  vol[e] = value;
}

// The same sums where bins and rows rise together (w > 0, off >= 0, size_z >
// 0).  A voxel's samples are then the bins of two neighbouring rows, so a
// workgroup takes one column's tile of 64 voxels and computes each sample of
// it once (a1_f64_kernel computes a sample for about seven voxels): three
// producer waves take three units -- a unit is a scan point and up to kBinsF64
// of its bins -- and leave in LDS each sample's two contributions and the bin
// at which each row starts; the fourth wave, a lane per voxel, adds the
// previous round's contributions in scan point and bin order.  Inactive
// samples hold +0, which leaves a sum that began at +0 unchanged.  Bound by
// the double-precision issue rate of the samples' square root and division.
// 32^3 voxels, 256 points, 256 bins: 1575 -> 197 us (with four
// producers, five waves: 277).
constexpr int kBinsF64 = 256, kProdF64 = 3, kTileF64 = 64;
// Of fewer rows a tile has too few voxels for a unit's samples: 256 x 256
// columns, 64 points, 128 bins take 2.42 ms with 8 rows (a1_f64_kernel: 3.09)
// and 3.59 ms with 4 (2.69).
constexpr int kMinRowsF64 = 8;
// Of few samples a workgroup's rounds cost more than they share (us a call with
// a1_f64_kernel and with tiles, 64 x 64 x 16 voxels: 4 points of 48 bins 23, 26, of
// 256 bins 44, 31; 100 x 100 x 8: 16 points of 32 bins 76, 84, of 48 bins 93, 83); in
// tiles of few rows a unit of few bins leaves lanes idle (64 points of 16 bins 199,
// 237, of 31 bins 265, 237).
constexpr int kMinSamplesF64 = 640, kShortTileF64 = 16, kMinBinsShortF64 = 24;
struct UnitF64 {
  double2 c[kBinsF64];        // alpha f2 G (row zi + 1), (1 - alpha) f2 G (row zi)
  double2 zero;               // c[kBinsF64].x = +0
  int start[kTileF64 + 2];    // first bin of the unit at or past row z0 - 1 + i
};

// The value lane `l` (uniform) holds.
__device__ __forceinline__ double lane_f64(double v, int l) {
  const unsigned long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, l);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), l);
  return __longlong_as_double(((unsigned long long)hi << 32) | lo);
}

__global__ __launch_bounds__(64 * (kProdF64 + 1)) void a1_rows_f64_kernel(
    double* __restrict__ vol, const double* __restrict__ mp, const double* __restrict__ G,
    GeomD g, int n_tiles, int chunks) {
  __shared__ UnitF64 buf[2][kProdF64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = blockIdx.x / n_tiles;
  const int z0 = (blockIdx.x - col * n_tiles) * kTileF64;
  const int xi = col / g.Y, yi = col - (col / g.Y) * g.Y;
  const double x = cell_centre_d(xi, g.ox, g.sx, g.X);
  const double y = cell_centre_d(yi, g.oy, g.sy, g.Y);
  const double o = (double)g.oz;
  const double s = (double)g.Z / (double)g.sz;
  const int z_last = min(z0 + kTileF64, g.Z) - 1;
  const unsigned units = (unsigned)g.N * (unsigned)chunks;  // < 2^32: N T < 2^31
  const unsigned rounds = units / kProdF64 + (units % kProdF64 != 0);
  if (threadIdx.x < 2 * kProdF64)
    buf[threadIdx.x / kProdF64][threadIdx.x % kProdF64].zero = make_double2(0.0, 0.0);
  __syncthreads();
  double value = 0.0;
  // Producers: lane r % 64 holds its wave's unit of round r: squared lateral
  // offsets, the wall's z, the scan point and the bins [first, last].
  double dx2l = 0.0, dy2l = 0.0, wzl = 0.0;
  int il = 0, t0l = 0, t1l = -1;
  for (unsigned r = 0; r <= rounds; ++r) {
    if (wave < kProdF64) {
      if ((r & 63u) == 0) {
        const unsigned u = min((r + lane) * kProdF64 + wave, units - 1u);
        il = (int)(u / (unsigned)chunks);
        if (r < rounds) {
          const double wx = mp[il], wy = mp[g.N + il];
          wzl = mp[2 * g.N + il];
          const double dx = wx - x, dy = wy - y;
          dx2l = dx * dx;
          dy2l = dy * dy;
          // The tile's bins: rows max(z0 - 1, 0) .. min(z_last, Z - 2), a
          // quarter row wider (2^20 rows round to 1/16 when narrowed).
          t0l = 0;
          t1l = -1;
          const double row_lo = (double)max(z0 - 1, 0), row_hi = (double)min(z_last + 1, g.Z - 1);
          const double dlo = fmax((row_lo + 0.25) / s + o - wzl, 0.0);
          const double dhi = (row_hi + 0.75) / s + o - wzl;
          if (dhi > 0.0) {
            const double rho2 = dx2l + dy2l;
            const double rlo = sqrt(rho2 + dlo * dlo) * (1.0 - 1e-6);
            const double rhi = sqrt(rho2 + dhi * dhi) * (1.0 + 1e-6);
            const double ta = floor((rlo - (double)g.off) / (double)g.w) - 2.0;
            const double tb = ceil((rhi - (double)g.off) / (double)g.w) + 2.0;
            t0l = ta < 0.0 ? 0 : (ta > (double)g.T ? g.T : (int)ta);
            t1l = tb > (double)(g.T - 1) ? g.T - 1 : (tb < -1.0 ? -1 : (int)tb);
          }
          t0l += (int)(u - (unsigned)il * (unsigned)chunks) * kBinsF64;
        }
      }
      const int rl = (int)(r & 63u);
      if (r * kProdF64 + wave < units) {
        UnitF64& b = buf[r & 1][wave];
        const double dx2 = lane_f64(dx2l, rl), dy2 = lane_f64(dy2l, rl);
        const double wz = lane_f64(wzl, rl);
        const int t0 = __builtin_amdgcn_readlane(t0l, rl);
        const int t1 = __builtin_amdgcn_readlane(t1l, rl);
        const double* gi = G + (size_t)__builtin_amdgcn_readlane(il, rl) * g.T;
        const int cnt = min(t1 + 1 - t0, kBinsF64);
        if (cnt <= 0) {
          for (int k = lane; k < kTileF64 + 2; k += 64) b.start[k] = 0;
        } else {
          int prev = 0;  // row of the bin before this lane's
          for (int j = 0; j < cnt; j += 64) {
            const int k = j + lane;
            const int t = min(t0 + k, t1);
            const double gt = gi[t];
            const double tc = (double)bin_distance(t, g.w, g.off);
            const double t2 = tc * tc;
            double d2 = t2 - dx2;
            d2 = d2 - dy2;
            const double depth = sqrt_mid_f64(d2);
            const double z = wz + depth;
            double zh = (z - o) * s;
            zh = zh - 0.5;
            const int zi = (int)floorf((float)zh);  // floorf narrows to float
            const bool below = !positive_f64(d2) | (zi < 0);
            const bool act = !below & (zi < g.Z - 1);
            const double alpha = zh - (double)zi;
            const double q = -depth / t2;
            const double q2 = q * q;
            const double fg = (q2 * q2) * gt;
            b.c[k] = make_double2(act ? alpha * fg : 0.0, act ? (1.0 - alpha) * fg : 0.0);
            const int row = below ? -1 : min(max(min(zi, g.Z) - (z0 - 1), -1), kTileF64 + 1);
            if (j == 0) {
              prev = __builtin_amdgcn_readfirstlane(row);
              for (int m = lane; m < kTileF64 + 2; m += 64) b.start[m] = m <= prev ? 0 : cnt;
            }
            const int up = __shfl_up(row, 1);
            const int before = lane == 0 ? prev : up;
            if (k < cnt)
              for (int m = before + 1; m <= row; ++m) b.start[m] = k;
            prev = __builtin_amdgcn_readlane(row, 63);
          }
        }
      }
    } else if (r > 0) {
      const unsigned u0 = (r - 1) * kProdF64;
      const int nu = (int)min(units - u0, (unsigned)kProdF64);
      for (int p = 0; p < nu; ++p) {
        const UnitF64& b = buf[(r - 1) & 1][p];
        const double* c = (const double*)b.c;
        // bins [ka, kb) are on row z - 1, [kb, kc) on row z: in halves of c
        const int ka = 2 * b.start[lane], kb = 2 * b.start[lane + 1], kc = 2 * b.start[lane + 2];
        for (int k = ka; __ballot(k < kc) != 0; k += 8) {
          double v[4];
#pragma unroll
          for (int m = 0; m < 4; ++m) {
            const int e = k + 2 * m + (k + 2 * m >= kb ? 1 : 0);
            v[m] = c[k + 2 * m < kc ? e : 2 * kBinsF64];
          }
#pragma unroll
          for (int m = 0; m < 4; ++m) value += v[m];
        }
      }
    }
    __syncthreads();
  }
  if (wave == kProdF64 && z0 + lane < g.Z) vol[(size_t)col * g.Z + z0 + lane] = value;
}

// The reference's window-form A1 in double (volume_cuda.cu:95-160): one
// thread per voxel, scan points and window bins in order.
__global__ __launch_bounds__(256) void a1_window_f64_kernel(double* __restrict__ vol,
                                                            const double* __restrict__ mp,
                                                            const double* __restrict__ G,
                                                            GeomD g) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (long long)g.X * g.Y * g.Z) return;
  const int zi = (int)(e % g.Z);
  const int col = (int)(e / g.Z);
  const int xi = col / g.Y, yi = col - (col / g.Y) * g.Y;
  const double x = cell_centre_d(xi, g.ox, g.sx, g.X);  // :107-109
  const double y = cell_centre_d(yi, g.oy, g.sy, g.Y);
  const double z = cell_centre_d(zi, g.oz, g.sz, g.Z);
  const double o = (double)g.oz;
  const double s = (double)g.Z / (double)g.sz;          // :112
  const double dz = (double)g.sz / (double)g.Z;         // :114
  double value = 0.0;
  for (int i = 0; i < g.N; ++i) {
    const double wx = mp[i], wy = mp[g.N + i], wz = mp[2 * g.N + i];
    const double zz = zi > 0 ? dz : 0.0;                // :123
    const double ax = x - wx, ay = y - wy;
    const double dps = ax * ax + ay * ay;               // :124
    const double a = (z - zz) - wz, b = z - wz, c = (z + dz) - wz;
    const double ds = sqrt(dps + a * a);                // :125-127
    const double dm = sqrt(dps + b * b);
    const double de = sqrt(dps + c * c);
    int ts = (int)ceilf((float)((ds - (double)g.off) / (double)g.w));  // :129-134
    int tm = (int)ceilf((float)((dm - (double)g.off) / (double)g.w));
    int te = (int)ceilf((float)((de - (double)g.off) / (double)g.w));
    ts = min(max(ts, 0), g.T);
    tm = min(max(tm, 0), g.T);
    te = min(max(te, 0), g.T);
    const double* gi = G + (size_t)i * g.T;
    for (int ti = ts; ti < te; ++ti) {                  // :135-156
      const double tc = (double)bin_distance(ti, g.w, g.off);
      const double t2 = tc * tc;
      const double d2 = t2 - dps;
      if (!(d2 > 0.0)) continue;
      const double depth = sqrt(d2);
      const double zc = wz + depth;
      double zh = (zc - o) * s;
      zh = zh - 0.5;
      const int zf = (int)floorf((float)zh);
      const double alpha = zh - (double)zf;
      const double df1 = ti >= tm ? 1.0 - alpha : alpha;
      const double q = -depth / t2;
      const double q2 = q * q;
      const double f2 = q2 * q2;
      value = value + (df1 * f2) * gi[ti];
    }
  }
  vol[e] = value;
}

// A2 in double (backprojection_cuda.cu:152-194): one thread per voxel of
// [B][D][H][W]; float points and distances, double bin arithmetic and sum.
__global__ __launch_bounds__(256) void velten_f64_kernel(
    const double* __restrict__ tr, const double* __restrict__ scan,
    const double* __restrict__ orig, double* __restrict__ vol, int B, int T, int S, int So,
    int D, int H, int W, float sx, float sy, float sz, float ex, float ey, float ez, float w,
    float off) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long nv = (long long)D * H * W;
  if (e >= (long long)B * nv) return;
  const int b = (int)(e / nv);
  const int v = (int)(e - (long long)b * nv);
  const int x = v % W, y = (v / W) % H, z = v / (W * H);
  const float qx = inclusive_coord(x, W, sx, ex);
  const float qy = inclusive_coord(y, H, sy, ey);
  const float qz = inclusive_coord(z, D, sz, ez);
  const double* sb = scan + (size_t)b * S * 3;
  const double* ob = orig + (size_t)b * So * 3;
  const double* tb = tr + (size_t)b * T * S;
  double value = 0.0;
  for (int s = 0; s < S; ++s) {
    const float px = (float)sb[3 * s], py = (float)sb[3 * s + 1], pz = (float)sb[3 * s + 2];
    const double dsv = (double)dist3(px, py, pz, qx, qy, qz);                 // :177
    const double dso = So > 0 ? (double)dist3(px, py, pz, (float)ob[3 * s],
                                              (float)ob[3 * s + 1], (float)ob[3 * s + 2])
                              : 0.0;                                          // :178-183
    const double dist = 2.0 * dso + 2.0 * dsv;                               // :185
    const double tf = (dist - (double)off) / (double)w + 0.5;
    const int ti = (int)floorf((float)tf);                                   // :187
    if (ti >= 0 && ti < T) value += tb[(size_t)ti * S + s];                  // :188-190
  }
  vol[e] = value;                                                            // :192
}

unsigned blocks_for(long long n) { return (unsigned)((n + 255) / 256); }

int check_conf_f64(int64_t X, int64_t Y, int64_t Z, int64_t N, int64_t T, const float* o,
                   const float* sz) {
  TOTRI_CHECK_ARG(X >= 0 && Y >= 0 && Z >= 0 && N >= 0 && T >= 0, "negative dimension");
  TOTRI_CHECK_ARG(X < (1ll << 31) && Y < (1ll << 31) && Z < (1ll << 31) && N < (1ll << 31) &&
                      T < (1ll << 31),
                  "dimension exceeds 32-bit indexing");
  TOTRI_CHECK_ARG(X * Y * Z < (1ll << 31) && N * T < (1ll << 31),
                  "tensor has more than 2^31 elements");
  TOTRI_CHECK_ARG(o != nullptr && sz != nullptr, "null geometry");
  return TOTRI_OK;
}

GeomD geom_d(int64_t X, int64_t Y, int64_t Z, int64_t N, int64_t T, const float* o,
             const float* sz, float w, float off) {
  GeomD g;
  g.X = (int)X;
  g.Y = (int)Y;
  g.Z = (int)Z;
  g.N = (int)N;
  g.T = (int)T;
  g.ox = o[0];
  g.oy = o[1];
  g.oz = o[2];
  g.sx = sz[0];
  g.sy = sz[1];
  g.sz = sz[2];
  g.w = w;
  g.off = off;
  return g;
}

// Units per scan point that cover every tile's bins: a tile's radii span at
// most its depth (64 voxels and 3 on either side), and the window's margins
// are relative to radii that a bin can have.
int unit_chunks_f64(const GeomD& g) {
  const double far = (double)g.T * g.w + g.off;
  const double depth = ((double)(g.Z < kTileF64 ? g.Z : kTileF64) + 6.0) * g.sz / g.Z;
  const double span = depth * (1.0 + 1e-6) + 3e-6 * far +
                      1e-11 * (far + fabs((double)g.oz) + (double)g.sz);
  const double bins = fmin(span / g.w + 10.0, (double)g.T);
  return (int)((bins + kBinsF64 - 1.0) / kBinsF64);
}

}  // namespace
}  // namespace totri_hip

using namespace totri_hip;

extern "C" int totri_volume_confocal_forward_f64(
    const double* volume, int64_t X, int64_t Y, int64_t Z, const double* measurement_points,
    int64_t N, double* transient, int64_t T, const float volume_origin[3],
    const float volume_size[3], float bin_width, float bin_offset, void* stream) {
  int rc = check_conf_f64(X, Y, Z, N, T, volume_origin, volume_size);
  if (rc) return rc;
  if (N * T == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(transient && measurement_points && (X * Y * Z == 0 || volume),
                  "null pointer");
  const GeomD g = geom_d(X, Y, Z, N, T, volume_origin, volume_size, bin_width, bin_offset);
  if (T >= kMinBinsF64) {
    const long long n_tiles = (T + 63) / 64;
    const long long blocks = N * n_tiles;
    const int rising = bin_width > 0.f && bin_offset >= 0.f && volume_size[2] > 0.f;
    hipLaunchKernelGGL(r1_tiles_f64_kernel, dim3((unsigned)(blocks < (1 << 22) ? blocks : 1 << 22)),
                       dim3(64 * (kProdR1F64 + 1)), 0, (hipStream_t)stream, volume,
                       measurement_points, transient, g, (int)n_tiles, rising);
    return check_launch("r1_tiles_f64_kernel");
  }
  hipLaunchKernelGGL(r1_f64_kernel, dim3(blocks_for(N * T)), dim3(256), 0,
                     (hipStream_t)stream, volume, measurement_points, transient, g);
  return check_launch("r1_f64_kernel");
}

extern "C" int totri_volume_confocal_grad_volume_f64(
    double* volume, int64_t X, int64_t Y, int64_t Z, const double* measurement_points,
    int64_t N, const double* transient, int64_t T, const float volume_origin[3],
    const float volume_size[3], float bin_width, float bin_offset, int window_form,
    void* stream) {
  int rc = check_conf_f64(X, Y, Z, N, T, volume_origin, volume_size);
  if (rc) return rc;
  const long long nv = X * Y * Z;
  if (nv == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume && (N * T == 0 || (measurement_points && transient)), "null pointer");
  const GeomD g = geom_d(X, Y, Z, N, T, volume_origin, volume_size, bin_width, bin_offset);
  if (window_form) {
    hipLaunchKernelGGL(a1_window_f64_kernel, dim3(blocks_for(nv)), dim3(256), 0,
                       (hipStream_t)stream, volume, measurement_points, transient, g);
    return check_launch("a1_window_f64_kernel");
  }
  const long long n_tiles = (Z + kTileF64 - 1) / kTileF64;
  const long long blocks = X * Y * n_tiles;
  if (bin_width > 0.f && bin_offset >= 0.f && volume_size[2] > 0.f && Z >= kMinRowsF64 &&
      N * T >= kMinSamplesF64 && (Z >= kShortTileF64 || T >= kMinBinsShortF64) &&
      Z <= (1 << 20) && blocks < (1ll << 23)) {
    hipLaunchKernelGGL(a1_rows_f64_kernel, dim3((unsigned)blocks), dim3(64 * (kProdF64 + 1)), 0,
                       (hipStream_t)stream, volume, measurement_points, transient, g,
                       (int)n_tiles, unit_chunks_f64(g));
    return check_launch("a1_rows_f64_kernel");
  }
  hipLaunchKernelGGL(a1_f64_kernel, dim3(blocks_for(nv)), dim3(256), 0, (hipStream_t)stream,
                     volume, measurement_points, transient, g);
  return check_launch("a1_f64_kernel");
}

extern "C" int totri_backprojection_confocal_velten_forward_f64(
    const double* transient, int64_t B, int64_t T, int64_t S, const double* scan_points,
    const double* scan_origin, int64_t So, double* volume, int64_t D, int64_t H, int64_t W,
    const float volume_start[3], const float volume_end[3], float bin_width, float bin_offset,
    void* stream) {
  for (int64_t d : {B, T, S, So, D, H, W})
    TOTRI_CHECK_ARG(d >= 0 && d < (1ll << 31), "dimension out of range");
  TOTRI_CHECK_ARG(B * T * S < (1ll << 31) && B * D * H * W < (1ll << 31),
                  "tensor has more than 2^31 elements");
  TOTRI_CHECK_ARG(So == 0 || So == S, "scan_origin must have 0 or S points");
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  const long long n = B * D * H * W;
  if (n == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume && (T * S == 0 || (transient && scan_points)), "null pointer");
  TOTRI_CHECK_ARG(So == 0 || scan_origin, "null scan_origin");
  hipLaunchKernelGGL(velten_f64_kernel, dim3(blocks_for(n)), dim3(256), 0, (hipStream_t)stream,
                     transient, scan_points, scan_origin, volume, (int)B, (int)T, (int)S,
                     (int)So, (int)D, (int)H, (int)W, volume_start[0], volume_start[1],
                     volume_start[2], volume_end[0], volume_end[1], volume_end[2], bin_width,
                     bin_offset);
  return check_launch("velten_f64_kernel");
}
