// Exhaustive (non-confocal) volume render R2 and its adjoint A5 for gfx950.
//
// Reference: src/render/volume_cuda.cu:297-466 (R2 kernel and the A5 launch,
// whose kernel body is empty), src/render/volume.cpp:83-111.
//
// R2 spreads each occupied voxel's occupancy over the bins of the path
// lengths |p_s - q| + |p_l - q| between its lower and upper z faces
// (volume_cuda.cu:330-375).  The reference scatters with global float
// atomics from one thread per (column, scan point, laser point).  Here one
// workgroup owns one (scan point, laser point) pair and its whole time
// histogram: every wave accumulates into a private copy of the histogram in
// LDS, the copies are summed and written once.  The histograms hold 64-bit
// fixed-point sums (integer LDS atomics, which run about three times as fast
// as float ones here): each weight is truncated to a multiple of 2^-e, with
// e chosen per batch so that no bin can overflow, and integer sums do not
// depend on the order of the atomics, so the result is the same on every
// run.  Occupied voxels come from a compacted list built in index order.
//
// A5 is written as R2's exact transpose with unit occupancy: one lane per
// voxel gathers, for every (scan, laser) pair, the weighted bins of the
// transposed upstream gradient staged in LDS.
//
// Decisions (bin span, clipping) follow the reference's FP32 formula with
// IEEE correctly rounded square roots and divisions.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "compact.h"
#include "stage.h"

namespace totri_hip {
namespace {

constexpr int kR2Waves = 4;
// Bins per R2 histogram tile: the waves' private 64-bit histograms fill 64
// KiB of LDS.  Longer transients take several tiles (grid z), each pass
// recomputing the voxel spans and keeping the bins of its tile.
constexpr int kR2Tile = 64 * 1024 / (kR2Waves * (int)sizeof(long long));

size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

struct ExGeom {
  int B, D, H, W, T;
  float sx, sy, sz, ex, ey, ez;
  float w, off;
};

// Voxel geometry (volume_cuda.cu:316-319,335-338): column centre (xf, yf)
// and the z of the voxel's lower and upper faces.
__device__ __forceinline__ void voxel_faces(const ExGeom& g, int xi, int yi, int zi,
                                            float* xf, float* yf, float* zf0, float* zf1) {
  float a = ((float)xi + 0.5f) / (float)g.W;
  *xf = g.sx + a * (g.ex - g.sx);
  a = ((float)yi + 0.5f) / (float)g.H;
  *yf = g.sy + a * (g.ey - g.sy);
  a = ((float)zi + 0.5f) / (float)g.D;
  const float zf = g.sz + a * (g.ez - g.sz);
  const float h = (0.5f / (float)g.D) * (g.ez - g.sz);
  *zf0 = zf - h;
  *zf1 = zf + h;
}

struct Span {
  int first, last;      // inclusive bin span; first > last when empty
  float wf, wm, wl;     // weights of the first, inner and last bins
};

// Bin span and weights of one voxel whose faces have path lengths d0 and d1
// (volume_cuda.cu:341-374).  With first == last the whole occupancy goes to
// that bin (wf = occ).
__device__ __forceinline__ Span span_of(const ExGeom& g, float occ, float d0, float d1) {
  Span r;
  if (d1 < d0) {
    const float t = d0;
    d0 = d1;
    d1 = t;
  }
  float bf0 = (d0 - g.off) / g.w;
  float bf1 = (d1 - g.off) / g.w;
  const float range = bf1 - bf0;
  int fb = (int)floorf(bf0), lb = (int)floorf(bf1);
  r.first = 1;
  r.last = 0;
  r.wf = r.wm = r.wl = 0.f;
  if (fb < 0) {
    if (lb < 0) return r;
    bf0 = 0.f;
    fb = 0;
  }
  if (lb >= g.T) {
    if (fb >= g.T) return r;
    bf1 = (float)(g.T - 1);
    lb = g.T - 1;
  }
  r.first = fb;
  r.last = lb;
  if (fb == lb) {
    r.wf = occ;
    return r;
  }
  const float frac = occ / range;
  r.wf = (1.f - (bf0 - (float)fb)) * frac;
  r.wm = frac;
  r.wl = (bf1 - (float)lb) * frac;
  return r;
}

// MID: every radicand lies in [2^-64, 2^64] (both points keep a distance
// from the box, sqrt_mid_range), so the short correctly rounded root serves.
template <bool MID>
__device__ __forceinline__ float ex_dist(float ax, float ay, float az, float bx, float by,
                                         float bz) {
  return MID ? sqrt_rn_mid(sqdist3(ax, ay, az, bx, by, bz)) : dist3(ax, ay, az, bx, by, bz);
}

template <bool MID>
__device__ __forceinline__ Span voxel_span(const ExGeom& g, float occ, float xf, float yf,
                                           float zf0, float zf1, float spx, float spy,
                                           float spz, float lpx, float lpy, float lpz) {
  const float d0 =
      ex_dist<MID>(spx, spy, spz, xf, yf, zf0) + ex_dist<MID>(lpx, lpy, lpz, xf, yf, zf0);
  const float d1 =
      ex_dist<MID>(spx, spy, spz, xf, yf, zf1) + ex_dist<MID>(lpx, lpy, lpz, xf, yf, zf1);
  return span_of(g, occ, d0, d1);
}
// Whether every squared distance from a point to the volume box lies in
// [2^-64, 2^64] (it is at least 2^-20 from the box and at most 2^30 from its
// far corner), so that the exhaustive kernels may take the short correctly
// rounded root for it.
__device__ __forceinline__ bool ex_point_mid(const ExGeom& g, float px, float py, float pz) {
  const float lo = box_sqdist(px, py, pz, g.sx, g.sy, g.sz, g.ex, g.ey, g.ez);
  float hi = 0.f;
  for (int c = 0; c < 8; ++c)
    hi = fmaxf(hi, sqdist3(px, py, pz, (c & 1) ? g.ex : g.sx, (c & 2) ? g.ey : g.sy,
                           (c & 4) ? g.ez : g.sz));
  return lo >= 0x1p-40f && hi <= 0x1p60f;  // false for NaN
}

// Headers {x, y, z, flag} of each batch's scan points, then laser points; and
// a zero per batch.
__global__ __launch_bounds__(256) void ex_point_head_kernel(const float* __restrict__ scan,
                                                            const float* __restrict__ laser,
                                                            int S, int L, ExGeom g,
                                                            float4* __restrict__ head,
                                                            int* __restrict__ zero) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int n = S + L;
  if (i < g.B) zero[i] = 0;
  if (i >= g.B * n) return;
  const int b = i / n, k = i - b * n;
  const int N = k < S ? S : L, at = k < S ? k : k - S;
  const float* p = (k < S ? scan : laser) + (size_t)b * 3 * N;
  const float x = p[at], y = p[N + at], z = p[2 * N + at];
  head[i] = make_float4(x, y, z, ex_point_mid(g, x, y, z) ? 1.f : 0.f);
}

// ---- R2 -------------------------------------------------------------------
// The occupied voxels' geometry in list order, computed once per call:
// geo[k] = {xf, yf, zf0, zf1} and occ[k] = the occupancy of list entry k;
// amax[b] collects the largest |occupancy| of batch b as float bits (zeroed
// before the launch; for non-negative floats the bit order is the value
// order, and NaN sorts above +inf).
__global__ __launch_bounds__(256) void r2_voxels_kernel(const float* __restrict__ vol,
                                                        const int* __restrict__ list,
                                                        const int* __restrict__ totals,
                                                        ExGeom g, float4* __restrict__ geo,
                                                        float* __restrict__ occ,
                                                        unsigned* __restrict__ amax) {
  const int b = blockIdx.y;
  const int nvox = g.D * g.H * g.W;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned bits = 0u;
  if (k < totals[b]) {
    const size_t bn = (size_t)b * nvox;
    const int v = list[bn + k];
    const int xi = v % g.W, yi = (v / g.W) % g.H, zi = v / (g.W * g.H);
    float xf, yf, zf0, zf1;
    voxel_faces(g, xi, yi, zi, &xf, &yf, &zf0, &zf1);
    geo[bn + k] = make_float4(xf, yf, zf0, zf1);
    const float o = vol[bn + v];
    occ[bn + k] = o;
    bits = __float_as_uint(fabsf(o));
  }
  // one atomic per wave
  for (int m = 32; m >= 1; m >>= 1) bits = max(bits, (unsigned)__shfl_xor((int)bits, m, 64));
  if ((threadIdx.x & 63) == 0 && bits) atomicMax(amax + b, bits);
}

__global__ void zero_u32_kernel(unsigned* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0u;
}

// trunc(x * 2^e) as an integer, for |x| * 2^e < 2^62: the float's mantissa
// shifted into place (zero for zeros and subnormals, which lie far below
// the resolution 2^-e, since the largest occupancy is normal on this path).
__device__ __forceinline__ long long r2_fixed(float x, int e) {
  const unsigned u = __float_as_uint(x);
  const int ex = (int)((u >> 23) & 255u);
  const unsigned long long m = (unsigned long long)((u & 0x7fffffu) | 0x800000u);
  const int sh = ex - 150 + e;  // x = m * 2^(ex - 150)
  unsigned long long q = sh >= 0 ? (m << min(sh, 63)) : (sh > -64 ? (m >> -sh) : 0ull);
  q = ex == 0 ? 0ull : q;
  return (u >> 31) ? -(long long)q : (long long)q;
}

// Fixed-point exponent of batch b: n occupied voxels of largest |occupancy|
// amax.  Every weight is at most |occupancy|, and a voxel adds to one bin at
// most once per pair, so a bin's sum stays below n * amax < 2^61 / 2^e.
__device__ __forceinline__ int r2_exponent(float amax, int n) {
  const int la = ilogbf(amax) + 1;    // amax < 2^la
  const int ln = 32 - __clz(n);       // n < 2^ln
  return 61 - la - ln;
}

// One workgroup per (scan point, laser point) pair and bin tile.  Lane j of
// the workgroup (0 <= j < 256) walks its own run of c = ceil(n / 256)
// consecutive occupied voxels, entries j * c .. j * c + c - 1, loading the
// next entry while it bins the current one.  So the 64 lanes of a wave work
// on voxels spread over the whole list at each step.  Batches whose
// occupancy holds an infinity or a NaN take float histograms instead (LDS
// float atomics), so that those values propagate as in the reference.
__global__ __launch_bounds__(kR2Waves * 64) void r2_forward_kernel(
    const float4* __restrict__ geo, const float* __restrict__ occ,
    const int* __restrict__ totals, const unsigned* __restrict__ amax,
    const float* __restrict__ scan,                                   // [B][3][S]
    const float* __restrict__ laser,                                  // [B][3][L]
    float* __restrict__ transient,                                    // [B][T][S][L]
    ExGeom g, int S, int L, int tile) {
  extern __shared__ long long hist64[];  // [kR2Waves][tile]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b = blockIdx.y;
  const int pair = blockIdx.x;
  const int s = pair / L, l = pair - s * L;
  const int nvox = g.D * g.H * g.W;
  const int t0 = (int)blockIdx.z * tile;  // this block's bins t0 .. t0 + tn - 1
  const int tn = min(tile, g.T - t0);
  const int n = totals[b];
  const float am = __uint_as_float(amax[b]);
  // fixed point unless the largest |occupancy| is subnormal, inf or NaN
  // (or zero: no occupied voxel)
  const bool fixed = am >= 1.17549435e-38f && am < INFINITY;
  const int e = fixed ? r2_exponent(am, n) : 0;
  long long* h = hist64 + wave * tile;
  float* hf = (float*)hist64 + wave * tile;
  for (int t = lane; t < tn; t += 64) {
    if (fixed)
      h[t] = 0;
    else
      hf[t] = 0.f;
  }
  const float spx = scan[(size_t)b * 3 * S + s], spy = scan[(size_t)b * 3 * S + S + s],
              spz = scan[(size_t)b * 3 * S + 2 * S + s];
  const float lpx = laser[(size_t)b * 3 * L + l], lpy = laser[(size_t)b * 3 * L + L + l],
              lpz = laser[(size_t)b * 3 * L + 2 * L + l];
  const float4* gb = geo + (size_t)b * nvox;
  const float* ob = occ + (size_t)b * nvox;
  const bool mid = ex_point_mid(g, spx, spy, spz) && ex_point_mid(g, lpx, lpy, lpz);
  const int c = (n + kR2Waves * 64 - 1) / (kR2Waves * 64);
  const int k0 = (int)threadIdx.x * c, k1 = min(k0 + c, n);
  float4 f = k0 < k1 ? gb[k0] : make_float4(0.f, 0.f, 0.f, 0.f);
  float o = k0 < k1 ? ob[k0] : 0.f;
  for (int j = 0; j < c; ++j) {
    const int k = k0 + j;
    const float4 fn = k + 1 < k1 ? gb[k + 1] : make_float4(0.f, 0.f, 0.f, 0.f);
    const float on = k + 1 < k1 ? ob[k + 1] : 0.f;
    if (k < k1) {
      const Span sp = mid ? voxel_span<true>(g, o, f.x, f.y, f.z, f.w, spx, spy, spz, lpx, lpy, lpz)
                          : voxel_span<false>(g, o, f.x, f.y, f.z, f.w, spx, spy, spz, lpx, lpy,
                                              lpz);
      // The span's bins inside this tile, in increasing order: wf at the
      // first bin, wl at the last (when it differs), wm between.
      const int lo = max(sp.first, t0), hi = min(sp.last, t0 + tn - 1);
      if (fixed) {
        const long long qf = r2_fixed(sp.wf, e), qm = r2_fixed(sp.wm, e),
                        ql = r2_fixed(sp.wl, e);
        for (int bn = lo; bn <= hi; ++bn) {
          const long long q = bn == sp.first ? qf : (bn == sp.last ? ql : qm);
          atomicAdd((unsigned long long*)(h + (bn - t0)), (unsigned long long)q);
        }
      } else {
        for (int bn = lo; bn <= hi; ++bn) {
          const float wgt = bn == sp.first ? sp.wf : (bn == sp.last ? sp.wl : sp.wm);
          atomicAdd(hf + (bn - t0), wgt);
        }
      }
    }
    f = fn;
    o = on;
  }
  __syncthreads();
  // Sum of the wave histograms; one write per bin.
  float* out = transient + (size_t)b * g.T * S * L;
  for (int t = threadIdx.x; t < tn; t += blockDim.x) {
    float v;
    if (fixed) {
      long long q = hist64[t];
      for (int w = 1; w < kR2Waves; ++w) q += hist64[w * tile + t];
      v = (float)ldexp((double)q, -e);
    } else {
      const float* hv = (const float*)hist64;
      v = hv[t];
      for (int w = 1; w < kR2Waves; ++w) v += hv[w * tile + t];
    }
    out[((size_t)(t0 + t) * S + s) * L + l] = v;
  }
}

// ---- A5 -------------------------------------------------------------------
// A voxel's share of a pair is wf g[first] + wm (g between) + wl g[last].
// Short spans (K > 0: first and last at most K bins apart) read the K - 1
// bins after the first at fixed offsets and mask them, without a loop.  For
// longer ones (K = 0) the rows are kept as running sums
// C[t] = g[0] + .. + g[t - 1] in double as well: three differences of four
// neighbouring entries give g[first], the sum between and g[last] for spans
// of any length.  The sums are formed in two doubles and rounded once, so a
// difference is off by at most 2^-52 of the row's largest |C|, and exact over
// empty bins.  A row where that exceeds 2^-24 of its smallest nonzero bin, or
// that holds an infinity or a NaN, is marked: its running sums are zeros, and
// its pairs add the bins (a5_marked_kernel).  Of rows of 1,000 normal deviates
// about one in 5,000 is marked; a batch of many marked rows takes the short
// form, which adds the bins of long spans from LDS.

// Row stride of the transposed gradient: whole float4s.
__host__ __device__ __forceinline__ int a5_row(int T) { return (T + 3) & ~3; }

// Row stride of the running sums: T + 1 rounded up to whole pairs.
__host__ __device__ __forceinline__ int a5_stride(int T) { return (T + 2) & ~1; }

struct A5Rows {
  const float* g;     // [B][S*L][a5_row(T)] the transposed gradient
  double* c;          // [B][S*L][a5_stride(T)] its running sums, or null
  int* marked;        // [B][S*L] whether a row's running sums are left out
  int* count;         // [B] marked rows
};

// The batches a launch takes, by their marked rows.
enum A5Take { kA5All, kA5Few, kA5Many };

// Adding bins in the short form takes about as long as everything else at one
// marked row in 32.
__device__ __forceinline__ bool a5_many(int count, int rows) { return count > rows / 32; }

// The rows, the point headers (which masked reads past the last row may touch)
// and the count come first; the running sums and the marks, two thirds of the
// whole, are needed by long spans only, and add the bins without them.
struct A5Layout {
  size_t head, count, least, prefix, marked, end;
};

A5Layout a5_layout(int64_t B, int64_t T, int64_t S, int64_t L) {
  A5Layout l;
  l.head = align256((size_t)B * S * L * a5_row((int)T) * sizeof(float));
  l.count = l.head + align256((size_t)B * (S + L) * sizeof(float4));
  l.least = l.count + align256((size_t)B * sizeof(int));
  l.prefix = l.least;
  l.marked = l.prefix + align256((size_t)B * S * L * a5_stride((int)T) * sizeof(double));
  l.end = l.marked + align256((size_t)B * S * L * sizeof(int));
  return l;
}

// An unevaluated sum of two doubles, |lo| at most half an ulp of hi.
struct Sum2 {
  double hi, lo;
};

__device__ __forceinline__ Sum2 add2(const Sum2& a, const Sum2& b) {
  const double s = a.hi + b.hi, v = s - a.hi;
  const double e = ((a.hi - (s - v)) + (b.hi - v)) + (a.lo + b.lo);
  Sum2 r;
  r.hi = s + e;
  r.lo = e - (r.hi - s);
  return r;
}

// One wave per row, eight bins per lane and step.
__device__ __forceinline__ void a5_prefix_row(const A5Rows& rows, const ExGeom& g, int n_rows,
                                              size_t r) {
  const int lane = threadIdx.x & 63;
  const float* src = rows.g + r * a5_row(g.T);
  double* dst = rows.c + r * a5_stride(g.T);
  Sum2 base = {0.0, 0.0};
  bool finite = true;
  float least = INFINITY;  // smallest nonzero |bin|
  double most = 0.0;       // largest |running sum|
  for (int t0 = 0; t0 < g.T; t0 += 512) {
    Sum2 s[8], sum = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t = t0 + lane * 8 + k;
      const float v = t < g.T ? src[t] : 0.f, m = fabsf(v);
      finite = finite && m < INFINITY;
      least = m > 0.f ? fminf(least, m) : least;
      s[k] = sum;
      sum = add2(sum, Sum2{(double)v, 0.0});
    }
    Sum2 up = sum;  // inclusive sum over the lanes
    for (int m = 1; m < 64; m <<= 1) {
      const Sum2 o = {__shfl_up(up.hi, m, 64), __shfl_up(up.lo, m, 64)};
      if (lane >= m) up = add2(up, o);
    }
    Sum2 before = {__shfl_up(up.hi, 1, 64), __shfl_up(up.lo, 1, 64)};
    before = lane > 0 ? add2(base, before) : base;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t = t0 + lane * 8 + k;
      const double v = add2(before, s[k]).hi;
      if (t < g.T) dst[t] = v;
      most = fmax(most, fabs(v));
    }
    base = add2(base, Sum2{__shfl(up.hi, 63, 64), __shfl(up.lo, 63, 64)});
  }
  if (lane == 0) dst[g.T] = base.hi;
  most = fmax(most, fabs(base.hi));
  for (int m = 32; m >= 1; m >>= 1) {
    least = fminf(least, __shfl_xor(least, m, 64));
    most = fmax(most, __shfl_xor(most, m, 64));
  }
  const bool mark = __any(!finite) || most > 0x1p28 * (double)least;
  if (mark)
    for (int t = lane; t <= g.T; t += 64) dst[t] = 0.0;
  if (lane != 0) return;
  rows.marked[r] = mark ? 1 : 0;
  if (mark) atomicAdd(rows.count + r / n_rows, 1);
}

__global__ __launch_bounds__(256) void a5_prefix_kernel(A5Rows rows, ExGeom g, int n_rows) {
  for (size_t r = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6); r < (size_t)g.B * n_rows;
       r += (size_t)gridDim.x * 4)
    a5_prefix_row(rows, g, n_rows, r);
}

__global__ void zero_f32_kernel(float* __restrict__ out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[(size_t)blockIdx.y * n + i] = 0.f;
}

// Gradient of one (voxel, pair) from its two path lengths, bin by bin (U at a
// time), in the reference's arithmetic (volume_cuda.cu:341-374), unit
// occupancy.  The bins between are added in double: in float, spans of hundreds
// of bins lose two digits.
template <int U>
__device__ __forceinline__ float a5_pair_any(const ExGeom& g, float d0, float d1,
                                             const float* row) {
  const Span sp = span_of(g, 1.f, d0, d1);
  if (sp.first > sp.last) return 0.f;
  if (sp.first == sp.last) return sp.wf * row[sp.first];
  double m = 0.0;
  for (int bn = sp.first + 1; bn < sp.last; bn += U) {
    float v[U];
#pragma unroll
    for (int k = 0; k < U; ++k) v[k] = row[min(bn + k, sp.last)];
#pragma unroll
    for (int k = 0; k < U; ++k) m += bn + k < sp.last ? (double)v[k] : 0.0;
  }
  return sp.wf * row[sp.first] + sp.wm * (float)m + sp.wl * row[sp.last];
}

// The marked rows of batches with few, added to the running sums' result: a lane
// per voxel, in row order.
__global__ __launch_bounds__(64) void a5_marked_kernel(A5Rows rows,
                                                       const float4* __restrict__ head,
                                                       float* __restrict__ grad, ExGeom g, int S,
                                                       int L) {
  const int b = blockIdx.y, n_rows = S * L, lane = threadIdx.x;
  const int n = rows.count[b];
  if (n == 0 || a5_many(n, n_rows)) return;
  const int nvox = g.D * g.H * g.W;
  const int v = (int)blockIdx.x * 64 + lane;
  const int vv = v < nvox ? v : 0;
  float xf, yf, zf0, zf1;
  voxel_faces(g, vv % g.W, (vv / g.W) % g.H, vv / (g.W * g.H), &xf, &yf, &zf0, &zf1);
  const float4* hs = head + (size_t)b * (S + L);
  const int* marked = rows.marked + (size_t)b * n_rows;
  float acc = 0.f;
  for (int r0 = 0; r0 < n_rows; r0 += 64) {
    unsigned long long todo = __ballot(r0 + lane < n_rows && marked[r0 + lane] != 0);
    for (; todo != 0; todo &= todo - 1) {
      const int r = r0 + (int)__builtin_ctzll(todo);
      const int s = r / L;
      const float4 ps = hs[s], pl = hs[S + r - s * L];
      const float d0 = dist3(ps.x, ps.y, ps.z, xf, yf, zf0) + dist3(pl.x, pl.y, pl.z, xf, yf, zf0);
      const float d1 = dist3(ps.x, ps.y, ps.z, xf, yf, zf1) + dist3(pl.x, pl.y, pl.z, xf, yf, zf1);
      acc += a5_pair_any<8>(g, d0, d1, rows.g + ((size_t)b * n_rows + r) * a5_row(g.T));
    }
  }
  if (v < nvox) grad[(size_t)b * nvox + v] += acc;
}

constexpr int kA5Pairs = 8;  // (scan, laser) pairs of a unit, at most
constexpr int kA5Slack = 8;  // floats past the staged rows that masked reads may touch

// One lane per voxel.  For each tile of KT laser points a lane keeps the
// tile's distances to the voxel's two faces in registers and walks the scan
// points in units of SG, so a pair costs two sums where each pair's four
// correctly rounded roots had taken a third of the kernel; the bin positions
// are exact divisions by a constant (DivConst).  A unit's rows lie in LDS
// (STAGED, U units per stage) or in global memory (long rows).  Units with a
// span that is clipped at the histogram's ends, or longer than K, take a
// second form (per wave).
//
// VALU issue bounds it.  64^3 voxels, 256 x 16 pairs, 512 bins (spans up to 6
// bins): 1.37 ms a call with K = 6 and 1.50 with running sums, against 5.3 ms
// with four roots and a loop over the bins per pair; 16 x 64 x 64 voxels,
// 144 x 16 pairs, 1000 bins (spans up to 34 bins), render included: 0.91 ms
// with running sums, 4.03 with the loop as the second form, 4.46 before.
//
// Off holds the offsets between a unit's rows; 64 bits only where 32 do not
// hold them (fewer loads are then in flight: 0.65 ms instead of 0.49 at 16 x 64
// x 64 voxels, 144 x 16 pairs, 3,000 bins).
template <int K, int KT, bool STAGED, int NTH, typename Off = int>
__global__ __launch_bounds__(NTH) void r2_adjoint_kernel(
    A5Rows rows, const float4* __restrict__ head,  // [B][S + L]
    float* __restrict__ grad,                      // [B][D][H][W]
    ExGeom g, int S, int L, int U, int cap, DivConst dw, int take) {
  extern __shared__ float4 lds4[];
  constexpr int SG = kA5Pairs / KT > 1 ? kA5Pairs / KT : 1;
  const int b = blockIdx.y;
  if (take != kA5All && a5_many(rows.count[b], S * L) != (take == kA5Many)) return;
  const int nvox = g.D * g.H * g.W;
  const Off P = K > 0 ? (Off)a5_row(g.T) : 2 * (Off)a5_stride(g.T);  // floats of a row
  const int v = blockIdx.x * NTH + threadIdx.x;
  const bool ok = v < nvox;
  const int vv = ok ? v : 0;
  const int xi = vv % g.W, yi = (vv / g.W) % g.H, zi = vv / (g.W * g.H);
  float xf, yf, zf0, zf1;
  voxel_faces(g, xi, yi, zi, &xf, &yf, &zf0, &zf1);
  const float4* hs = head + (size_t)b * (S + L);
  const float4* hl = hs + S;
  const float* gb = rows.g + (size_t)b * S * L * a5_row(g.T);
  const float* cb = K > 0 ? gb : (const float*)(rows.c + (size_t)b * S * L * a5_stride(g.T));
  float* stage = (float*)lds4;
  const int n_units = (S + SG - 1) / SG;
  // distances of n points (uniform) to the voxel's faces
  auto faces = [&](auto at, auto& d0, auto& d1, auto n) {
    float mid = 1.f;
#pragma unroll
    for (int j = 0; j < n; ++j) mid = fminf(mid, at(j).w);
    if (mid != 0.f) {
#pragma unroll
      for (int j = 0; j < n; ++j) {
        d0[j] = ex_dist<true>(at(j).x, at(j).y, at(j).z, xf, yf, zf0);
        d1[j] = ex_dist<true>(at(j).x, at(j).y, at(j).z, xf, yf, zf1);
      }
    } else {
#pragma unroll
      for (int j = 0; j < n; ++j) {
        d0[j] = ex_dist<false>(at(j).x, at(j).y, at(j).z, xf, yf, zf0);
        d1[j] = ex_dist<false>(at(j).x, at(j).y, at(j).z, xf, yf, zf1);
      }
    }
  };
  // The weighted bins of a span; x0 <= x1 are the clipped bin positions of
  // the faces, f = floor(x0), l = floor(x1), range their unclipped difference.
  auto weigh = [&](const float* row, float x0, float x1, int f, int l, float range) {
    float first, in, last;
    if constexpr (K > 0) {
      const float* r = row + f;
      const int m = l - f;
      first = r[0];
      last = r[m];
      in = 0.f;
#pragma unroll
      for (int k = 1; k < K; ++k) {
        const float val = r[k];
        in += k < m ? val : 0.f;
      }
    } else {
      const double* c = (const double*)row;
      const double c0 = c[f], c1 = c[f + 1], c2 = c[l], c3 = c[l + 1];
      first = (float)(c1 - c0);
      in = (float)(c2 - c1);
      last = (float)(c3 - c2);
    }
    float frac = __builtin_amdgcn_rcpf(range);
    frac = fmaf(fmaf(-range, frac, 1.f), frac, frac);
    const float wf = 1.f - (x0 - (float)f), wl = x1 - (float)l;
    const float sum = fmaf(wf, first, fmaf(wl, last, in)) * frac;
    return f == l ? first : sum;
  };

  float acc = 0.f;
  for (int l0 = 0; l0 < L; l0 += KT) {
    const int nl = min(KT, L - l0);
    float dl0[KT], dl1[KT];
    faces([&](int j) { return hl[min(l0 + j, L - 1)]; }, dl0, dl1,
          std::integral_constant<int, KT>{});
    // rows of scan points s0 .. : nl consecutive rows each, L rows apart,
    // packed in the stage
    RowStage<NTH> next;
    const int n4s = STAGED ? (int)(nl * P / 4) : 0;  // float4s per scan point
    auto points = [&](int u) { return min(U * SG, S - u * SG); };
    auto load = [&](int u) {
      next.load_pieces(cb + ((size_t)u * SG * L + l0) * P, points(u) * n4s, n4s,
                       (int64_t)L * P / 4);
    };
    auto put = [&](int u, int buf) { next.store(stage + buf * cap, points(u) * n4s); };
    if (STAGED) {
      load(0);
      put(0, 0);
      if (U < n_units) load(U);
      __syncthreads();
    }
    int cur = 0;
    for (int u0 = 0; u0 < n_units; u0 += U) {
      const int ue = min(u0 + U, n_units);
      if (STAGED && ue < n_units) {
        put(ue, cur ^ 1);
        if (ue + U < n_units) load(ue + U);
      }
      for (int u = u0; u < ue; ++u) {
        const int s0 = u * SG, ns = min(SG, S - s0);
        // row of pair (s0 + i, l0 + j)
        const float* base = STAGED ? stage + cur * cap + (u - u0) * SG * nl * P
                                   : cb + ((size_t)s0 * L + l0) * P;
        const Off si = SG > 1 ? (STAGED ? nl : L) * P : 0;
        float ds0[SG], ds1[SG];
        faces([&](int i) { return hs[min(s0 + i, S - 1)]; }, ds0, ds1,
              std::integral_constant<int, SG>{});
        if (dw.ok && take != kA5Many) {  // (most units of those add the bins)
          float x0[SG][KT], x1[SG][KT];
          int f[SG][KT], l[SG][KT];
          bool clipped = ns < SG || nl < KT, odd = false;
#pragma unroll
          for (int i = 0; i < SG; ++i)
#pragma unroll
            for (int j = 0; j < KT; ++j) {
              const float a = ds0[i] + dl0[j], c = ds1[i] + dl1[j];
              x0[i][j] = div_const(fminf(a, c) - g.off, dw);                  // :341-347
              x1[i][j] = div_const(fmaxf(a, c) - g.off, dw);
              f[i][j] = floor_to_int(x0[i][j]);                               // :349-350
              l[i][j] = floor_to_int(x1[i][j]);
              clipped |= f[i][j] < 0 | l[i][j] >= g.T;
              if (K > 0) clipped |= l[i][j] - f[i][j] > K;
              odd |= !(x1[i][j] - x0[i][j] < 0x1p60f);  // NaN or infinite
            }
          if (!__any(clipped | odd)) {
#pragma unroll
            for (int i = 0; i < SG; ++i)
#pragma unroll
              for (int j = 0; j < KT; ++j)
                acc += weigh(base + i * si + j * P, x0[i][j], x1[i][j], f[i][j], l[i][j],
                             x1[i][j] - x0[i][j]);
            continue;
          }
          if (K == 0 && !__any(odd)) {
#pragma unroll
            for (int i = 0; i < SG; ++i)
#pragma unroll
              for (int j = 0; j < KT; ++j)
                if (i < ns && j < nl) {
                  const bool empty = l[i][j] < 0 || f[i][j] >= g.T;           // :351-364
                  const float range = x1[i][j] - x0[i][j];
                  const float e1 = l[i][j] >= g.T ? (float)(g.T - 1) : x1[i][j];
                  const float sum = weigh(base + i * si + j * P, fmaxf(x0[i][j], 0.f), e1,
                                          min(max(f[i][j], 0), g.T - 1),
                                          min(max(l[i][j], 0), g.T - 1), range);
                  acc += empty ? 0.f : sum;
                }
            continue;
          }
        }
        const float* any = K > 0 ? base : gb + ((size_t)s0 * L + l0) * a5_row(g.T);
        const int64_t ai = K > 0 || SG == 1 ? (int64_t)si : (int64_t)L * a5_row(g.T);
#pragma unroll
        for (int i = 0; i < SG; ++i)
#pragma unroll
          for (int j = 0; j < KT; ++j)
            if (i < ns && j < nl &&
                !(K == 0 && rows.marked[((size_t)b * S + s0 + i) * L + l0 + j]))
              acc += a5_pair_any<1>(g, ds0[i] + dl0[j], ds1[i] + dl1[j],
                                 any + i * ai + j * (Off)a5_row(g.T));
      }
      if (STAGED) {
        __syncthreads();
        cur ^= 1;
      }
    }
  }
  if (ok) grad[(size_t)b * nvox + v] = acc;
}

template <int K, int KT>
int a5_launch_tile(const A5Rows& rows, const float4* head, float* grad, const ExGeom& g,
                   int64_t S, int64_t L, const StagePlan& sp, int64_t P, int take,
                   hipStream_t st) {
  constexpr int SG = kA5Pairs / KT > 1 ? kA5Pairs / KT : 1;
  const int64_t n = (int64_t)SG * std::min<int64_t>(KT, L);  // rows of a unit
  // masked reads may touch K floats past the last row
  const int64_t U = std::min<int64_t>((S + SG - 1) / SG, (sp.cap - kA5Slack) / (n * P));
  auto kernel = sp.threads == 1024 ? r2_adjoint_kernel<K, KT, true, 1024>
                                   : r2_adjoint_kernel<K, KT, true, 256>;
  const int rc = allow_stage(kernel);
  if (rc) return rc;
  const unsigned blocks = (unsigned)(((size_t)g.D * g.H * g.W + sp.threads - 1) / sp.threads);
  hipLaunchKernelGGL(kernel, dim3(blocks, (unsigned)g.B), dim3(sp.threads),
                     2 * (size_t)sp.cap * sizeof(float), st, rows, head, grad, g, (int)S, (int)L,
                     (int)U, sp.cap, make_div_const(g.w), take);
  return check_launch("r2_adjoint_kernel");
}

// The stage and the laser points per tile of rows of P floats; 0 where the
// rows of a unit do not fit.
int a5_tile(const ExGeom& g, int64_t L, int64_t P, StagePlan* sp) {
  *sp = stage_plan(g.B, (int64_t)g.D * g.H * g.W);
  // fewer, larger buffers rather than rows from global memory
  if (kA5Pairs * P > sp->cap - kA5Slack) sp->cap = kStageMax;
  const int64_t fit = (sp->cap - kA5Slack) / P;
  // The tile with the least work: every slot of a tile costs a pair (about
  // 50 instructions), every scan point of a tile two roots (about 35).
  static const int sizes[] = {1, 2, 3, 4, 6, 8};
  int kt = 0;
  int64_t least = 0;
  for (int k : sizes) {
    if ((int64_t)(kA5Pairs / k) * std::min<int64_t>(k, L) > fit) continue;
    const int64_t cost = (L + k - 1) / k * (50 * k + 35);
    if (kt == 0 || cost <= least) {
      kt = k;
      least = cost;
    }
  }
  return kt;
}

// Floats of a row that a stage holds, by form.
template <int K>
int64_t a5_floats(int T) {
  return K > 0 ? a5_row(T) : 2 * (int64_t)a5_stride(T);
}

template <int K>
int a5_launch_form(const A5Rows& rows, const float4* head, float* grad, const ExGeom& g,
                   int64_t S, int64_t L, int take, hipStream_t st) {
  const int64_t P = a5_floats<K>(g.T);
  StagePlan sp;
  const int kt = a5_tile(g, L, P, &sp);
  if (kt == 1) return a5_launch_tile<K, 1>(rows, head, grad, g, S, L, sp, P, take, st);
  if (kt == 2) return a5_launch_tile<K, 2>(rows, head, grad, g, S, L, sp, P, take, st);
  if (kt == 3) return a5_launch_tile<K, 3>(rows, head, grad, g, S, L, sp, P, take, st);
  if (kt == 4) return a5_launch_tile<K, 4>(rows, head, grad, g, S, L, sp, P, take, st);
  if (kt == 6) return a5_launch_tile<K, 6>(rows, head, grad, g, S, L, sp, P, take, st);
  if (kt == 8) return a5_launch_tile<K, 8>(rows, head, grad, g, S, L, sp, P, take, st);
  // rows too long for the stage: from global memory
  const int64_t nvox = (int64_t)g.D * g.H * g.W;
  auto kernel = 8 * P < (1ll << 31) ? r2_adjoint_kernel<K, 8, false, 256>
                                    : r2_adjoint_kernel<K, 8, false, 256, int64_t>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)((nvox + 255) / 256), (unsigned)g.B), dim3(256), 0,
                     st, rows, head, grad, g, (int)S, (int)L, (int)S, 0, make_div_const(g.w),
                     take);
  return check_launch("r2_adjoint_kernel");
}

// The form (K) of a call.  A voxel's faces are at most 2 dz / w bins apart
// (each leg of a path changes by at most the voxel's height), so their bins at
// most floor(2 dz / w) + 1.  A wrong guess costs the second form, no error.
int a5_form(const ExGeom& g, int64_t L) {
  const double bins = 2.0 * fabs((double)g.ez - g.sz) / g.D / (double)g.w;
  StagePlan sp;
  if (a5_tile(g, L, a5_floats<6>(g.T), &sp) == 0) return 0;
  return bins < 1.99 ? 2 : bins < 5.95 ? 6 : 0;
}

int a5_launch(const A5Rows& rows, const float4* head, float* grad, const ExGeom& g, int64_t S,
              int64_t L, hipStream_t st) {
  const int form = a5_form(g, L);
  if (form == 2) return a5_launch_form<2>(rows, head, grad, g, S, L, kA5All, st);
  if (form == 6 || rows.c == nullptr)
    return a5_launch_form<6>(rows, head, grad, g, S, L, kA5All, st);
  const int64_t blocks = (g.B * S * L + 3) / 4;
  hipLaunchKernelGGL(a5_prefix_kernel, dim3((unsigned)(blocks < (1 << 22) ? blocks : 1 << 22)),
                     dim3(256), 0, st, rows, g, (int)(S * L));
  int rc = check_launch("a5_prefix_kernel");
  if (rc) return rc;
  rc = a5_launch_form<0>(rows, head, grad, g, S, L, kA5Few, st);
  if (rc) return rc;
  rc = a5_launch_form<6>(rows, head, grad, g, S, L, kA5Many, st);
  if (rc) return rc;
  const int64_t nvox = (int64_t)g.D * g.H * g.W;
  hipLaunchKernelGGL(a5_marked_kernel, dim3((unsigned)((nvox + 63) / 64), (unsigned)g.B), dim3(64),
                     0, st, rows, head, grad, g, (int)S, (int)L);
  return check_launch("a5_marked_kernel");
}

ExGeom ex_geom(int64_t B, int64_t D, int64_t H, int64_t W, int64_t T, const float* vs,
               const float* ve, float w, float off) {
  ExGeom g;
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

int check_sizes(int64_t B, int64_t D, int64_t H, int64_t W, int64_t T, int64_t S, int64_t L) {
  for (int64_t d : {B, D, H, W, T, S, L})
    TOTRI_CHECK_ARG(d >= 0 && d < (1ll << 31), "dimension out of range");
  TOTRI_CHECK_ARG(B * D * H * W < (1ll << 31) && B * T * S * L < (1ll << 31),
                  "tensor has more than 2^31 elements");
  return TOTRI_OK;
}

}  // namespace
}  // namespace totri_hip

using namespace totri_hip;

namespace totri_hip {
namespace {

// Workspace of R2: the compaction, then the occupied voxels' geometry
// (float4) and occupancy, [B][D*H*W] each, and the largest |occupancy| of
// each batch.
struct R2Layout {
  CompactLayout cl;
  size_t geo_off, occ_off, amax_off, end;
};

R2Layout r2_layout(int64_t B, int64_t nvox) {
  R2Layout l;
  l.cl = compact_layout(B, nvox, 0);
  l.geo_off = align256(l.cl.end);
  l.occ_off = align256(l.geo_off + (size_t)B * nvox * sizeof(float4));
  l.amax_off = align256(l.occ_off + (size_t)B * nvox * sizeof(float));
  l.end = align256(l.amax_off + (size_t)B * sizeof(unsigned));
  return l;
}

}  // namespace
}  // namespace totri_hip

extern "C" size_t totri_volume_render_exhaustive_forward_workspace(int64_t B, int64_t D,
                                                                   int64_t H, int64_t W) {
  return r2_layout(B, D * H * W).end;
}

extern "C" int totri_volume_render_exhaustive_forward(
    const float* volume, int64_t B, int64_t D, int64_t H, int64_t W, const float* scan_points,
    int64_t S, const float* laser_points, int64_t L, float* transient, int64_t T,
    const float volume_start[3], const float volume_end[3], float bin_width,
    float bin_offset, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_sizes(B, D, H, W, T, S, L);
  if (rc) return rc;
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  hipStream_t st = (hipStream_t)stream;
  if (B == 0 || T == 0 || S == 0 || L == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(transient && scan_points && laser_points, "null input");
  const size_t nvox = (size_t)D * H * W;
  const ExGeom g = ex_geom(B, D, H, W, T, volume_start, volume_end, bin_width, bin_offset);
  const size_t need = totri_volume_render_exhaustive_forward_workspace(B, D, H, W);
  if (workspace_bytes < need)
    return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", need,
                workspace_bytes);
  TOTRI_CHECK_ARG(workspace != nullptr, "null workspace");
  TOTRI_CHECK_ARG(nvox == 0 || volume != nullptr, "null volume");
  TOTRI_CHECK_ARG(((uintptr_t)workspace & 15) == 0, "workspace must be 16-byte aligned");
  const R2Layout lay = r2_layout(B, (int64_t)nvox);
  const CompactLayout& cl = lay.cl;
  char* ws = (char*)workspace;
  const int* totals = (const int*)(ws + cl.totals_off);
  const int* list = (const int*)(ws + cl.list_off);
  float4* geo = (float4*)(ws + lay.geo_off);
  float* occ = (float*)(ws + lay.occ_off);
  unsigned* amax = (unsigned*)(ws + lay.amax_off);
  TOTRI_CHECK_ARG(B <= 65535, "B=%lld too large", (long long)B);
  hipLaunchKernelGGL(zero_u32_kernel, dim3((unsigned)((B + 255) / 256)), dim3(256), 0, st, amax,
                     (int)B);
  rc = check_launch("zero_u32_kernel");
  if (rc) return rc;
  if (nvox > 0) {
    rc = launch_compact(volume, (int)B, (int)nvox, cl, workspace, NonZero(), st);
    if (rc) return rc;
    hipLaunchKernelGGL(r2_voxels_kernel, dim3((unsigned)((nvox + 255) / 256), (unsigned)B),
                       dim3(256), 0, st, volume, list, totals, g, geo, occ, amax);
    rc = check_launch("r2_voxels_kernel");
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(compact_scan_kernel, dim3((unsigned)B), dim3(kCompactScanLanes), 0, st,
                       (int*)(ws + cl.counts_off), 0, (int*)(ws + cl.totals_off));
    rc = check_launch("compact_scan_kernel");
    if (rc) return rc;
  }
  const int tile = T < kR2Tile ? (int)T : kR2Tile;
  const int64_t tiles = (T + tile - 1) / tile;
  TOTRI_CHECK_ARG(S * L < (1ll << 31) && tiles <= 65535,
                  "launch grid too large (S*L=%lld, %lld bin tiles)", (long long)(S * L),
                  (long long)tiles);
  hipLaunchKernelGGL(r2_forward_kernel, dim3((unsigned)(S * L), (unsigned)B, (unsigned)tiles),
                     dim3(kR2Waves * 64), (size_t)kR2Waves * tile * sizeof(long long), st, geo,
                     occ, totals, amax, scan_points, laser_points, transient, g, (int)S, (int)L,
                     tile);
  return check_launch("r2_forward_kernel");
}

extern "C" size_t totri_volume_render_exhaustive_grad_volume_workspace(int64_t B, int64_t T,
                                                                       int64_t S, int64_t L) {
  if (B <= 0 || T < 0 || S <= 0 || L <= 0) return 0;
  return a5_layout(B, T, S, L).least;
}

extern "C" size_t totri_volume_render_exhaustive_grad_volume_workspace_box(
    int64_t B, int64_t T, int64_t S, int64_t L, int64_t D, int64_t H, int64_t W,
    const float volume_start[3], const float volume_end[3], float bin_width) {
  if (B <= 0 || T < 0 || S <= 0 || L <= 0 || !volume_start || !volume_end) return 0;
  const A5Layout l = a5_layout(B, T, S, L);
  if (T == 0 || D <= 0 || H <= 0 || W <= 0) return l.least;
  const ExGeom g = ex_geom(B, D, H, W, T, volume_start, volume_end, bin_width, 0.f);
  return a5_form(g, L) == 0 ? l.end : l.least;
}

extern "C" int totri_volume_render_exhaustive_grad_volume(
    const float* transient_grad, int64_t B, int64_t T, int64_t S, int64_t L,
    const float* scan_points, const float* laser_points, float* volume_grad, int64_t D,
    int64_t H, int64_t W, const float volume_start[3], const float volume_end[3],
    float bin_width, float bin_offset, void* workspace, size_t workspace_bytes,
    void* stream) {
  int rc = check_sizes(B, D, H, W, T, S, L);
  if (rc) return rc;
  TOTRI_CHECK_ARG(volume_start && volume_end, "null volume box");
  TOTRI_CHECK_ARG(T < (1 << 30), "T=%lld too large", (long long)T);
  hipStream_t st = (hipStream_t)stream;
  const size_t nvox = (size_t)D * H * W;
  if (B == 0 || nvox == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume_grad != nullptr, "null volume_grad");
  const ExGeom g = ex_geom(B, D, H, W, T, volume_start, volume_end, bin_width, bin_offset);
  const dim3 grid((unsigned)((nvox + 255) / 256), (unsigned)B);
  if (T == 0 || S == 0 || L == 0) {  // no bins or no pairs: a zero gradient
    hipLaunchKernelGGL(zero_f32_kernel, grid, dim3(256), 0, st, volume_grad, (int)nvox);
    return check_launch("zero_f32_kernel");
  }
  TOTRI_CHECK_ARG(transient_grad && scan_points && laser_points, "null input");
  const size_t need = totri_volume_render_exhaustive_grad_volume_workspace(B, T, S, L);
  if (workspace_bytes < need)
    return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", need,
                workspace_bytes);
  TOTRI_CHECK_ARG(workspace != nullptr && ((uintptr_t)workspace & 15) == 0,
                  "workspace must be a non-null, 16-byte aligned device pointer");
  const A5Layout lay = a5_layout(B, T, S, L);
  char* ws = (char*)workspace;
  A5Rows rows;
  rows.g = (float*)ws;
  rows.c = workspace_bytes >= lay.end ? (double*)(ws + lay.prefix) : nullptr;
  rows.marked = (int*)(ws + lay.marked);
  rows.count = (int*)(ws + lay.count);
  float4* head = (float4*)(ws + lay.head);
  // [B][T][S*L] -> [B][S*L][a5_row(T)]
  rc = transpose_strided(transient_grad, (float*)ws, (int)B, (int)T, (int)(S * L),
                         a5_row((int)T), 0, st);
  if (rc) return rc;
  hipLaunchKernelGGL(ex_point_head_kernel, dim3((unsigned)((B * (S + L) + 255) / 256)), dim3(256),
                     0, st, scan_points, laser_points, (int)S, (int)L, g, head, rows.count);
  rc = check_launch("ex_point_head_kernel");
  if (rc) return rc;
  return a5_launch(rows, head, volume_grad, g, S, L, st);
}

namespace totri_hip {
namespace {

__global__ void sqrt_mid_check_kernel(uint32_t lo, uint32_t hi,
                                      unsigned long long* __restrict__ count) {
  unsigned long long bad = 0;
  const uint64_t n = (uint64_t)hi - lo + 1;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    const float x = __uint_as_float((uint32_t)(lo + i));
    bad += __float_as_uint(sqrt_rn_mid(x)) != __float_as_uint(sqrt_rn(x)) ? 1 : 0;
  }
  for (int m = 32; m >= 1; m >>= 1) bad += __shfl_xor(bad, m, 64);
  if ((threadIdx.x & 63) == 0 && bad) atomicAdd(count, bad);
}

__global__ void zero_u64_kernel(unsigned long long* p) { *p = 0ull; }

}  // namespace
}  // namespace totri_hip

extern "C" int totri_debug_sqrt_mid_mismatches(uint32_t lo_bits, uint32_t hi_bits,
                                               unsigned long long* mismatches, void* stream) {
  TOTRI_CHECK_ARG(mismatches != nullptr && lo_bits <= hi_bits, "invalid arguments");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(zero_u64_kernel, dim3(1), dim3(1), 0, st, mismatches);
  int rc = check_launch("zero_u64_kernel");
  if (rc) return rc;
  hipLaunchKernelGGL(sqrt_mid_check_kernel, dim3(device_cu_count() * 16), dim3(256), 0, st,
                     lo_bits, hi_bits, mismatches);
  return check_launch("sqrt_mid_check_kernel");
}
