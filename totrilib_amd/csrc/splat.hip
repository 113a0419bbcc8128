// Gaussian RBF -> volume splat (S1) and its parameter gradient (S2), gfx950.
//
// Reference: src/util/rbf2volume_cuda.cu:15-232, src/util/rbf2volume.cpp:7-27.
//
//   g_i(q)   = exp(-0.5 |q - c_i|^2 / sigma_i^2)             (:15-29)
//   V0(q)    = sum_i g_i(q)
//   Va(q)    = sum_i g_i(q) a_{i,a} / (V0 < 1e-8 ? 1 : V0)    (:49-93)
// on the inclusive voxel grid from `start` to `end`.  The reference sums all
// N RBFs for every voxel.  Here a truncation radius (in units of sigma) may
// be given: RBFs with |q - c|^2 > (trunc sigma)^2 are skipped (trunc <= 0
// keeps every RBF, which reproduces the reference).
//
// S1, truncated: a workgroup owns a brick of 8 x 8 x 4 voxels (one per lane).
// RBFs are streamed through LDS in chunks; each chunk is culled against the
// brick's bounding box and the survivors are compacted in index order, so
// every voxel sums its RBFs in the reference's order.
//
// S2, truncated: one wave per RBF walks the voxels of the RBF's support box
// and reduces its gradient over the wave in a fixed order; the reference
// instead launches one block per (16 columns x 4 slices, RBF) and adds
// per-block partial sums with float atomics.
//
// Without truncation every RBF reaches every voxel, and a Gaussian on a grid
// is a product of one factor per axis: both directions are contractions on
// the matrix cores (splat_sep_kernel, splat_grad_sep_kernel).
#include <math.h>
#include <string.h>

#include <type_traits>

#include "common.h"

namespace totri_hip {
namespace {

constexpr int kMaxAttr = 8;  // rbf2volume_cuda.cu:13
constexpr int kBX = 8, kBY = 8, kBZ = 4;
constexpr int kChunk = 256;

struct SplatGeom {
  int B, N, A, D, H, W;
  float sx, sy, sz, ex, ey, ez;
  float trunc;
};

// rbf2volume_cuda.cu:58-60: (end - start) * i / (n - 1) + start, or the box
// centre when n == 1.
__device__ __forceinline__ float splat_coord(int i, int n, float a, float b) {
  if (n == 1) return 0.5f * (a + b);
  float t = (b - a) * (float)i;
  t = t / (float)(n - 1);
  return a + t;
}

// |q - c|^2 in the reference's order (rbf2volume_cuda.cu:21-24).
__device__ __forceinline__ float rbf_r2(float x, float y, float z, float xr, float yr,
                                        float zr) {
  float r2 = (xr - x) * (xr - x);
  r2 = r2 + (yr - y) * (yr - y);
  r2 = r2 + (zr - z) * (zr - z);
  return r2;
}

// The Gaussian exp(-r2 / (2 sigma^2)) (rbf2volume_cuda.cu:15-29, written
// there as expf(-0.5 r2 / sigma^2)) as 2^(r2 * k), with the RBF's
// k = -log2(e) / (2 sigma^2) computed once per RBF: the hardware base-2
// exponential (within 1 ulp) of a product rounded once, two instructions
// per (voxel, RBF) instead of a division and expf's expansion.  The result
// differs from the reference's by a relative |r2 k| 2^-23 or so, far inside
// the splat's 1e-5 bar (its terms with |r2 k| above 30 are below 1e-9 of the
// peak).
__device__ __forceinline__ float gauss_k(float sg) { return -0.72134752f / (sg * sg); }

__device__ __forceinline__ float gauss_exp2(float r2, float k) {
  return __builtin_amdgcn_exp2f(r2 * k);
}

// Truncation test: keep the RBF when r2 <= (trunc * sigma)^2.
__device__ __forceinline__ bool within(float r2, float sg, float trunc) {
  const float lim = trunc * sg;
  return !(r2 > lim * lim);
}

// Binned lists (truncated splats): per (batch, brick) the RBFs whose support
// may reach the brick, found with the brick-cull test of the full scan, so a
// brick sums the same RBFs in the same (index) order either way.  Each brick
// has `cap` list slots; a brick reached by more RBFs scans all of them.
struct SplatBins {
  int* count;  // [B][bricks] RBFs that may reach the brick (the fill cursor)
  int* list;   // [B][bricks][cap] the first cap of their indices, in fill order
  int cap;
};

constexpr int kSlotMax = 512;  // list slots per brick, at most (LDS sort buffers)
constexpr int kSlotMin = 64;

// Conservative brick cull (the full scan's test): the squared distance from
// the RBF centre to the brick's sample box against (trunc sigma)^2.
__device__ __forceinline__ bool brick_may_hold(float xr, float yr, float zr, float sg,
                                               float trunc, float lox, float hix, float loy,
                                               float hiy, float loz, float hiz) {
  const float dx = fmaxf(fmaxf(lox - xr, xr - hix), 0.f);
  const float dy = fmaxf(fmaxf(loy - yr, yr - hiy), 0.f);
  const float dz = fmaxf(fmaxf(loz - zr, zr - hiz), 0.f);
  const float lim = trunc * fabsf(sg);
  return !((dx * dx + dy * dy + dz * dz) > lim * lim * 1.0001f + 1e-12f);
}

// The sample box of voxels [x0, x1] x [y0, y1] x [z0, z1] (inclusive, inside
// the grid).
__device__ __forceinline__ void voxel_box(const SplatGeom& g, int x0, int x1, int y0, int y1,
                                          int z0, int z1, float* lox, float* hix, float* loy,
                                          float* hiy, float* loz, float* hiz) {
  const float bxa = splat_coord(x0, g.W, g.sx, g.ex), bxb = splat_coord(x1, g.W, g.sx, g.ex);
  const float bya = splat_coord(y0, g.H, g.sy, g.ey), byb = splat_coord(y1, g.H, g.sy, g.ey);
  const float bza = splat_coord(z0, g.D, g.sz, g.ez), bzb = splat_coord(z1, g.D, g.sz, g.ez);
  *lox = fminf(bxa, bxb);
  *hix = fmaxf(bxa, bxb);
  *loy = fminf(bya, byb);
  *hiy = fmaxf(bya, byb);
  *loz = fminf(bza, bzb);
  *hiz = fmaxf(bza, bzb);
}

// The sample box of brick (bx, by, bz): the voxels it really holds.
__device__ __forceinline__ void brick_box(const SplatGeom& g, int bx, int by, int bz,
                                          float* lox, float* hix, float* loy, float* hiy,
                                          float* loz, float* hiz) {
  const int x0 = bx * kBX, x1 = min(bx * kBX + kBX, g.W) - 1;
  const int y0 = by * kBY, y1 = min(by * kBY + kBY, g.H) - 1;
  const int z0 = bz * kBZ, z1 = min(bz * kBZ + kBZ, g.D) - 1;
  voxel_box(g, x0, x1, y0, y1, z0, z1, lox, hix, loy, hiy, loz, hiz);
}

// Brick index range [lo, hi] along an axis whose bricks hold `bs` samples
// each, covering the samples within [c - r, c + r] (one sample of margin; the
// exact test is brick_may_hold).
__device__ __forceinline__ void brick_range(float c, float r, int n, int bs, float a, float b,
                                            int* lo, int* hi) {
  const int nb = (n + bs - 1) / bs;
  if (n == 1) {
    *lo = 0;
    *hi = nb - 1;
    return;
  }
  const float step = (b - a) / (float)(n - 1);
  float u0 = (c - r - a) / step, u1 = (c + r - a) / step;
  if (u0 > u1) {
    const float t = u0;
    u0 = u1;
    u1 = t;
  }
  u0 = fminf(fmaxf(u0 - 1.f, -1.f), (float)n);
  u1 = fminf(fmaxf(u1 + 1.f, -1.f), (float)n);
  *lo = max((int)floorf(u0), 0) / bs;
  *hi = min((int)ceilf(u1), n - 1) / bs;
  if (!(r < INFINITY)) {
    *lo = 0;
    *hi = nb - 1;
  }
}

// One pass: per brick, the RBFs that may reach it take the next slot of the
// brick's list (the count past cap makes the brick scan instead).  One wave
// per RBF, its lanes over the bricks of the RBF's support box.
constexpr int kBinWaves = 4;

__global__ __launch_bounds__(kBinWaves * 64) void splat_bin_kernel(
    const float* __restrict__ rbf, SplatGeom g, int bricks_x, int bricks_y, int bricks_z,
    SplatBins bins) {
  const int lane = threadIdx.x & 63;
  const int i = blockIdx.x * kBinWaves + (threadIdx.x >> 6);
  const int b = blockIdx.y;
  if (i >= g.N) return;  // whole wave; no barrier follows
  const int C = 4 + g.A;
  const float* p = rbf + ((size_t)b * g.N + i) * C;
  const float xr = p[0], yr = p[1], zr = p[2], sg = p[3];
  const float r = g.trunc * fabsf(sg) * 1.0001f + 1e-6f;
  int xa, xb, ya, yb, za, zb;
  brick_range(xr, r, g.W, kBX, g.sx, g.ex, &xa, &xb);
  brick_range(yr, r, g.H, kBY, g.sy, g.ey, &ya, &yb);
  brick_range(zr, r, g.D, kBZ, g.sz, g.ez, &za, &zb);
  const int nx = xb - xa + 1, ny = yb - ya + 1, nz = zb - za + 1;
  if (nx <= 0 || ny <= 0 || nz <= 0) return;
  const int total = nx * ny * nz;
  const size_t nb = (size_t)bricks_x * bricks_y * bricks_z;
  for (int e = lane; e < total; e += 64) {
    const int bx = xa + e % nx;
    const int by = ya + (e / nx) % ny;
    const int bz = za + e / (nx * ny);
    float lox, hix, loy, hiy, loz, hiz;
    brick_box(g, bx, by, bz, &lox, &hix, &loy, &hiy, &loz, &hiz);
    if (!brick_may_hold(xr, yr, zr, sg, g.trunc, lox, hix, loy, hiy, loz, hiz)) continue;
    const size_t k = b * nb + ((size_t)bz * bricks_y + by) * bricks_x + bx;
    const int at = atomicAdd(bins.count + k, 1);
    if (at < bins.cap) bins.list[k * bins.cap + at] = i;
  }
}

__global__ __launch_bounds__(256) void splat_forward_kernel(
    const float* __restrict__ rbf,  // [B][N][4+A]
    float* __restrict__ vol,        // [B][1+A][D][H][W]
    SplatGeom g, int bricks_x, int bricks_y, SplatBins bins, int binned) {
  __shared__ float prm[kChunk * (4 + kMaxAttr)];
  __shared__ float pk[kChunk];  // gauss_k of the staged RBFs
  __shared__ int keep[kSlotMax > kChunk ? kSlotMax : kChunk];
  __shared__ int fill[kSlotMax];
  __shared__ int wave_cnt[4];
  const int C = 4 + g.A;
  const int b = blockIdx.y;
  int brick = blockIdx.x;
  const int bx = brick % bricks_x;
  brick /= bricks_x;
  const int by = brick % bricks_y;
  const int bz = brick / bricks_y;
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  // Each wave holds a 4x4x4 quarter of the brick (quarter `wave` of its 8x8
  // footprint, all 4 z), so that it can skip the RBFs that miss its quarter.
  static_assert(kBX == 8 && kBY == 8 && kBZ == 4, "four 4x4x4 quarters per brick");
  const int qx0 = bx * kBX + (wave & 1) * 4, qy0 = by * kBY + (wave >> 1) * 4;
  const int xi = qx0 + (lane & 3);
  const int yi = qy0 + ((lane >> 2) & 3);
  const int zi = bz * kBZ + (lane >> 4);
  const bool ok = xi < g.W && yi < g.H && zi < g.D;
  const float x = splat_coord(xi, g.W, g.sx, g.ex);
  const float y = splat_coord(yi, g.H, g.sy, g.ey);
  const float z = splat_coord(zi, g.D, g.sz, g.ez);
  // Brick bounding box over the voxels it really holds.
  float lox, hix, loy, hiy, loz, hiz;
  brick_box(g, bx, by, bz, &lox, &hix, &loy, &hiy, &loz, &hiz);

  float sum = 0.f;
  float attr[kMaxAttr];
#pragma unroll
  for (int a = 0; a < kMaxAttr; ++a) attr[a] = 0.f;
  const float* rb = rbf + (size_t)b * g.N * C;

  // Binned path: this brick's list, sorted into index order in LDS, then
  // evaluated in chunks.  A brick whose count passed its slots scans instead.
  int n_list = -1;
  if (binned) {
    const size_t k = (size_t)b * gridDim.x + blockIdx.x;
    const int cnt = bins.count[k];
    if (cnt <= bins.cap) n_list = cnt;
    if (n_list >= 0) {
      const int* src = bins.list + k * bins.cap;
      for (int e = tid; e < n_list; e += blockDim.x) fill[e] = src[e];
      __syncthreads();
      // Rank sort (the indices are distinct): an entry's place is the number
      // of smaller entries; every lane reads fill[j] in step (broadcast).
      for (int e = tid; e < n_list; e += blockDim.x) {
        const int v = fill[e];
        int rank = 0;
        for (int j = 0; j < n_list; ++j) rank += fill[j] < v ? 1 : 0;
        keep[rank] = v;
      }
    }
  }
  if (n_list >= 0) {
    // The wave's quarter box (empty past the grid's edge): an RBF that fails
    // the brick test on it reaches none of the wave's voxels, so skipping it
    // leaves every voxel's sum, taken in index order, unchanged.
    const int qx1 = min(qx0 + 3, g.W - 1), qy1 = min(qy0 + 3, g.H - 1);
    const int qz0 = bz * kBZ, qz1 = min(qz0 + kBZ, g.D) - 1;
    const bool qnonempty = qx0 <= qx1 && qy0 <= qy1 && qz0 <= qz1;
    float qlox = 0.f, qhix = 0.f, qloy = 0.f, qhiy = 0.f, qloz = 0.f, qhiz = 0.f;
    if (qnonempty)
      voxel_box(g, qx0, qx1, qy0, qy1, qz0, qz1, &qlox, &qhix, &qloy, &qhiy, &qloz, &qhiz);
    for (int c0 = 0; c0 < n_list; c0 += kChunk) {
      const int nc = min(kChunk, n_list - c0);
      __syncthreads();
      for (int e = tid; e < nc * C; e += blockDim.x) {
        const int r = e / C;
        prm[e] = rb[(size_t)keep[c0 + r] * C + (e - r * C)];
      }
      for (int e = tid; e < nc; e += blockDim.x) pk[e] = gauss_k(rb[(size_t)keep[c0 + e] * C + 3]);
      __syncthreads();
      for (int k0 = 0; k0 < nc; k0 += 64) {
        const int kk = k0 + lane;
        bool pass = false;
        if (qnonempty && kk < nc) {
          const float* p = prm + kk * C;
          pass = brick_may_hold(p[0], p[1], p[2], p[3], g.trunc, qlox, qhix, qloy, qhiy, qloz,
                                qhiz);
        }
        unsigned long long m = __ballot(pass);
        while (m) {  // the wave's RBFs of this group, in index order
          const int k = k0 + __builtin_ctzll(m);
          m &= m - 1;
          const float* p = prm + k * C;
          const float r2 = rbf_r2(x, y, z, p[0], p[1], p[2]);
          if (!within(r2, p[3], g.trunc)) continue;
          const float wgt = gauss_exp2(r2, pk[k]);           // :77
#pragma unroll
          for (int a = 0; a < kMaxAttr; ++a)
            if (a < g.A) attr[a] += wgt * p[4 + a];          // :78-80
          sum += wgt;                                        // :81
        }
      }
    }
  }

  for (int c0 = 0; n_list < 0 && c0 < g.N; c0 += kChunk) {
    const int nc = min(kChunk, g.N - c0);
    __syncthreads();
    for (int e = tid; e < nc * C; e += blockDim.x) prm[e] = rb[(size_t)c0 * C + e];
    for (int e = tid; e < nc; e += blockDim.x) pk[e] = gauss_k(rb[(size_t)(c0 + e) * C + 3]);
    __syncthreads();
    // Cull the chunk against the brick (conservative: squared distance from
    // the centre to the box, against the truncation radius plus a margin).
    bool pass = false;
    if (tid < nc)
      pass = brick_may_hold(prm[tid * C], prm[tid * C + 1], prm[tid * C + 2], prm[tid * C + 3],
                            g.trunc, lox, hix, loy, hiy, loz, hiz);
    const unsigned long long m = __ballot(pass);
    if (lane == 0) wave_cnt[wave] = __popcll(m);
    __syncthreads();
    int base = 0;
    for (int k = 0; k < wave; ++k) base += wave_cnt[k];
    const int nkeep = wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
    if (pass) keep[base + __popcll(m & ((1ull << lane) - 1ull))] = tid;
    __syncthreads();
    for (int k = 0; k < nkeep; ++k) {
      const float* p = prm + keep[k] * C;
      const float r2 = rbf_r2(x, y, z, p[0], p[1], p[2]);
      if (!within(r2, p[3], g.trunc)) continue;
      const float wgt = gauss_exp2(r2, pk[keep[k]]);         // :77
#pragma unroll
      for (int a = 0; a < kMaxAttr; ++a)
        if (a < g.A) attr[a] += wgt * p[4 + a];              // :78-80
      sum += wgt;                                            // :81
    }
  }
  if (!ok) return;
  const size_t V = (size_t)g.D * g.H * g.W;
  const size_t vi = ((size_t)zi * g.H + yi) * g.W + xi;
  float* ob = vol + (size_t)b * (1 + g.A) * V;
  ob[vi] = sum;                                              // :83
  const float den = sum < 1.e-8f ? 1.f : sum;                // :85-87
#pragma unroll
  for (int a = 0; a < kMaxAttr; ++a)
    if (a < g.A) ob[(size_t)(1 + a) * V + vi] = attr[a] / den;  // :89-91
}

// Index range of grid samples within [c - r, c + r] along one axis (widened
// by one sample; the exact test is done per voxel).
__device__ __forceinline__ void axis_range(float c, float r, int n, float a, float b,
                                           int* lo, int* hi) {
  if (n == 1 || !(r < INFINITY)) {
    *lo = 0;
    *hi = n - 1;
    return;
  }
  const float step = (b - a) / (float)(n - 1);
  float u0 = (c - r - a) / step, u1 = (c + r - a) / step;
  if (u0 > u1) {
    const float t = u0;
    u0 = u1;
    u1 = t;
  }
  u0 = fminf(fmaxf(u0 - 1.f, -1.f), (float)n);
  u1 = fminf(fmaxf(u1 + 1.f, -1.f), (float)n);
  *lo = max((int)floorf(u0), 0);
  *hi = min((int)ceilf(u1), n - 1);
}

// Waves (RBFs) per workgroup of the truncated gradient.  Support boxes
// differ by up to ~70x in voxels, and a workgroup holds its slot until its
// slowest wave ends, so each RBF gets a workgroup of its own (0.28 ms at
// 20,000 RBFs -> 128^3, against 0.32 ms with two and 0.37 ms with four).
constexpr int kS2Waves = 1;

__global__ __launch_bounds__(kS2Waves * 64) void splat_grad_kernel(
    const float* __restrict__ rbf, const float* __restrict__ vol,
    const float* __restrict__ vgrad, float* __restrict__ rbf_grad, SplatGeom g) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i = blockIdx.x * kS2Waves + wave;
  const int b = blockIdx.y;
  if (i >= g.N) return;
  const int C = 4 + g.A;
  const float* p = rbf + ((size_t)b * g.N + i) * C;
  const float xr = p[0], yr = p[1], zr = p[2], sg = p[3];
  float av[kMaxAttr];
#pragma unroll
  for (int a = 0; a < kMaxAttr; ++a) av[a] = a < g.A ? p[4 + a] : 0.f;
  const float rad = g.trunc * fabsf(sg) * 1.0001f + 1e-6f;
  int xa, xb, ya, yb, za, zb;
  axis_range(xr, rad, g.W, g.sx, g.ex, &xa, &xb);
  axis_range(yr, rad, g.H, g.sy, g.ey, &ya, &yb);
  axis_range(zr, rad, g.D, g.sz, g.ez, &za, &zb);
  const int nx = xb - xa + 1, ny = yb - ya + 1, nz = zb - za + 1;
  const size_t V = (size_t)g.D * g.H * g.W;
  const float* v0b = vol + (size_t)b * (1 + g.A) * V;
  const float* g0b = vgrad + (size_t)b * (1 + g.A) * V;
  float acc[4 + kMaxAttr];
#pragma unroll
  for (int c = 0; c < 4 + kMaxAttr; ++c) acc[c] = 0.f;
  const float si = 1.f / sg;                                   // :38
  const float kg = gauss_k(sg);
  // Voxel coordinates of the support box, one table per axis per wave when
  // each side has at most 64 voxels (written and read by the same wave).
  __shared__ float ctab[kS2Waves][3][64];
  const bool tabbed = nx <= 64 && ny <= 64 && nz <= 64;
  if (tabbed) {
    ctab[wave][0][lane] = splat_coord(xa + min(lane, nx - 1), g.W, g.sx, g.ex);
    ctab[wave][1][lane] = splat_coord(ya + min(lane, ny - 1), g.H, g.sy, g.ey);
    ctab[wave][2][lane] = splat_coord(za + min(lane, nz - 1), g.D, g.sz, g.ez);
  }
  if (nx > 0 && ny > 0 && nz > 0) {
    const int total = nx * ny * nz;
    // lane offsets (xo, yo, zo) of entry e = xo + nx (yo + ny zo), advanced
    // by 64 entries per step as a mixed-radix addition
    int xo = lane % nx, yo = (lane / nx) % ny, zo = lane / (nx * ny);
    const int r1 = 64 % nx, q1 = 64 / nx, r2 = q1 % ny, q2 = q1 / ny;
    for (int e = lane; e < total; e += 64) {
      const int xi = xa + xo, yi = ya + yo, zi = za + zo;
      const float x = tabbed ? ctab[wave][0][xo] : splat_coord(xi, g.W, g.sx, g.ex);
      const float y = tabbed ? ctab[wave][1][yo] : splat_coord(yi, g.H, g.sy, g.ey);
      const float z = tabbed ? ctab[wave][2][zo] : splat_coord(zi, g.D, g.sz, g.ez);
      const float r2v = rbf_r2(x, y, z, xr, yr, zr);
      if (within(r2v, sg, g.trunc)) {
        const float wgt = gauss_exp2(r2v, kg);                 // :150
        const size_t vi = ((size_t)zi * g.H + yi) * g.W + xi;
        const float dl0 = g0b[vi];                             // :151
        const float dxr = (((x - xr) * si) * si) * wgt;        // :39-41
        const float dyr = (((y - yr) * si) * si) * wgt;
        const float dzr = (((z - zr) * si) * si) * wgt;
        const float dsr = (((r2v * si) * si) * si) * wgt;      // :42-46
        if (g.A == 0) {                                        // :159-163
          acc[0] += dl0 * dxr;
          acc[1] += dl0 * dyr;
          acc[2] += dl0 * dzr;
          acc[3] += dl0 * dsr;
        } else {
          float v0 = v0b[vi];                                  // :165
          if (v0 < 1.e-8f) v0 = 1.f;                           // :167-169
          const float inv = 1.f / v0;                          // :170
          float sum = 0.f;
#pragma unroll
          for (int a = 0; a < kMaxAttr; ++a) {
            if (a < g.A) {
              const float at = v0b[(size_t)(1 + a) * V + vi];
              const float dla = g0b[(size_t)(1 + a) * V + vi];
              sum += dla * (av[a] - at);                       // :176
              acc[4 + a] += (dla * wgt) * inv;                 // :178
            }
          }
          sum = sum * inv;                                     // :180
          acc[0] += dxr * (dl0 + sum);                         // :181-184
          acc[1] += dyr * (dl0 + sum);
          acc[2] += dzr * (dl0 + sum);
          acc[3] += dsr * (dl0 + sum);
        }
      }
      xo += r1;
      const int c1 = xo >= nx ? 1 : 0;
      xo -= c1 * nx;
      yo += r2 + c1;
      const int c2 = yo >= ny ? 1 : 0;
      yo -= c2 * ny;
      zo += q2 + c2;
    }
  }
  float* out = rbf_grad + ((size_t)b * g.N + i) * C;
#pragma unroll
  for (int c = 0; c < 4 + kMaxAttr; ++c) {
    if (c < C) {
      const float s = wave_sum_f32(acc[c]);
      if (lane == 0) out[c] = s;
    }
  }
}

// ---------------------------------------------------------------------------
// Untruncated splats (the reference's default) as matrix products
// ---------------------------------------------------------------------------
//
// g_i(z, y, x) = exp2(k dz^2) * exp2(k (dx^2 + dy^2)), so with the (y, x)
// columns flattened
//   V0[z][col]         = sum_i Ez[z][i] * Exy[i][col]
//   (V0 Va)[z][col]    = sum_i Ez[z][i] * (Exy[i][col] a_i)
// is a matrix product over the RBFs: per (voxel, RBF) pair and channel one
// multiply-add on the FP32 matrix cores, where the direct form spends about
// ten vector instructions.  Both factors are formed in registers as the
// product's operands (an exponential serves MT or NT tiles), so nothing but
// the RBFs is read and only the volume is written.
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma_16x16x4(float a, float b, f32x4 c) {
  // D[row][col] += sum_k A[row][k] B[k][col]; lane l holds A[l % 16][l / 16],
  // B[l / 16][l % 16] and D[4 (l / 16) + 0..3][l % 16]
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

constexpr int kSepWaves = 8;    // waves per workgroup; they share an output tile
constexpr int kSepChunk = 32;   // RBFs a wave stages at once
constexpr int kSepCols = 32;    // columns per tile: two 16-column products
constexpr int kSepNT = kSepCols / 16;
constexpr int kSepAttr = 3;     // attribute channels per workgroup, at most

// exp2(r2 k) of an RBF whose sigma^2 underflows (k = -inf) is NaN on its
// centre and 0 elsewhere, which no product of axis factors reproduces: such
// RBFs take no part in the product and are added afterwards.
__device__ __forceinline__ bool sep_degenerate(float k) { return k == -INFINITY; }

// One workgroup: 16 MT z rows x 32 columns, C channels (the sum and C - 1
// attributes from a0), over the RBF chunks of its split.  Its eight waves
// take every eighth chunk and add their tiles through LDS in wave order.
// part == nullptr: writes the volume; else raw sums [split][B][1 + A][V].
// Bound by the matrix cores: 20,000 RBFs -> 128^3 with one attribute take
// 1.6 ms (106 TFLOP/s of matrix products; the card's library FP32 product
// reaches 154), where the direct form took 16.1 ms; 2,000 -> 64 x 80 x 96
// 0.050 ms (0.52).
template <int C, int MT>
__global__ __launch_bounds__(kSepWaves * 64) void splat_sep_kernel(
    const float* __restrict__ rbf, float* __restrict__ vol, float* __restrict__ part,
    SplatGeom g, int n_split, unsigned first) {
  constexpr int P = MT * kSepNT;  // 16 x 16 tiles of a workgroup
  // staged RBFs during the walk, partial tiles after it
  constexpr int kStage = kSepWaves * kSepChunk * (4 + C - 1) * (int)sizeof(float);
  constexpr int kRed = P * kSepWaves * 64 * (int)sizeof(f32x4);
  __shared__ __align__(16) char lds[kStage > kRed ? kStage : kRed];
  const int lane = threadIdx.x & 63, wave = uniform_i32(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int HW = g.H * g.W;
  const int n_col = (HW + kSepCols - 1) / kSepCols, n_z = (g.D + 16 * MT - 1) / (16 * MT);
  const unsigned block = first + blockIdx.x;
  const int tile = block / n_col;
  const int col0 = (block - tile * n_col) * kSepCols;
  const int z0 = (tile % n_z) * (16 * MT);
  const int a0 = (tile / n_z) * kSepAttr;
  const int b = blockIdx.y, split = blockIdx.z;
  const int RC = 4 + g.A;
  const float* rb = rbf + (size_t)b * g.N * RC;

  float x[kSepNT], y[kSepNT], z[MT];
#pragma unroll
  for (int n = 0; n < kSepNT; ++n) {
    const int col = min(col0 + 16 * n + r, HW - 1);
    x[n] = splat_coord(col % g.W, g.W, g.sx, g.ex);
    y[n] = splat_coord(col / g.W, g.H, g.sy, g.ey);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) z[m] = splat_coord(min(z0 + 16 * m + r, g.D - 1), g.D, g.sz, g.ez);

  f32x4 acc[MT][kSepNT][C];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < kSepNT; ++n)
#pragma unroll
      for (int c = 0; c < C; ++c) acc[m][n][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  float4* prm = (float4*)lds + wave * kSepChunk;                     // {x, y, z, k}
  float* att = (float*)((float4*)lds + kSepWaves * kSepChunk) + wave * kSepChunk * (C - 1);
  const int n_chunk = (g.N + kSepChunk - 1) / kSepChunk;
  int degenerate = 0;
  for (int ch = split * kSepWaves + wave; ch < n_chunk; ch += kSepWaves * n_split) {
    if (lane < kSepChunk) {
      const int i = ch * kSepChunk + lane;
      // past the end: infinitely far away
      float4 v = make_float4(INFINITY, 0.f, 0.f, -1.f);
      float a[C > 1 ? C - 1 : 1];
#pragma unroll
      for (int c = 0; c < C - 1; ++c) a[c] = 0.f;
      if (i < g.N) {
        const float* p = rb + (size_t)i * RC;
        const float k = gauss_k(p[3]);
        if (sep_degenerate(k)) {
          degenerate = 1;
        } else {
          v = make_float4(p[0], p[1], p[2], k);
#pragma unroll
          for (int c = 0; c < C - 1; ++c) a[c] = a0 + c < g.A ? p[4 + a0 + c] : 0.f;
        }
      }
      prm[lane] = v;
#pragma unroll
      for (int c = 0; c < C - 1; ++c) att[c * kSepChunk + lane] = a[c];
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int j = 0; j < kSepChunk / 4; ++j) {  // four RBFs a product
      const float4 p = prm[4 * j + q];
      float at[C > 1 ? C - 1 : 1];
#pragma unroll
      for (int c = 0; c < C - 1; ++c) at[c] = att[c * kSepChunk + 4 * j + q];
      float ez[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float dz = z[m] - p.z;
        ez[m] = gauss_exp2(dz * dz, p.w);
      }
#pragma unroll
      for (int n = 0; n < kSepNT; ++n) {
        const float dx = x[n] - p.x, dy = y[n] - p.y;
        const float e = gauss_exp2(fmaf(dx, dx, dy * dy), p.w);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const float ec = c == 0 ? e : e * at[c - 1];
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[m][n][c] = mfma_16x16x4(ez[m], ec, acc[m][n][c]);
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }

  const int any_degenerate = __syncthreads_or(degenerate);
  // Tile p of the workgroup goes to wave p, which adds the waves' parts (of
  // those that had RBFs).
  f32x4* red = (f32x4*)lds;  // [P][kSepWaves][64]
  const int busy = min(max(n_chunk - split * kSepWaves, 0), kSepWaves);
  f32x4 sum[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if (c > 0) __syncthreads();
    if (wave < busy) {
#pragma unroll
      for (int p = 0; p < P; ++p)
        red[(p * kSepWaves + wave) * 64 + lane] = acc[p / kSepNT][p % kSepNT][c];
    }
    __syncthreads();
    sum[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (wave < P)
      for (int w = 0; w < busy; ++w) sum[c] += red[(wave * kSepWaves + w) * 64 + lane];
  }
  if (wave >= P) return;
  const int col = col0 + 16 * (wave % kSepNT) + r;
  const int zr = z0 + 16 * (wave / kSepNT) + 4 * q;
  if (col >= HW) return;
  if (any_degenerate) {  // of this split's RBFs
    const float xc = splat_coord(col % g.W, g.W, g.sx, g.ex);
    const float yc = splat_coord(col / g.W, g.H, g.sy, g.ey);
    constexpr int G = kSepWaves * kSepChunk;
    for (int64_t i0 = (int64_t)split * G; i0 < g.N; i0 += (int64_t)n_split * G) {
      const int end = (int)(i0 + G < g.N ? i0 + G : g.N);
      for (int i = (int)i0; i < end; ++i) {
        const float* p = rb + (size_t)i * RC;
        const float k = gauss_k(p[3]);
        if (!sep_degenerate(k)) continue;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float zc = splat_coord(min(zr + u, g.D - 1), g.D, g.sz, g.ez);
          const float w = gauss_exp2(rbf_r2(xc, yc, zc, p[0], p[1], p[2]), k);
          sum[0][u] += w;
#pragma unroll
          for (int c = 1; c < C; ++c)
            if (a0 + c - 1 < g.A) sum[c][u] += w * p[4 + a0 + c - 1];
        }
      }
    }
  }
  const size_t V = (size_t)g.D * HW;
  float* ob = (part ? part + (size_t)split * g.B * (1 + g.A) * V : vol) + (size_t)b * (1 + g.A) * V;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    if (zr + u >= g.D) break;
    const size_t vi = (size_t)(zr + u) * HW + col;
    const float s0 = sum[0][u];
    if (a0 == 0) ob[vi] = s0;                                  // :83
    const float den = part || s0 < 1.e-8f ? 1.f : s0;          // :85-87
#pragma unroll
    for (int c = 1; c < C; ++c)
      if (a0 + c - 1 < g.A) ob[(size_t)(a0 + c) * V + vi] = sum[c][u] / den;  // :89-91
  }
}

// The splits' raw sums, added in split order and normalised.
__global__ void splat_sep_finish_kernel(const float* __restrict__ part, int n_split,
                                        float* __restrict__ vol, int B, int A, size_t V) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < (size_t)B * V;
       e += (size_t)gridDim.x * blockDim.x) {
    const size_t b = e / V, v = e - b * V;
    const size_t at = b * (1 + A) * V + v, step = (size_t)B * (1 + A) * V;
    float den = 1.f;
    for (int c = 0; c <= A; ++c) {
      float s = 0.f;
      for (int k = 0; k < n_split; ++k) s += part[(size_t)k * step + at + (size_t)c * V];
      vol[at + (size_t)c * V] = s / den;
      if (c == 0) den = s < 1.e-8f ? 1.f : s;
    }
  }
}

// S2 without truncation.  With F0 = dL/dV0 - sum_a dL/dVa Va / V0 and
// Fa = dL/dVa / V0 (V0 guarded as in the forward), an RBF's gradient is a set
// of moments of F = F0 + sum_a a_{i,a} Fa under its Gaussian: of 1, dx, dy,
// dz and r^2, and of 1 under each Fa.  The sum over x of a (z, y) row,
//   P_j[row][i] = sum_x F[row][x] * (exp2(k dx^2) dx^j),  j = 0, 1, 2
// is a matrix product, and holds nearly all of the work: each of its entries
// stands for W (voxel, RBF) pairs.  The rest, exp2(k (dy^2 + dz^2)) and its
// moments, is done once per (row, RBF) on the product's output registers,
// where a lane holds one RBF (column) and four rows.
//
// One workgroup: 32 RBFs, the row tiles (16 rows, or a chunk of x of them) of
// its segment, dealt over its four waves.  The attribute channels come in pairs, one walk over the
// rows per pair (more accumulators would halve the waves in flight).
// 20,000 RBFs -> 128^3 with one attribute take 6.1 ms (83 TFLOP/s of matrix
// products; forming F and the Gaussians takes most of the rest), where the
// direct form (a voxel tile in LDS, every RBF against every voxel) took
// 34.8 ms; 2,000 -> 64 x 80 x 96 0.17 ms (2.19).
constexpr int kGradWaves = 4;
constexpr int kGradRbf = 32;  // RBFs per workgroup: two 16-column products
constexpr int kGradNT = kGradRbf / 16;
constexpr int kGradCoord = 4096;  // coordinates kept in LDS, at most

// AT: the attribute count when known at compile time (0 or 1), or -1.
template <int NC, int AT>
__global__ __launch_bounds__(kGradWaves * 64, AT < 0 ? 3 : 4) void splat_grad_sep_kernel(
    const float* __restrict__ rbf, const float* __restrict__ vol,
    const float* __restrict__ vgrad, float* __restrict__ out, SplatGeom g, int n_seg, int n_xc,
    int xw) {
  __shared__ float coord[kGradCoord + 16];
  __shared__ float red[kGradWaves][kGradRbf][4 + kMaxAttr];
  __shared__ float common[kMaxAttr];
  const int lane = threadIdx.x & 63, wave = uniform_i32(threadIdx.x >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int i0 = blockIdx.x * kGradRbf, seg = blockIdx.y, b = blockIdx.z;
  const int A = AT >= 0 ? AT : g.A, RC = 4 + A, W = g.W;
  const int n_rows = g.D * g.H, n_units = (n_rows + 15) / 16 * n_xc;
  const size_t V = (size_t)n_rows * W;
  const float* v0b = vol + (size_t)b * (1 + A) * V;
  const float* g0b = vgrad + (size_t)b * (1 + A) * V;

  // coordinate tables [D][H][W, to 16]: usual grids fit
  const bool tabled = (size_t)g.D + g.H + W <= kGradCoord;
  const float* cz = coord;
  const float* cy = coord + g.D;
  const float* cx = coord + g.D + g.H;
  if (tabled) {
    for (int e = threadIdx.x; e < g.D; e += blockDim.x) coord[e] = splat_coord(e, g.D, g.sz, g.ez);
    for (int e = threadIdx.x; e < g.H; e += blockDim.x)
      coord[g.D + e] = splat_coord(e, g.H, g.sy, g.ey);
    for (int e = threadIdx.x; e < ((W + 15) & ~15); e += blockDim.x)
      coord[g.D + g.H + e] = splat_coord(min(e, W - 1), W, g.sx, g.ex);
  }
  // A common attribute value c taken out of both terms of F0 + a Fa, which
  // nearly cancel where one RBF stands alone (Va = a there): the mean of the
  // workgroup's RBFs, no larger than 64 times the smallest magnitude among them.
  // What is left of an RBF's own terms, a - c, is then bounded by its own a,
  // whatever its neighbours in the list hold (the plain mean of one attribute of
  // 1e7 and 31 of about 1 cost those 31 six digits); a tighter bound costs
  // attributes in [0, 1) accuracy (twice the smallest: errors of 24 sizes 2 % up).
  if ((int)threadIdx.x < A) {
    float m = 0.f, least = INFINITY;
    for (int n = 0; n < kGradRbf; ++n) {
      const float a = rbf[((size_t)b * g.N + min(i0 + n, g.N - 1)) * RC + 4 + threadIdx.x];
      m += a;
      least = fminf(least, fabsf(a));
    }
    m *= 1.f / kGradRbf;
    common[threadIdx.x] = fabsf(m) < INFINITY ? fminf(fmaxf(m, -64.f * least), 64.f * least) : 0.f;
  }
  __syncthreads();

  // this lane's RBFs (past N: sigma 1, not written)
  float xr[kGradNT], yr[kGradNT], zr[kGradNT], kg[kGradNT];
  float mx[kGradNT], my[kGradNT], mz[kGradNT], mr[kGradNT];
#pragma unroll
  for (int n = 0; n < kGradNT; ++n) {
    const int i = i0 + 16 * n + r;
    const float* p = rbf + ((size_t)b * g.N + min(i, g.N - 1)) * RC;
    xr[n] = p[0];
    yr[n] = p[1];
    zr[n] = p[2];
    kg[n] = gauss_k(i < g.N ? p[3] : 1.f);
    mx[n] = my[n] = mz[n] = mr[n] = 0.f;
  }
  for (int c0 = 0; c0 <= A; c0 += NC) {  // channels c0 .. c0 + NC - 1 (0: F0)
    float av[kGradNT][NC], ms[kGradNT][NC];
#pragma unroll
    for (int n = 0; n < kGradNT; ++n)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int i = min(i0 + 16 * n + r, g.N - 1);
        av[n][c] = c0 + c == 0 ? 1.f : 0.f;
        if (c0 + c >= 1 && c0 + c <= A)
          av[n][c] = rbf[((size_t)b * g.N + i) * RC + 3 + c0 + c] - common[c0 + c - 1];
        ms[n][c] = 0.f;
      }
    for (int unit = seg * kGradWaves + wave; unit < n_units; unit += kGradWaves * n_seg) {
      const int t = unit / n_xc, xb = (unit - t * n_xc) * xw, xe = min(xb + xw, W);
      f32x4 acc[kGradNT][NC][3];
#pragma unroll
      for (int n = 0; n < kGradNT; ++n)
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int j = 0; j < 3; ++j) acc[n][c][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      const int row = t * 16 + r;
      const size_t at = (size_t)min(row, n_rows - 1) * W;
      // One step of 16 x.  Whole steps load without branches, so that their
      // loads are in flight together (a branch per load: 2.5 times the time);
      // rows past the last read it again and count as zero.
      auto step = [&](int x0, auto whole) {
        const int xa = x0 + 4 * q;
        auto load4 = [&](const float* src, float* v) {
          if constexpr (whole) {
            __builtin_memcpy(v, src + at + xa, 16);
          } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = src[at + min(xa + u, W - 1)];
          }
        };
        float F[NC][4], inv[4], xs[4];
#pragma unroll
        for (int c = 0; c < NC; ++c) load4(g0b + (size_t)min(c0 + c, A) * V, F[c]);
        if (A > 0) {
          load4(v0b, inv);
#pragma unroll
          for (int u = 0; u < 4; ++u) inv[u] = 1.f / (inv[u] < 1.e-8f ? 1.f : inv[u]);  // :167-170
        }
        if (A > 0 && c0 == 0) {
#pragma unroll 1
          for (int a = 1; a <= A; ++a) {
            float dla[4], va[4];
            if (AT == 1) {
#pragma unroll
              for (int u = 0; u < 4; ++u) dla[u] = F[NC - 1][u];
            } else {
              load4(g0b + (size_t)a * V, dla);
            }
            load4(v0b + (size_t)a * V, va);
#pragma unroll
            for (int u = 0; u < 4; ++u)  // by the rounded Fa, which the products take too
              F[0][u] = fmaf(-(dla[u] * inv[u]), va[u] - common[a - 1], F[0][u]);
          }
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (c0 + c > 0) F[c][u] *= inv[u];
            if (row >= n_rows || c0 + c > A || (!whole && xa + u >= W)) F[c][u] = 0.f;
          }
        if (tabled) {
#pragma unroll
          for (int u = 0; u < 4; ++u) xs[u] = cx[xa + u];
        } else {
#pragma unroll
          for (int u = 0; u < 4; ++u) xs[u] = splat_coord(min(xa + u, W - 1), W, g.sx, g.ex);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
          for (int n = 0; n < kGradNT; ++n) {
            const float dx = xs[u] - xr[n];
            float e0 = gauss_exp2(dx * dx, kg[n]);
            if (sep_degenerate(kg[n])) e0 = 0.f;
            const float e1 = dx * e0, e2 = dx * e1;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              acc[n][c][0] = mfma_16x16x4(F[c][u], e0, acc[n][c][0]);
              acc[n][c][1] = mfma_16x16x4(F[c][u], e1, acc[n][c][1]);
              acc[n][c][2] = mfma_16x16x4(F[c][u], e2, acc[n][c][2]);
            }
          }
        }
      };
      int x0 = xb;
      for (; x0 + 16 <= xe; x0 += 16) step(x0, std::true_type{});
      if (x0 < xe) step(x0, std::false_type{});
      // rows 4 q .. 4 q + 3 of the tile, one RBF per lane and product
      const int first = min(t * 16 + 4 * q, n_rows - 1);
      int zi = first / g.H, yi = first - zi * g.H;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float yc = tabled ? cy[yi] : splat_coord(yi, g.H, g.sy, g.ey);
        const float zc = tabled ? cz[zi] : splat_coord(zi, g.D, g.sz, g.ez);
#pragma unroll
        for (int n = 0; n < kGradNT; ++n) {
          const float dy = yc - yr[n], dz = zc - zr[n];
          const float r2 = fmaf(dy, dy, dz * dz);
          float e = gauss_exp2(r2, kg[n]);
          if (sep_degenerate(kg[n])) e = 0.f;
          float p0 = 0.f, p1 = 0.f, p2 = 0.f;
#pragma unroll
          for (int c = 0; c < NC; ++c) {
            const float s = acc[n][c][0][u] * e;
            ms[n][c] += s;
            p0 = fmaf(av[n][c], s, p0);
            p1 = fmaf(av[n][c], acc[n][c][1][u], p1);
            p2 = fmaf(av[n][c], acc[n][c][2][u], p2);
          }
          mx[n] = fmaf(p1, e, mx[n]);
          my[n] = fmaf(p0, dy, my[n]);
          mz[n] = fmaf(p0, dz, mz[n]);
          mr[n] += fmaf(p2, e, p0 * r2);
        }
        if (t * 16 + 4 * q + u + 1 < n_rows && ++yi == g.H) {
          yi = 0;
          ++zi;
        }
      }
    }
    // attribute sums of this pair of channels, over the wave's row groups
#pragma unroll
    for (int n = 0; n < kGradNT; ++n)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        float s = ms[n][c];
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        if (q == 0 && c0 + c >= 1 && c0 + c <= A) red[wave][16 * n + r][3 + c0 + c] = s;
      }
  }
#pragma unroll
  for (int n = 0; n < kGradNT; ++n) {
    float m[4] = {mx[n], my[n], mz[n], mr[n]};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      m[c] += __shfl_xor(m[c], 16, 64);
      m[c] += __shfl_xor(m[c], 32, 64);
      if (q == 0) red[wave][16 * n + r][c] = m[c];
    }
  }
  __syncthreads();
  float* ob = out + ((size_t)seg * g.B + b) * g.N * RC;
  for (int e = threadIdx.x; e < kGradRbf * RC; e += blockDim.x) {
    const int n = e / RC, c = e - n * RC;
    if (i0 + n >= g.N) continue;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kGradWaves; ++w) s += red[w][n][c];
    const float si = 1.f / rbf[((size_t)b * g.N + i0 + n) * RC + 3];       // :38
    if (c < 3) s = (s * si) * si;                                          // :39-41
    if (c == 3) s = ((s * si) * si) * si;                                  // :42-46
    ob[(size_t)(i0 + n) * RC + c] = s;
  }
}

// out[e] = sum over segments: sixteen lanes take every sixteenth segment and
// add up pairwise, in a fixed order.  (One lane per element took 29 us for
// 768 segments of 300 elements.)
__global__ __launch_bounds__(256) void splat_sum_segments_kernel(const float* __restrict__ part,
                                                                 int n_seg,
                                                                 float* __restrict__ out,
                                                                 size_t n) {
  const int k0 = threadIdx.x >> 4;
  const size_t e = (size_t)blockIdx.x * 16 + (threadIdx.x & 15);
  __shared__ float red[16][16];
  float s = 0.f;
  if (e < n)
    for (int k = k0; k < n_seg; k += 16) s += part[(size_t)k * n + e];
  red[k0][threadIdx.x & 15] = s;
  __syncthreads();
  for (int m = 8; m >= 1; m >>= 1) {
    if (k0 < m) red[k0][threadIdx.x & 15] += red[k0 + m][threadIdx.x & 15];
    __syncthreads();
  }
  if (k0 == 0 && e < n) out[e] = red[0][threadIdx.x & 15];
}

__global__ void fill_zero_i32_kernel(int* __restrict__ p, size_t n) {
  for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < n;
       e += (size_t)gridDim.x * blockDim.x)
    p[e] = 0;
}

SplatGeom splat_geom(int64_t B, int64_t N, int64_t A, int64_t D, int64_t H, int64_t W,
                     const float* vs, const float* ve, float trunc) {
  SplatGeom g;
  g.B = (int)B;
  g.N = (int)N;
  g.A = (int)A;
  g.D = (int)D;
  g.H = (int)H;
  g.W = (int)W;
  g.sx = vs[0];
  g.sy = vs[1];
  g.sz = vs[2];
  g.ex = ve[0];
  g.ey = ve[1];
  g.ez = ve[2];
  g.trunc = trunc;
  return g;
}

int check_splat(int64_t B, int64_t N, int64_t A, int64_t D, int64_t H, int64_t W,
                const float* vs, const float* ve) {
  for (int64_t d : {B, N, D, H, W})
    TOTRI_CHECK_ARG(d >= 0 && d < (1ll << 31), "dimension out of range");
  TOTRI_CHECK_ARG(A >= 0 && A <= kMaxAttr, "attributes per RBF must be in [0, %d], got %lld",
                  kMaxAttr, (long long)A);
  TOTRI_CHECK_ARG(B * (1 + A) * D * H * W < (1ll << 31) && B * N * (4 + A) < (1ll << 31),
                  "tensor has more than 2^31 elements");
  TOTRI_CHECK_ARG(vs && ve, "null volume box");
  return TOTRI_OK;
}

}  // namespace
}  // namespace totri_hip

using namespace totri_hip;

namespace totri_hip {
namespace {

struct BinLayout {
  size_t nb;     // bricks per batch entry
  size_t count;  // byte offset of the [B][nb] counts
  size_t list;   // byte offset of the [B][nb][cap] lists
  int cap;       // list slots per brick
  size_t end;
};

// Workspace of the binned splat (truncated splats only): a count per brick
// and `cap` list slots per brick, kSlotMax at most and fewer for large grids
// (at most 2^24 slots in all, at least kSlotMin per brick).  About 20-60
// RBFs reach a brick at the usual sigma / voxel ratios; a brick reached by
// more than cap scans all RBFs.
BinLayout bin_layout(int64_t B, int64_t D, int64_t H, int64_t W) {
  BinLayout l;
  const size_t bx = (size_t)((W + kBX - 1) / kBX), by = (size_t)((H + kBY - 1) / kBY),
               bz = (size_t)((D + kBZ - 1) / kBZ);
  l.nb = bx * by * bz;
  const size_t bricks = (size_t)B * l.nb;
  size_t cap = ((size_t)1 << 24) / (bricks > 0 ? bricks : 1);
  if (cap > (size_t)kSlotMax) cap = kSlotMax;
  if (cap < (size_t)kSlotMin) cap = kSlotMin;
  l.cap = (int)cap;
  l.count = 0;
  l.list = (bricks * sizeof(int) + 255) & ~(size_t)255;
  l.end = l.list + ((bricks * cap * sizeof(int) + 255) & ~(size_t)255);
  return l;
}

}  // namespace
}  // namespace totri_hip

namespace totri_hip {
namespace {

unsigned blocks_for(size_t n) {
  const size_t b = (n + 255) / 256;
  return (unsigned)(b < 65536 ? (b > 0 ? b : 1) : 65536);
}

struct SepPlan {
  int mt;       // 16-row z tiles per workgroup
  int groups;   // attribute groups
  int split;    // RBF splits (more than one only with room for their sums)
  unsigned grid;  // tiles x groups
  size_t bytes;   // of the splits' sums
};

// The RBFs are split over workgroups only where the tiles of the volume leave
// more than half of the CUs without one; a split costs a write and a read of
// the volume, and each wave keeps at least two chunks of RBFs.
SepPlan sep_plan(int64_t B, int64_t N, int64_t A, int64_t D, int64_t H, int64_t W) {
  SepPlan p;
  const int64_t zt = (D + 15) / 16, nz = (zt + 3) / 4;
  p.mt = (int)((zt + nz - 1) / nz);
  p.groups = A > 0 ? (int)((A + kSepAttr - 1) / kSepAttr) : 1;
  const int64_t gz = (zt + p.mt - 1) / p.mt;
  p.grid = (unsigned)((H * W + kSepCols - 1) / kSepCols * gz * p.groups);
  const int64_t wgs = (int64_t)p.grid * B;
  const int64_t chunks = (N + kSepChunk - 1) / kSepChunk;
  int64_t split = wgs > 0 && wgs * 2 <= 256 ? 256 / wgs : 1;
  if (split > chunks / (2 * kSepWaves)) split = chunks / (2 * kSepWaves);
  if (split < 1) split = 1;
  p.split = (int)split;
  p.bytes = split > 1 ? (size_t)split * B * (1 + A) * D * H * W * sizeof(float) : 0;
  return p;
}

template <int C, int MT>
void launch_sep(const float* rbf, float* vol, float* part, const SplatGeom& g, const SepPlan& p,
                int split, hipStream_t st) {
  // a launch holds less than 2^32 lanes along x: flat volumes take several
  constexpr unsigned most = 1u << 22;
  for (unsigned first = 0; first < p.grid; first += most)
    hipLaunchKernelGGL((splat_sep_kernel<C, MT>),
                       dim3(p.grid - first < most ? p.grid - first : most, (unsigned)g.B,
                            (unsigned)split),
                       dim3(kSepWaves * 64), 0, st, rbf, vol, part, g, split, first);
}

template <int C>
void launch_sep_c(const float* rbf, float* vol, float* part, const SplatGeom& g,
                  const SepPlan& p, int split, hipStream_t st) {
  switch (p.mt) {
    case 1: return launch_sep<C, 1>(rbf, vol, part, g, p, split, st);
    case 2: return launch_sep<C, 2>(rbf, vol, part, g, p, split, st);
    case 3: return launch_sep<C, 3>(rbf, vol, part, g, p, split, st);
    default: return launch_sep<C, 4>(rbf, vol, part, g, p, split, st);
  }
}

int splat_forward_full(const float* rbf, float* vol, const SplatGeom& g, void* ws,
                       size_t ws_bytes, hipStream_t st) {
  const SepPlan p = sep_plan(g.B, g.N, g.A, g.D, g.H, g.W);
  const int split = ws != nullptr && ws_bytes >= p.bytes ? p.split : 1;
  float* part = split > 1 ? (float*)ws : nullptr;
  const int c = 1 + (g.A < kSepAttr ? g.A : kSepAttr);
  if (c == 1) launch_sep_c<1>(rbf, vol, part, g, p, split, st);
  if (c == 2) launch_sep_c<2>(rbf, vol, part, g, p, split, st);
  if (c == 3) launch_sep_c<3>(rbf, vol, part, g, p, split, st);
  if (c == 4) launch_sep_c<4>(rbf, vol, part, g, p, split, st);
  int rc = check_launch("splat_sep_kernel");
  if (rc || split == 1) return rc;
  const size_t V = (size_t)g.D * g.H * g.W;
  hipLaunchKernelGGL(splat_sep_finish_kernel, dim3(blocks_for(g.B * V)), dim3(256), 0, st, part,
                     split, vol, g.B, g.A, V);
  return check_launch("splat_sep_finish_kernel");
}

// The untruncated gradient's work of one workgroup of 32 RBFs: row tiles, each
// in n_xc chunks of xw voxels along x, dealt over seg segments.
struct GradPlan {
  int seg, n_xc, xw;
};

// Enough segments for six workgroups per CU, while each wave keeps at least two
// units; chunks of at least 64 voxels where there are too few rows for that (a
// grid of 2 x 2 rows of 2,048 voxels, 50 RBFs with one attribute: 162 -> 32 us).
// Below 16 steps of 16 rows x 16 x a wave (about 10 us) the second launch costs
// more than the segments give: 50 RBFs on 16^3 took 8 us longer a call with them.
GradPlan grad_plan(int64_t B, int64_t N, int64_t A, int64_t D, int64_t H, int64_t W) {
  const int64_t wgs = B * ((N + kGradRbf - 1) / kGradRbf);
  const int64_t tiles = (D * H + 15) / 16, xs = (W + 15) / 16;
  const int64_t walks = A == 0 ? 1 : (A + 2) / 2;  // channel pairs
  const int64_t target = wgs > 0 ? (6 * 256 + wgs - 1) / wgs : 1;
  int64_t xc = (2 * kGradWaves * target + tiles - 1) / tiles;
  if (xc > xs / 4) xc = xs / 4;
  if (xc < 1) xc = 1;
  GradPlan p;
  p.xw = (int)((xs + xc - 1) / xc * 16);
  p.n_xc = (int)((W + p.xw - 1) / p.xw);
  const int64_t units = tiles * p.n_xc;
  int64_t seg = units / (2 * kGradWaves);
  if (seg > target) seg = target;
  if ((units + kGradWaves - 1) / kGradWaves * (p.xw / 16) * walks < 16) seg = 1;
  p.seg = (int)(seg < 1 ? 1 : seg);
  return p;
}

int splat_grad_full(const float* rbf, const float* vol, const float* vgrad, float* out,
                    const SplatGeom& g, void* ws, size_t ws_bytes, hipStream_t st) {
  const GradPlan p = grad_plan(g.B, g.N, g.A, g.D, g.H, g.W);
  int seg = p.seg;
  const size_t n = (size_t)g.B * g.N * (4 + g.A);
  if (ws == nullptr || ws_bytes < seg * n * sizeof(float)) seg = 1;
  float* dst = seg > 1 ? (float*)ws : out;
  const dim3 grid((unsigned)((g.N + kGradRbf - 1) / kGradRbf), (unsigned)seg, (unsigned)g.B);
  auto kernel = g.A == 0   ? splat_grad_sep_kernel<1, 0>
                : g.A == 1 ? splat_grad_sep_kernel<2, 1>
                           : splat_grad_sep_kernel<2, -1>;
  hipLaunchKernelGGL(kernel, grid, dim3(kGradWaves * 64), 0, st, rbf, vol, vgrad, dst, g, seg,
                     p.n_xc, p.xw);
  int rc = check_launch("splat_grad_sep_kernel");
  if (rc || seg == 1) return rc;
  hipLaunchKernelGGL(splat_sum_segments_kernel, dim3((unsigned)((n + 15) / 16)), dim3(256), 0, st,
                     dst, seg, out, n);
  return check_launch("splat_sum_segments_kernel");
}

}  // namespace
}  // namespace totri_hip

extern "C" size_t totri_rbf2volume_gaussian_forward_workspace(int64_t B, int64_t N, int64_t A,
                                                              int64_t D, int64_t H, int64_t W,
                                                              float truncation) {
  if (B <= 0 || N <= 0 || A < 0 || D <= 0 || H <= 0 || W <= 0) return 0;
  if (!(truncation > 0.f)) return sep_plan(B, N, A, D, H, W).bytes;
  return bin_layout(B, D, H, W).end;
}

extern "C" int totri_rbf2volume_gaussian_forward(const float* rbf, int64_t B, int64_t N,
                                                 int64_t A, float* volume, int64_t D,
                                                 int64_t H, int64_t W,
                                                 const float volume_start[3],
                                                 const float volume_end[3],
                                                 float truncation, void* workspace,
                                                 size_t workspace_bytes, void* stream) {
  int rc = check_splat(B, N, A, D, H, W, volume_start, volume_end);
  if (rc) return rc;
  const size_t V = (size_t)D * H * W;
  if (B == 0 || V == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(volume != nullptr && (N == 0 || rbf != nullptr), "null pointer");
  hipStream_t st = (hipStream_t)stream;
  const SplatGeom g = splat_geom(B, N, A, D, H, W, volume_start, volume_end, truncation);
  if (!(truncation > 0.f))
    return splat_forward_full(rbf, volume, g, workspace, workspace_bytes, st);
  const int bx = (int)((W + kBX - 1) / kBX), by = (int)((H + kBY - 1) / kBY),
            bz = (int)((D + kBZ - 1) / kBZ);
  SplatBins bins;
  memset(&bins, 0, sizeof(bins));
  const size_t need = totri_rbf2volume_gaussian_forward_workspace(B, N, A, D, H, W, truncation);
  const int binned = need > 0 ? 1 : 0;
  if (binned) {
    if (workspace_bytes < need)
      return fail(TOTRI_EWORKSPACE, "workspace too small: need %zu bytes, got %zu", need,
                  workspace_bytes);
    TOTRI_CHECK_ARG(workspace != nullptr, "null workspace");
    const BinLayout l = bin_layout(B, D, H, W);
    char* w = (char*)workspace;
    bins.count = (int*)(w + l.count);
    bins.list = (int*)(w + l.list);
    bins.cap = l.cap;
    const size_t n = (size_t)B * l.nb;
    TOTRI_CHECK_ARG(n < (1u << 31), "too many bricks");
    hipLaunchKernelGGL(fill_zero_i32_kernel, dim3(blocks_for(n)), dim3(256), 0, st, bins.count, n);
    rc = check_launch("fill_zero_i32_kernel");
    if (rc) return rc;
    const dim3 grid((unsigned)((N + kBinWaves - 1) / kBinWaves), (unsigned)B);
    hipLaunchKernelGGL(splat_bin_kernel, grid, dim3(kBinWaves * 64), 0, st, rbf, g, bx, by, bz,
                       bins);
    rc = check_launch("splat_bin_kernel");
    if (rc) return rc;
  }
  hipLaunchKernelGGL(splat_forward_kernel, dim3((unsigned)(bx * by * bz), (unsigned)B),
                     dim3(256), 0, st, rbf, volume, g, bx, by, bins, binned);
  return check_launch("splat_forward_kernel");
}

extern "C" size_t totri_rbf2volume_gaussian_grad_workspace(int64_t B, int64_t N, int64_t A,
                                                           int64_t D, int64_t H, int64_t W,
                                                           float truncation) {
  if (truncation > 0.f || B <= 0 || N <= 0 || A < 0 || D <= 0 || H <= 0 || W <= 0) return 0;
  const int seg = grad_plan(B, N, A, D, H, W).seg;
  return seg > 1 ? (size_t)seg * B * N * (4 + A) * sizeof(float) : 0;
}

extern "C" int totri_rbf2volume_gaussian_grad_split(const float* rbf, int64_t B, int64_t N,
                                                    int64_t A, const float* volume,
                                                    const float* volume_grad, float* rbf_grad,
                                                    int64_t D, int64_t H, int64_t W,
                                                    const float volume_start[3],
                                                    const float volume_end[3],
                                                    float truncation, void* workspace,
                                                    size_t workspace_bytes, void* stream) {
  int rc = check_splat(B, N, A, D, H, W, volume_start, volume_end);
  if (rc) return rc;
  if (B == 0 || N == 0) return TOTRI_OK;
  TOTRI_CHECK_ARG(rbf && volume && volume_grad && rbf_grad, "null pointer");
  const SplatGeom g = splat_geom(B, N, A, D, H, W, volume_start, volume_end, truncation);
  if (!(truncation > 0.f))
    return splat_grad_full(rbf, volume, volume_grad, rbf_grad, g, workspace, workspace_bytes,
                           (hipStream_t)stream);
  hipLaunchKernelGGL(splat_grad_kernel,
                     dim3((unsigned)((N + kS2Waves - 1) / kS2Waves), (unsigned)B),
                     dim3(kS2Waves * 64), 0, (hipStream_t)stream, rbf, volume, volume_grad,
                     rbf_grad, g);
  return check_launch("splat_grad_kernel");
}

extern "C" int totri_rbf2volume_gaussian_grad(const float* rbf, int64_t B, int64_t N,
                                              int64_t A, const float* volume,
                                              const float* volume_grad, float* rbf_grad,
                                              int64_t D, int64_t H, int64_t W,
                                              const float volume_start[3],
                                              const float volume_end[3], float truncation,
                                              void* stream) {
  return totri_rbf2volume_gaussian_grad_split(rbf, B, N, A, volume, volume_grad, rbf_grad, D, H,
                                              W, volume_start, volume_end, truncation, nullptr, 0,
                                              stream);
}
