// AW-towers imaging (examples/notebooks/awtowers.ipynb cells 17, 19, 22):
// w-towers whose (chunk, w-plane) images are built per antenna pair, each
// pre-gridded with the anti-aliasing kernel on a twice-larger sub-grid at
// twice the field of view, transformed, cut to the middle, corrected by the
// anti-aliasing windows and multiplied by the pair's A-screen ratio
// aimage[a2] / aimage[a1] in image space before the pairs are summed.
//
// Work unit: a group = (chunk, w-plane, antenna pair), groups sorted by that
// key.  Three launches per batch of groups plus two per call:
//   k_awt_pregrid  visibilities of the batch onto [G][M][M] (M = 2S) grids
//                  with the separable anti-aliasing kernel (one thread per
//                  visibility and kernel row);
//   (batched inverse FFT of the stack, rocFFT, unscaled: win holds 1 / M^2)
//   k_awt_apply    per chunk and sub-grid pixel: the sum over the chunk's
//                  groups of pixel * ratio * wkern^-wp, times the window;
//   (batched forward FFT of the chunk images, rocFFT)
//   k_awt_place    chunk grids added into the grid, clipped at its edges.
// Groups of few visibilities skip the pre-grids and the inverse FFT: the
// cut-out image of a visibility is the outer product of two S-vectors (the
// transforms of its kernel rows), summed straight into the chunk images
// (k_awt_direct).
// With even S and M = 2S the centring signs of the M-grid's inverse
// transform and of the S-grid's forward transform cancel on the cut-out
// pixels, so k_awt_apply applies none; the pre-grid carries the input sign
// of the inverse transform and k_awt_place the output sign of the forward
// one.
#include <algorithm>
#include <climits>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "internal.h"

namespace {

// One (visibility, kernel row): p = rel / lam_sub, cell and sub-offset by
// synthesis.py's frac_coord on the M grid, row y - K//2 + i of the window
// += gcf[yf][i] * gcf[xf][j] * v (synthesis.py:451-481, separable table).
// With apply == 0 only the checks run (every visibility of the call).
__global__ void k_awt_pregrid(float2 *__restrict__ stack, int M,
                              const double *__restrict__ rel, int64_t v0, int64_t v1,
                              double lam_sub, int Q, int K,
                              const float2 *__restrict__ gcf,
                              const float2 *__restrict__ vis,
                              const int32_t *__restrict__ gid, int32_t g0, int apply,
                              uint32_t *status) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t v = v0 + t / K;
  const int i = (int)(t % K);
  if (v >= v1) return;
  const double px = grid_fraction(rel[v * 3], lam_sub);
  const double py = grid_fraction(rel[v * 3 + 1], lam_sub);
  int x, xf, y, yf;
  if (!frac_coord_dev(M, Q, px, &x, &xf) || !frac_coord_dev(M, Q, py, &y, &yf)) {
    if (i == 0) atomicOr(status, (uint32_t)ST_DOMAIN);
    return;
  }
  const int xs = x - K / 2, ys = y - K / 2;
  if (xs < 0 || ys < 0 || xs + K > M || ys + K > M) {
    if (i == 0) atomicOr(status, (uint32_t)ST_BOUNDS);
    return;
  }
  if (!apply) return;
  const float2 a = vis[v];
  const float2 ky = gcf[(int64_t)yf * K + i];
  // ky * v, then times each column's tap
  float2 r;
  r.x = ky.x * a.x - ky.y * a.y;
  r.y = ky.x * a.y + ky.y * a.x;
  const int row = ys + i;
  float *g = (float *)(stack + ((int64_t)(gid[v] - g0) * M + row) * M + xs);
  for (int j = 0; j < K; ++j) {
    const float2 kx = gcf[(int64_t)xf * K + j];
    float ox = kx.x * r.x - kx.y * r.y;
    float oy = kx.x * r.y + kx.y * r.x;
    if ((row + xs + j) & 1) {
      ox = -ox;
      oy = -oy;
    }
    unsafeAtomicAdd(g + 2 * j, ox);
    unsafeAtomicAdd(g + 2 * j + 1, oy);
  }
}

// bins[c0 + k][y][x] += win[y][x] * sum over groups g in [start[k],
// start[k + 1]) of stack[g][y + S/2][x + S/2] * ascreen[a2[g]] / ascreen[a1[g]]
// * wkern^-wp[g], wkern = 2^lmag exp(2 pi i turns) per pixel; the power's
// phase is reduced to turns in FP64 before the FP32 sincospi.
__global__ void k_awt_apply(float2 *__restrict__ bins, int c0,
                            const float2 *__restrict__ stack, int S,
                            const int32_t *__restrict__ start,
                            const int32_t *__restrict__ gwp,
                            const int32_t *__restrict__ ga1,
                            const int32_t *__restrict__ ga2,
                            const float2 *__restrict__ ascreen,
                            const float *__restrict__ win,
                            const double *__restrict__ turns,
                            const float *__restrict__ lmag) {
  const int SS = S * S;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= SS) return;
  const int k = blockIdx.y;
  const int y = pix / S, x = pix - y * S;
  const int M = 2 * S;
  const int64_t off = (int64_t)(y + S / 2) * M + (x + S / 2);
  const double tw = turns[pix];
  const float lm = lmag[pix];
  double ax = 0.0, ay = 0.0;
  const int gs = start[k], ge = start[k + 1];
  for (int g = gs; g < ge; ++g) {
    const float2 v = stack[(int64_t)g * M * M + off];
    const float2 p = ascreen[(int64_t)ga1[g] * SS + pix];
    const float2 q = ascreen[(int64_t)ga2[g] * SS + pix];
    // q / p = q conj(p) / |p|^2
    const float inv = 1.0f / (p.x * p.x + p.y * p.y);
    const float rx = (q.x * p.x + q.y * p.y) * inv;
    const float ry = (q.y * p.x - q.x * p.y) * inv;
    const int wp = gwp[g];
    const double t = -(double)wp * tw;
    float s, c;
    sincospif((float)(2.0 * (t - rint(t))), &s, &c);
    const float mag = lm == 0.0f ? 1.0f : exp2f(-(float)wp * lm);
    const float fx = c * mag, fy = s * mag;
    // v * r * f
    const float vx = v.x * rx - v.y * ry;
    const float vy = v.x * ry + v.y * rx;
    ax += (double)(vx * fx - vy * fy);
    ay += (double)(vx * fy + vy * fx);
  }
  const float w = win[pix];
  float2 *o = bins + (int64_t)(c0 + k) * SS + pix;
  float2 b = *o;
  b.x += (float)ax * w;
  b.y += (float)ay * w;
  *o = b;
}

// Chunk numbers ub, vb = floor(u theta / chunk + 0.5) and w-plane rint(w /
// wstep) of every visibility, their ranges, and the antenna indices checked.
__global__ void k_awt_bins(const double *__restrict__ uvw, int64_t nv, int64_t stride,
                           double theta, double wstep, int chunk,
                           const int64_t *__restrict__ src, int64_t nant, int4 *__restrict__ bin,
                           int *__restrict__ range, uint32_t *__restrict__ status) {
#pragma clang fp contract(off)
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int v[3] = {INT_MAX, INT_MAX, INT_MAX}, w[3] = {INT_MIN, INT_MIN, INT_MIN};
  if (i < nv) {
    const double a = floor(uvw[i * stride] * theta / (double)chunk + 0.5);
    const double b = floor(uvw[i * stride + 1] * theta / (double)chunk + 0.5);
    const double c = rint(uvw[i * stride + 2] / wstep);
    const int64_t s1 = src[2 * i], s2 = src[2 * i + 1];
    if (!(fabs(a) < 0x1p30 && fabs(b) < 0x1p30 && fabs(c) < 0x1p30)) {
      atomicOr(status, (uint32_t)ST_DOMAIN);
    } else if (s1 < 0 || s2 < 0 || s1 >= nant || s2 >= nant) {
      atomicOr(status, (uint32_t)ST_PLANE);
    } else {
      v[0] = w[0] = (int)a;
      v[1] = w[1] = (int)b;
      v[2] = w[2] = (int)c;
      bin[i] = make_int4((int)a, (int)b, (int)c, 0);
    }
  }
  __shared__ int s_lo[3], s_hi[3];
  if (threadIdx.x < 3) {
    s_lo[threadIdx.x] = INT_MAX;
    s_hi[threadIdx.x] = INT_MIN;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
      v[k] = min(v[k], __shfl_xor(v[k], off, 64));
      w[k] = max(w[k], __shfl_xor(w[k], off, 64));
    }
    if ((threadIdx.x & 63) == 0) {
      atomicMin(&s_lo[k], v[k]);
      atomicMax(&s_hi[k], w[k]);
    }
  }
  barrier_after_lds_atomics();
  if (threadIdx.x < 3 && s_lo[threadIdx.x] <= s_hi[threadIdx.x]) {
    atomicMin(&range[threadIdx.x], s_lo[threadIdx.x]);
    atomicMax(&range[3 + threadIdx.x], s_hi[threadIdx.x]);
  }
}

__global__ void k_awt_range_init(int *range, uint32_t *status) {
  if (threadIdx.x < 3) range[threadIdx.x] = INT_MAX;
  else if (threadIdx.x < 6) range[threadIdx.x] = INT_MIN;
  if (threadIdx.x == 6) *status = 0u;
}

// Groups whose chunk keys and starts come to the host at a time: 1 MiB of the
// context's pinned staging, which lives as long as the context.
constexpr int AWG_STAGE = 65536;

struct AwtRange {
  int ub, vb, wp;      // lowest
  int64_t nvb, P, nant;
};

// Group key (chunk, plane, antenna pair) and index of every visibility.
__global__ void k_awt_keys(const int4 *__restrict__ bin, const int64_t *__restrict__ src,
                           int64_t nv, AwtRange r, uint64_t *__restrict__ key,
                           int32_t *__restrict__ idx) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const int4 b = bin[i];
  const uint64_t cid = (uint64_t)(b.x - r.ub) * r.nvb + (uint64_t)(b.y - r.vb);
  key[i] = ((cid * r.P + (uint64_t)(b.z - r.wp)) * r.nant + (uint64_t)src[2 * i]) * r.nant +
           (uint64_t)src[2 * i + 1];
  idx[i] = (int32_t)i;
}

// Per group its plane and antennas, and for the host its chunk key and start;
// vstart's end.
__global__ void k_awt_groups(const uint64_t *__restrict__ gkey, int ng, int64_t nv, AwtRange r,
                             int32_t *__restrict__ gwp, int32_t *__restrict__ ga1,
                             int32_t *__restrict__ ga2, ulonglong2 *__restrict__ gout,
                             int32_t *__restrict__ vstart) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g == 0) vstart[ng] = (int32_t)nv;
  if (g >= ng) return;
  uint64_t k = gkey[g];
  ga2[g] = (int32_t)(k % r.nant);
  k /= r.nant;
  ga1[g] = (int32_t)(k % r.nant);
  k /= r.nant;
  gwp[g] = (int32_t)(k % r.P) + r.wp;
  gout[g] = make_ulonglong2(k / r.P, (unsigned long long)vstart[g]);
}

// Sorted visibility v: its group (the last start <= v) and its coordinates
// relative to the group's chunk middle and plane.
__global__ void k_awt_rel(const double *__restrict__ uvw, int64_t nv, int64_t stride,
                          const int32_t *__restrict__ order, const int4 *__restrict__ bin,
                          const int32_t *__restrict__ vstart, int ng, double theta, double wstep,
                          int chunk, int32_t *__restrict__ gid, double *__restrict__ rel) {
#pragma clang fp contract(off)
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  int lo = 0, hi = ng - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (vstart[mid] <= v) lo = mid; else hi = mid - 1;
  }
  gid[v] = lo;
  const int64_t i = order[v];
  const int4 b = bin[i];
  rel[3 * v] = uvw[i * stride] - (double)chunk * (double)b.x / theta;
  rel[3 * v + 1] = uvw[i * stride + 1] - (double)chunk * (double)b.y / theta;
  rel[3 * v + 2] = uvw[i * stride + 2] - (double)b.z * wstep;
}

// Window corner and sub-offsets {xs, ys, xf, yf} of every visibility on the M
// grid, as k_awt_pregrid places it.
__global__ void k_awt_locate(const double *__restrict__ rel, int64_t nv, double lam_sub, int M,
                             int Q, int K, int4 *__restrict__ loc, uint32_t *status) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  const double px = grid_fraction(rel[v * 3], lam_sub);
  const double py = grid_fraction(rel[v * 3 + 1], lam_sub);
  int x, xf, y, yf;
  if (!frac_coord_dev(M, Q, px, &x, &xf) || !frac_coord_dev(M, Q, py, &y, &yf)) {
    atomicOr(status, (uint32_t)ST_DOMAIN);
    return;
  }
  const int xs = x - K / 2, ys = y - K / 2;
  if (xs < 0 || ys < 0 || xs + K > M || ys + K > M) {
    atomicOr(status, (uint32_t)ST_BOUNDS);
    return;
  }
  loc[v] = make_int4(xs, ys, xf, yf);
}

// Chunk images without pre-grids: pixel (y, x) of the cut-out inverse
// transform of a group's pre-grid (times M^2) is
//   sum over its visibilities of v Y[y] X[x],
//   X[x] = sum_j gcf[xf][j] W^((xs + j - S)(x - S/2)),  W = exp(2 pi i / M),
// Y likewise with the rows.  segs[blockIdx.y] = (first group, first
// visibility, end visibility, out): the workgroup sums its AWD_T x AWD_T
// pixel tile (blockIdx.x) over the segment's visibilities -- per group times
// the pair's A-screen ratio and wkern^-wp, the plane factor taken once per
// plane -- and writes bins[~out] times win (out < 0) or the FP64 sum to
// part[out].  A group may be cut between segments: its parts are summed in
// FP64, like everything above a run of at most AWD_FOLD + AWD_VB - 1
// visibilities.
//
// Work: 8 S^2 operations per visibility and ~30 S^2 per group in registers,
// no traffic but the screens (L2) and 24 + 32 bytes per visibility.  A
// pre-grid and its (2S)^2 transform move 24 (2S)^2 bytes per group, whatever
// the group holds; AW-towers groups hold a few visibilities (27 antennas x
// 36 dumps at S = 128: 1.8).  The exponents are integers reduced mod M and
// looked up in an FP64-rounded table, so the vectors carry FP32 rounding of
// K terms only.  awtowers1800 (6991 groups, 12636 visibilities): 289 us in
// place of 6.1 ms (clear, pre-grid, transform and its copies, apply).  Bound
// mainly by VALU issue: 126 million wave instructions, 205 us at 4 clocks on
// 1024 SIMDs, against 3.8 million LDS and 5.4 million vector load ones.  So
// 8, 16 or 32 vectors staged at a time differ by 3 % at most.
//
// The vectors are centred, so the images carry the centring sign
// (-1)^(x + y) that the pre-grids' uncentred transforms leave out (the input
// half of the chunk images' forward transform).
__device__ __forceinline__ float chunk_window(const float *__restrict__ win, int pix, int S) {
  const int y = pix / S, x = pix - y * S;
  return ((x + y) & 1) ? -win[pix] : win[pix];
}

constexpr int AWD_T = 32;    // tile edge (pixels)
constexpr int AWD_NT = 256;  // threads: column tid % 32, rows 4 (tid / 32) + q
constexpr int AWD_VB = 16;   // visibilities whose vectors are staged at a time
constexpr int AWD_FOLD = 32;  // visibilities after which a group's FP32 sum is folded
constexpr int AWD_MAX_M = 4096;  // twiddle table in LDS: 8 M bytes

__global__ __launch_bounds__(AWD_NT) void k_awt_direct(
    float2 *__restrict__ bins, double2 *__restrict__ part, int S, const int4 *__restrict__ segs,
    const int32_t *__restrict__ vstart, const int32_t *__restrict__ gwp,
    const int32_t *__restrict__ ga1, const int32_t *__restrict__ ga2,
    const int4 *__restrict__ loc, const float2 *__restrict__ vis,
    const float2 *__restrict__ gcf, int K, const float2 *__restrict__ ascreen,
    const float *__restrict__ win, const double *__restrict__ turns,
    const float *__restrict__ lmag) {
  extern __shared__ float2 s_tw[];                // [M]
  __shared__ __align__(16) float2 s_xy[AWD_VB][2 * AWD_T];  // X (first AWD_T), then v Y
  const int tid = threadIdx.x, M = 2 * S, SS = S * S;
  for (int k = tid; k < M; k += AWD_NT) {
    double s, c;
    sincospi(2.0 * (double)k / (double)M, &s, &c);
    s_tw[k] = make_float2((float)c, (float)s);
  }
  const int nt = (S + AWD_T - 1) / AWD_T;
  const int ty0 = (int)(blockIdx.x / nt) * AWD_T, tx0 = (int)(blockIdx.x % nt) * AWD_T;
  const int4 seg = segs[blockIdx.y];
  const int lx = tid & (AWD_T - 1), ly = tid / AWD_T;
  const int x = tx0 + lx;
  int pix[4];
  double tw[4];
  float lm[4];
  bool in[4];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int y = ty0 + 4 * ly + q;
    in[q] = x < S && y < S;
    pix[q] = in[q] ? y * S + x : 0;  // pixel 0 stands in (never written)
    tw[q] = turns[pix[q]];
    lm[q] = lmag[pix[q]];
  }
  double ax[4] = {0.0, 0.0, 0.0, 0.0}, ay[4] = {0.0, 0.0, 0.0, 0.0};  // finished planes
  double sx[4] = {0.0, 0.0, 0.0, 0.0}, sy[4] = {0.0, 0.0, 0.0, 0.0};  // the open plane
  float ix[4] = {0.f, 0.f, 0.f, 0.f}, iy[4] = {0.f, 0.f, 0.f, 0.f};   // the open group
  int g = seg.x;
  int wp = gwp[g];
  int gend = vstart[g + 1];
  float2 p[4], r[4];  // the open group's screens
  auto screens = [&]() {
    const float2 *a = ascreen + (int64_t)ga1[g] * SS, *b = ascreen + (int64_t)ga2[g] * SS;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      p[q] = a[pix[q]];
      r[q] = b[pix[q]];
    }
  };
  auto close_group = [&]() {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      // r / p = r conj(p) / |p|^2
      const float inv = 1.0f / (p[q].x * p[q].x + p[q].y * p[q].y);
      const float rx = (r[q].x * p[q].x + r[q].y * p[q].y) * inv;
      const float ry = (r[q].y * p[q].x - r[q].x * p[q].y) * inv;
      sx[q] += (double)(ix[q] * rx - iy[q] * ry);
      sy[q] += (double)(ix[q] * ry + iy[q] * rx);
      ix[q] = 0.f;
      iy[q] = 0.f;
    }
  };
  auto close_plane = [&]() {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const double t = -(double)wp * tw[q];
      float s, c;
      sincospif((float)(2.0 * (t - rint(t))), &s, &c);
      const float mag = lm[q] == 0.0f ? 1.0f : exp2f(-(float)wp * lm[q]);
      const double fx = c * mag, fy = s * mag;
      ax[q] += sx[q] * fx - sy[q] * fy;
      ay[q] += sx[q] * fy + sy[q] * fx;
      sx[q] = 0.0;
      sy[q] = 0.0;
    }
  };
  screens();
  const int v1 = seg.z;
  int open = seg.y;  // first visibility of the open FP32 sum
  for (int v0 = seg.y; v0 < v1; v0 += AWD_VB) {
    const int m = min(AWD_VB, v1 - v0);
    if (v0 - open >= AWD_FOLD) {
      close_group();
      open = v0;
    }
    __syncthreads();  // table written; the previous vectors read
    for (int e = tid; e < m * 2 * AWD_T; e += AWD_NT) {
      const int k = e / (2 * AWD_T), j = e % (2 * AWD_T);
      const bool row = j >= AWD_T;
      const int4 L = loc[v0 + k];
      const int b = (row ? ty0 + j - AWD_T : tx0 + j) - S / 2;  // centred pixel
      const float2 *gk = gcf + (int64_t)(row ? L.w : L.z) * K;
      int idx = ((row ? L.y : L.x) - S) * b % M;
      if (idx < 0) idx += M;
      int step = b % M;
      if (step < 0) step += M;
      float2 a = make_float2(0.f, 0.f);
      for (int i = 0; i < K; i++) {
        const float2 w = s_tw[idx], t = gk[i];
        a.x = fmaf(t.x, w.x, fmaf(-t.y, w.y, a.x));
        a.y = fmaf(t.x, w.y, fmaf(t.y, w.x, a.y));
        idx += step;
        if (idx >= M) idx -= M;
      }
      s_xy[k][j] = row ? cmul(vis[v0 + k], a) : a;
    }
    __syncthreads();
    for (int k = 0; k < m; k++) {
      if (v0 + k == gend) {  // groups hold at least one visibility
        close_group();
        open = v0 + k;
        g++;
        const int w = gwp[g];
        if (w != wp) close_plane();
        wp = w;
        gend = vstart[g + 1];
        screens();
      }
      const float2 X = s_xy[k][lx];
      const float4 *Y4 = (const float4 *)&s_xy[k][AWD_T + 4 * ly];
      const float4 ya = Y4[0], yb = Y4[1];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float4 y2 = q < 2 ? ya : yb;
        const float2 Y = q % 2 ? make_float2(y2.z, y2.w) : make_float2(y2.x, y2.y);
        ix[q] = fmaf(X.x, Y.x, fmaf(-X.y, Y.y, ix[q]));
        iy[q] = fmaf(X.x, Y.y, fmaf(X.y, Y.x, iy[q]));
      }
    }
  }
  close_group();
  close_plane();
#pragma unroll
  for (int q = 0; q < 4; q++) {
    if (!in[q]) continue;
    if (seg.w < 0) {
      const float w = chunk_window(win, pix[q], S);
      bins[(int64_t)~seg.w * SS + pix[q]] = make_float2((float)ax[q] * w, (float)ay[q] * w);
    } else {
      part[(int64_t)seg.w * SS + pix[q]] = make_double2(ax[q], ay[q]);
    }
  }
}

// bins[red[k].x] = win * sum of part[red[k].y .. red[k].z - 1], in order.
__global__ void k_awt_reduce(float2 *__restrict__ bins, const double2 *__restrict__ part, int S,
                             const int4 *__restrict__ red, const float *__restrict__ win) {
  const int SS = S * S;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= SS) return;
  const int4 r = red[blockIdx.y];
  double ax = 0.0, ay = 0.0;
#pragma unroll 4
  for (int k = r.y; k < r.z; k++) {
    const double2 a = part[(int64_t)k * SS + pix];
    ax += a.x;
    ay += a.y;
  }
  const float w = chunk_window(win, pix, S);
  bins[(int64_t)r.x * SS + pix] = make_float2((float)ax * w, (float)ay * w);
}

// grid[y0 + y][x0 + x] += (-1)^(x+y) * bins[c][y][x] inside the grid.
__global__ void k_awt_place(float2 *__restrict__ grid, int N,
                            const float2 *__restrict__ bins, int S,
                            const int32_t *__restrict__ corner) {
  const int SS = S * S;
  const int pix = blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= SS) return;
  const int c = blockIdx.y;
  const int y = pix / S, x = pix - y * S;
  const int gx = corner[2 * c] + x, gy = corner[2 * c + 1] + y;
  if (gx < 0 || gy < 0 || gx >= N || gy >= N) return;
  float2 b = bins[(int64_t)c * SS + pix];
  if ((x + y) & 1) {
    b.x = -b.x;
    b.y = -b.y;
  }
  float *g = (float *)(grid + (int64_t)gy * N + gx);
  unsafeAtomicAdd(g, b.x);
  unsafeAtomicAdd(g + 1, b.y);
}

}  // namespace

extern "C" int croc_awt_pregrid(croc_ctx *ctx, void *stack, int M, const double *rel,
                                int64_t v0, int64_t v1, double lam_sub, int Q, int K,
                                const void *gcf, const void *vis, const int32_t *gid,
                                int32_t g0, int check_only) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(M >= 2 && M % 2 == 0 && Q >= 1 && K >= 1 && K <= M && lam_sub > 0 &&
                   v0 >= 0 && v1 >= v0,
               CROC_EINVAL, "bad arguments");
  if (v1 == v0) return CROC_OK;
  CROC_REQUIRE(rel && gcf && vis && gid && (check_only || stack), CROC_EINVAL, "null array");
  uint32_t *st;
  if ((rc = small_status(ctx, &st))) return rc;
  const int64_t nt = (v1 - v0) * K;
  k_awt_pregrid<<<(unsigned)((nt + 255) / 256), 256, 0, ctx->stream>>>(
      (float2 *)stack, M, rel, v0, v1, lam_sub, Q, K, (const float2 *)gcf,
      (const float2 *)vis, gid, g0, check_only ? 0 : 1, st);
  CROC_HIP(hipGetLastError());
  if (check_only) return finish_status(ctx, st);
  return CROC_OK;
}

extern "C" int croc_awt_apply(croc_ctx *ctx, void *bins, int c0, int nc, const void *stack,
                              int S, const int32_t *start, const int32_t *gwp,
                              const int32_t *ga1, const int32_t *ga2, const void *ascreen,
                              const float *win, const double *turns, const float *lmag) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(S >= 2 && S % 2 == 0 && c0 >= 0 && nc >= 0 && nc < 65536, CROC_EINVAL,
               "bad arguments");
  if (nc == 0) return CROC_OK;
  CROC_REQUIRE(bins && stack && start && gwp && ga1 && ga2 && ascreen && win && turns && lmag,
               CROC_EINVAL, "null array");
  dim3 grid((unsigned)((S * S + 255) / 256), (unsigned)nc);
  k_awt_apply<<<grid, 256, 0, ctx->stream>>>((float2 *)bins, c0, (const float2 *)stack, S,
                                             start, gwp, ga1, ga2,
                                             (const float2 *)ascreen, win, turns, lmag);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}

extern "C" int croc_awt_groups(croc_ctx *ctx, const double *uvw, int64_t nv, int64_t stride,
                               double theta, double wstep, int chunk, const int64_t *src,
                               int64_t nant, int32_t *order, int32_t *vstart, int32_t *gid,
                               double *rel, int32_t *gwp, int32_t *ga1, int32_t *ga2,
                               int64_t *ngroups, int64_t *nchunks, int32_t *vstart_h,
                               int64_t *cstart, int32_t *cub, int32_t *cvb) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(nv >= 1 && nv < (int64_t)INT32_MAX && stride >= 3 && theta > 0 && wstep != 0 &&
                   chunk >= 1 && nant >= 1,
               CROC_EINVAL, "bad arguments");
  CROC_REQUIRE(uvw && src && order && vstart && gid && rel && gwp && ga1 && ga2 && ngroups &&
                   nchunks && vstart_h && cstart && cub && cvb,
               CROC_EINVAL, "null array");
  const size_t n = (size_t)nv;
  hipStream_t s = ctx->stream;
  uint64_t *key = nullptr, *skey = nullptr, *gkey = nullptr;
  int32_t *idx = nullptr, *count = nullptr;
  size_t t_sort = 0, t_rle = 0, t_scan = 0;
  CROC_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, t_sort, key, skey, idx, order, (int)n, 0,
                                              64, s));
  CROC_HIP(hipcub::DeviceRunLengthEncode::Encode(nullptr, t_rle, skey, gkey, count,
                                                 (int32_t *)nullptr, (int)n, s));
  CROC_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, t_scan, count, vstart, (int)n, s));
  const size_t tb = std::max(t_sort, std::max(t_rle, t_scan));
  char *w = (char *)ws_get(ctx, WS_SORT, 512 + n * (16 + 3 * 8 + 2 * 4) + tb + 256);
  int *small = (int *)ws_get(ctx, WS_SMALL, 256);
  ulonglong2 *h = (ulonglong2 *)host_stage(
      ctx, std::max<size_t>(sizeof(ulonglong2) * std::min<size_t>(n, AWG_STAGE), 256));
  if (!w || !small || !h) return CROC_ENOMEM;
  int4 *bin = (int4 *)w;
  key = (uint64_t *)(bin + n);
  skey = key + n;
  gkey = skey + n;
  idx = (int32_t *)(gkey + n);
  count = idx + n;
  void *temp = (void *)(((uintptr_t)(count + n) + 255) & ~(uintptr_t)255);
  uint32_t *st = (uint32_t *)small;
  int *range = small + 8, *nruns = small + 16;
  const unsigned nb = (unsigned)((nv + 255) / 256);
  k_awt_range_init<<<1, 64, 0, s>>>(range, st);
  k_awt_bins<<<nb, 256, 0, s>>>(uvw, nv, stride, theta, wstep, chunk, src, nant, bin, range, st);
  CROC_HIP(hipGetLastError());
  CROC_HIP(hipMemcpyAsync(h, small, 128, hipMemcpyDeviceToHost, s));
  CROC_HIP(hipStreamSynchronize(s));
  {
    const uint32_t bits = *(const uint32_t *)h;
    if (bits & ST_PLANE) {
      croc_set_error("antenna index outside the A-screens");
      return CROC_EPLANE;
    }
    if ((rc = croc_status_to_code(bits))) return rc;
  }
  const int *hr = (const int *)h + 8;
  AwtRange r{hr[0], hr[1], hr[2], (int64_t)hr[4] - hr[1] + 1, (int64_t)hr[5] - hr[2] + 1, nant};
  const double keys = ((double)hr[3] - hr[0] + 1) * (double)r.nvb * (double)r.P * (double)nant *
                      (double)nant;
  CROC_REQUIRE(keys < 0x1p62, CROC_EINVAL,
               "too many (chunk, w-plane, antenna pair) groups; increase wstep");
  int end_bit = 1;
  while (end_bit < 62 && ldexp(1.0, end_bit) < keys) end_bit++;
  k_awt_keys<<<nb, 256, 0, s>>>(bin, src, nv, r, key, idx);
  size_t t = tb;
  CROC_HIP(hipcub::DeviceRadixSort::SortPairs(temp, t, key, skey, idx, order, (int)n, 0, end_bit,
                                              s));
  t = tb;
  CROC_HIP(hipcub::DeviceRunLengthEncode::Encode(temp, t, skey, gkey, count, nruns, (int)n, s));
  CROC_HIP(hipMemcpyAsync(h, nruns, sizeof(int), hipMemcpyDeviceToHost, s));
  CROC_HIP(hipStreamSynchronize(s));
  const int ng = *(const int *)h;
  t = tb;
  CROC_HIP(hipcub::DeviceScan::ExclusiveSum(temp, t, count, vstart, ng, s));
  ulonglong2 *gout = (ulonglong2 *)key;  // over key and skey, no longer needed
  k_awt_groups<<<(unsigned)((ng + 255) / 256), 256, 0, s>>>(gkey, ng, nv, r, gwp, ga1, ga2, gout,
                                                            vstart);
  k_awt_rel<<<nb, 256, 0, s>>>(uvw, nv, stride, order, bin, vstart, ng, theta, wstep, chunk, gid,
                               rel);
  CROC_HIP(hipGetLastError());
  int64_t nc = 0;
  uint64_t last = 0;
  for (int g0 = 0; g0 < ng; g0 += AWG_STAGE) {
    const int m = std::min(AWG_STAGE, ng - g0);
    CROC_HIP(hipMemcpyAsync(h, gout + g0, sizeof(ulonglong2) * m, hipMemcpyDeviceToHost, s));
    CROC_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < m; k++) {
      const uint64_t cid = h[k].x;
      vstart_h[g0 + k] = (int32_t)h[k].y;
      if (g0 + k == 0 || cid != last) {
        cub[nc] = (int32_t)(cid / (uint64_t)r.nvb) + r.ub;
        cvb[nc] = (int32_t)(cid % (uint64_t)r.nvb) + r.vb;
        cstart[nc++] = g0 + k;
      }
      last = cid;
    }
  }
  vstart_h[ng] = (int32_t)nv;
  cstart[nc] = ng;
  *ngroups = ng;
  *nchunks = nc;
  return CROC_OK;
}

extern "C" int croc_awt_direct(croc_ctx *ctx, void *bins, int nc, int S, const double *rel,
                               int64_t nv, double lam_sub, int Q, int K, const void *gcf,
                               const void *vis, const int32_t *vstart,
                               const int32_t *vstart_h, const int64_t *cstart,
                               const int32_t *gwp, const int32_t *ga1, const int32_t *ga2,
                               const void *ascreen, const float *win, const double *turns,
                               const float *lmag, int64_t max_bytes) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  const int M = 2 * S;
  CROC_REQUIRE(S >= 2 && S % 2 == 0 && M <= AWD_MAX_M && Q >= 1 && K >= 1 && K <= M &&
                   lam_sub > 0 && nc >= 0 && nv >= 0 && nv < (int64_t)INT32_MAX,
               CROC_EINVAL, "bad arguments");
  if (nc == 0 || nv == 0) return CROC_OK;
  CROC_REQUIRE(bins && rel && gcf && vis && vstart && vstart_h && cstart && gwp && ga1 && ga2 && ascreen &&
                   win && turns && lmag,
               CROC_EINVAL, "null array");
  for (int c = 0; c < nc; c++) {
    const int64_t a = cstart[c], b = cstart[c + 1];
    CROC_REQUIRE(a >= 0 && a < b && b <= nv, CROC_EINVAL, "chunk %d holds no groups", c);
    CROC_REQUIRE(vstart_h[a] >= 0 && vstart_h[b] <= nv, CROC_EINVAL, "bad group range");
  }
  // Segments of one chunk of at most `groups` groups and `visibs`
  // visibilities, cutting through groups, so that the crowded chunks at the
  // centre of the uv plane and the groups of a dense core spread over the
  // chip; a chunk of one segment writes its image itself, the others leave
  // FP64 partial sums (longer segments where those would exceed max_bytes).
  // 512 visibilities, a few times what 64 groups of the sparse arrays hold,
  // take their workgroups about 0.1 ms.
  const int SS = S * S;
  int64_t groups = 64, visibs = 512;
  std::vector<int4> segs, red;
  int64_t npart;
  for (;; groups *= 2, visibs *= 2) {
    segs.clear();
    red.clear();
    npart = 0;
    for (int c = 0; c < nc; c++) {
      const size_t first = segs.size();
      int64_t g = cstart[c], v = vstart_h[g];
      const int64_t gend = cstart[c + 1], vend = vstart_h[gend];
      while (v < vend) {
        const int64_t e =
            std::min<int64_t>(v + visibs, vstart_h[std::min(gend, g + groups)]);
        CROC_REQUIRE(e > v, CROC_EINVAL, "empty group %lld", (long long)g);
        segs.push_back(make_int4((int)g, (int)v, (int)e, ~c));
        v = e;  // in the last group that starts at or before it
        g = std::upper_bound(vstart_h + g, vstart_h + gend, (int32_t)v) - vstart_h - 1;
      }
      const int64_t n = (int64_t)(segs.size() - first);
      if (n > 1) {
        red.push_back(make_int4(c, (int)npart, (int)(npart + n), 0));
        for (int64_t k = 0; k < n; k++) segs[first + k].w = (int)(npart + k);
        npart += n;
      }
    }
    if (npart == 0 || npart * SS * (int64_t)sizeof(double2) <= max_bytes) break;
  }
  const size_t ns = segs.size(), nr = red.size();
  int4 *d = (int4 *)ws_get(ctx, WS_TOWER, sizeof(int4) * (ns + nr));
  int4 *loc = (int4 *)ws_get(ctx, WS_LOC, sizeof(int4) * (size_t)nv);
  double2 *part = (double2 *)ws_get(ctx, WS_SUB, sizeof(double2) * (size_t)npart * SS);
  int4 *h = (int4 *)host_stage(ctx, sizeof(int4) * (ns + nr));
  if (!d || !loc || !part || !h) return CROC_ENOMEM;
  std::copy(segs.begin(), segs.end(), h);
  std::copy(red.begin(), red.end(), h + ns);
  hipStream_t s = ctx->stream;
  CROC_HIP(hipMemcpyAsync(d, h, sizeof(int4) * (ns + nr), hipMemcpyHostToDevice, s));
  uint32_t *st;
  if ((rc = small_status(ctx, &st))) return rc;
  k_awt_locate<<<(unsigned)((nv + 255) / 256), 256, 0, s>>>(rel, nv, lam_sub, M, Q, K, loc, st);
  CROC_HIP(hipGetLastError());
  // every window checked before any is used; the upload has been read, too
  if ((rc = finish_status(ctx, st))) return rc;
  const int nt = (S + AWD_T - 1) / AWD_T;
  for (size_t k = 0; k < ns; k += 65535) {
    const unsigned n = (unsigned)std::min<size_t>(65535, ns - k);
    k_awt_direct<<<dim3((unsigned)(nt * nt), n), AWD_NT, sizeof(float2) * M, s>>>(
        (float2 *)bins, part, S, d + k, vstart, gwp, ga1, ga2, loc, (const float2 *)vis,
        (const float2 *)gcf, K, (const float2 *)ascreen, win, turns, lmag);
    CROC_HIP(hipGetLastError());
  }
  for (size_t k = 0; k < nr; k += 65535) {
    const unsigned n = (unsigned)std::min<size_t>(65535, nr - k);
    k_awt_reduce<<<dim3((unsigned)((SS + 255) / 256), n), 256, 0, s>>>(
        (float2 *)bins, part, S, d + ns + k, win);
    CROC_HIP(hipGetLastError());
  }
  return CROC_OK;
}

extern "C" int croc_awt_place(croc_ctx *ctx, void *grid, int N, const void *bins, int nc,
                              int S, const int32_t *corner) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(N >= 1 && S >= 2 && S % 2 == 0 && nc >= 0 && nc < 65536, CROC_EINVAL,
               "bad arguments");
  if (nc == 0) return CROC_OK;
  CROC_REQUIRE(grid && bins && corner, CROC_EINVAL, "null array");
  dim3 g((unsigned)((S * S + 255) / 256), (unsigned)nc);
  k_awt_place<<<g, 256, 0, ctx->stream>>>((float2 *)grid, N, (const float2 *)bins, S, corner);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}
