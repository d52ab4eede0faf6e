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
#include <vector>

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
// Y likewise with the rows.  segs[blockIdx.y] = (chunk, first group, end
// group, out): the workgroup sums its AWD_T x AWD_T pixel tile (blockIdx.x)
// over the segment's groups -- per group times the pair's A-screen ratio and
// wkern^-wp, the plane factor taken once per plane -- and writes
// bins[chunk] times win (out < 0) or the FP64 sum to part[out].
//
// Work: 8 S^2 operations per visibility and ~30 S^2 per group in registers,
// no traffic but the screens (L2) and 24 + 32 bytes per visibility.  A
// pre-grid and its (2S)^2 transform move 24 (2S)^2 bytes per group, whatever
// the group holds; AW-towers groups hold a few visibilities (27 antennas x
// 36 dumps at S = 128: 1.8).  The exponents are integers reduced mod M and
// looked up in an FP64-rounded table, so the vectors carry FP32 rounding of
// K terms only.  awtowers1800 (6991 groups, 12636 visibilities): 312 us in
// place of 6.1 ms (clear, pre-grid, transform and its copies, apply); bound by
// the LDS reads of the vectors (5 per 4 pixels and visibility).
//
// The vectors are centred, so the images carry the centring sign
// (-1)^(x + y) that the pre-grids' uncentred transforms leave out (the input
// half of the chunk images' forward transform).
__device__ __forceinline__ float chunk_window(const float *__restrict__ win, int pix, int S) {
  const int y = pix / S, x = pix - y * S;
  return ((x + y) & 1) ? -win[pix] : win[pix];
}

constexpr int AWD_T = 32;    // tile edge (pixels)
constexpr int AWD_NT = 256;  // threads: column tid % 32, rows tid / 32 + 8 q
constexpr int AWD_VB = 16;   // visibilities whose vectors are staged at a time
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
  __shared__ float2 s_xy[AWD_VB][2 * AWD_T];      // X (first AWD_T), then v Y
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
    const int y = ty0 + ly + 8 * q;
    in[q] = x < S && y < S;
    pix[q] = in[q] ? y * S + x : 0;  // pixel 0 stands in (never written)
    tw[q] = turns[pix[q]];
    lm[q] = lmag[pix[q]];
  }
  double ax[4] = {0.0, 0.0, 0.0, 0.0}, ay[4] = {0.0, 0.0, 0.0, 0.0};  // finished planes
  double sx[4] = {0.0, 0.0, 0.0, 0.0}, sy[4] = {0.0, 0.0, 0.0, 0.0};  // the open plane
  float ix[4] = {0.f, 0.f, 0.f, 0.f}, iy[4] = {0.f, 0.f, 0.f, 0.f};   // the open group
  int g = seg.y;
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
  const int v1 = vstart[seg.z];
  for (int v0 = vstart[g]; v0 < v1; v0 += AWD_VB) {
    const int m = min(AWD_VB, v1 - v0);
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
        g++;
        const int w = gwp[g];
        if (w != wp) close_plane();
        wp = w;
        gend = vstart[g + 1];
        screens();
      }
      const float2 X = s_xy[k][lx];
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float2 Y = s_xy[k][AWD_T + ly + 8 * q];
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
      bins[(int64_t)seg.x * SS + pix[q]] = make_float2((float)ax[q] * w, (float)ay[q] * w);
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

extern "C" int croc_awt_direct(croc_ctx *ctx, void *bins, int nc, int S, const double *rel,
                               int64_t nv, double lam_sub, int Q, int K, const void *gcf,
                               const void *vis, const int32_t *vstart, const int64_t *cstart,
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
  CROC_REQUIRE(bins && rel && gcf && vis && vstart && cstart && gwp && ga1 && ga2 && ascreen &&
                   win && turns && lmag,
               CROC_EINVAL, "null array");
  // Segments of at most `seg` groups of one chunk, so that the crowded chunks
  // at the centre of the uv plane spread over the chip; a chunk of one
  // segment writes its image itself, the others leave FP64 partial sums
  // (longer segments where those would exceed max_bytes).
  const int SS = S * S;
  int64_t seg = 64, most = 0;
  for (int c = 0; c < nc; c++) {
    const int64_t n = cstart[c + 1] - cstart[c];
    CROC_REQUIRE(cstart[c] >= 0 && n > 0 && cstart[c + 1] <= nv, CROC_EINVAL,
                 "chunk %d holds no groups", c);
    most = std::max(most, n);
  }
  auto parts_at = [&](int64_t len) {
    int64_t k = 0;
    for (int c = 0; c < nc; c++) {
      const int64_t n = (cstart[c + 1] - cstart[c] + len - 1) / len;
      k += n > 1 ? n : 0;
    }
    return k;
  };
  while (seg < most && parts_at(seg) * SS * (int64_t)sizeof(double2) > max_bytes) seg *= 2;
  std::vector<int4> segs, red;
  int npart = 0;
  for (int c = 0; c < nc; c++) {
    const int64_t a = cstart[c], b = cstart[c + 1], n = (b - a + seg - 1) / seg;
    for (int64_t k = 0; k < n; k++)
      segs.push_back(make_int4(c, (int)(a + k * seg), (int)std::min(b, a + (k + 1) * seg),
                               n == 1 ? -1 : npart + (int)k));
    if (n > 1) {
      red.push_back(make_int4(c, npart, npart + (int)n, 0));
      npart += (int)n;
    }
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
