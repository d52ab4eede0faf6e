// W-stacking (examples/notebooks/wstacking.ipynb, cell 10, JSON lines
// 191-240): visibilities binned by w-plane round-half-even(w / wstep), each
// plane gridded nearest-cell onto its own full grid, transformed, divided by
// the plane's Fresnel pattern w_kernel_function(l, m, mean w) and summed in
// image space.
//
// A batch of planes is one [P][N][N] stack: k_wstack_grid fills it in one
// pass over the visibilities (a plane -> slot table selects the batch), a
// batched inverse FFT runs over the stack (rocFFT), and k_wstack_add reads
// the P transformed planes of each pixel once, applies each plane's Fresnel
// phase and adds the sum into the FP64 image.  For even N the centring
// shifts of the centred FFT are folded into both kernels as the
// checkerboard sign (-1)^(x+y) (the product of the two axes' global factors
// exp(i pi N / 2) is 1), so no shift pass touches the stack.
#include <algorithm>

#include "fft128.h"

namespace {

// One visibility onto its plane's slot of the stack, nearest cell
// (synthesis.py:389-401: cell N//2 + floor(0.5 + N p), p = uvw / lam, every
// column of p, w included, below 0.5).  With apply == 0 only the checks run.
__global__ void k_wstack_grid(float2 *__restrict__ stack, int N,
                              const double *__restrict__ uvw, int64_t nv,
                              int64_t stride, double lam, double wstep,
                              int64_t plane0, int ntab,
                              const int32_t *__restrict__ slot_of,
                              const float2 *__restrict__ vis, int centred,
                              int apply, uint32_t *status) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nv) return;
  const double w = uvw[i * stride + 2];
  const int64_t t = wbin_dev(w, wstep) - plane0;
  if (t < 0 || t >= ntab) {
    atomicOr(status, (uint32_t)ST_PLANE);
    return;
  }
  const int slot = slot_of[t];
  if (slot < 0) return;
  const double px = grid_fraction(uvw[i * stride], lam);
  const double py = grid_fraction(uvw[i * stride + 1], lam);
  if (!(px < 0.5 && py < 0.5 && grid_fraction(w, lam) < 0.5)) {
    atomicOr(status, (uint32_t)ST_DOMAIN);
    return;
  }
  int x, y;
  if (!nearest_cell(N, px, &x) || !nearest_cell(N, py, &y)) {
    atomicOr(status, (uint32_t)ST_BOUNDS);
    return;
  }
  if (!apply) return;
  float2 v = vis[i];
  if (centred && ((x + y) & 1)) {
    v.x = -v.x;
    v.y = -v.y;
  }
  float *g = (float *)(stack + ((int64_t)slot * N + y) * N + x);
  unsafeAtomicAdd(g, v.x);
  unsafeAtomicAdd(g + 1, v.y);
}

// image[y][x] += sign * sum_p plane_p[y][x] * exp(-2 pi i midw[p] n1) with
// n1 = 1 - sqrt(1 - l^2 - m^2), l = theta (x - N//2) / N, m likewise in y
// (synthesis.py:66-80 coordinates2, :273-293 w_kernel_function; dividing by
// exp(2 pi i w n1) is multiplying by its conjugate).  The phase is reduced
// to turns in FP64 (midw n1 - rint(midw n1)) before the FP32 sincospi, so
// large |w| n1 keep their accuracy.
__global__ void k_wstack_add(double2 *__restrict__ image,
                             const float2 *__restrict__ stack, int P, int N,
                             double theta, const double *__restrict__ midw,
                             int centred) {
#pragma clang fp contract(off)
  const int64_t NN = (int64_t)N * N;
  const int64_t pix = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pix >= NN) return;
  const int y = (int)(pix / N), x = (int)(pix - (int64_t)y * N);
  const double l = theta * ((double)(x - N / 2) / (double)N);
  const double m = theta * ((double)(y - N / 2) / (double)N);
  const double n1 = 1.0 - sqrt(1.0 - (l * l + m * m));
  double ax = 0.0, ay = 0.0;
  const float2 *src = stack + pix;
  int p = 0;
  for (; p + 4 <= P; p += 4) {
    float2 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = src[(int64_t)(p + k) * NN];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const double t = midw[p + k] * n1;
      float s, c;
      sincospif((float)(2.0 * (t - rint(t))), &s, &c);
      ax += (double)v[k].x * c + (double)v[k].y * s;
      ay += (double)v[k].y * c - (double)v[k].x * s;
    }
  }
  for (; p < P; ++p) {
    const float2 v = src[(int64_t)p * NN];
    const double t = midw[p] * n1;
    float s, c;
    sincospif((float)(2.0 * (t - rint(t))), &s, &c);
    ax += (double)v.x * c + (double)v.y * s;
    ay += (double)v.y * c - (double)v.x * s;
  }
  if (centred && ((x + y) & 1)) {
    ax = -ax;
    ay = -ay;
  }
  double2 o = image[pix];
  o.x += ax;
  o.y += ay;
  image[pix] = o;
}

__global__ void k_w_bins(const double *__restrict__ w, int64_t nv, int64_t stride, double wstep,
                         int64_t *__restrict__ bin) {
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += step)
    bin[i] = wbin_dev(w[i * stride], wstep);
}

// Visibility count and sum of w of every w-plane t = round-half-even(w /
// wstep) - plane0, t < ntab: block-private histograms in LDS (sums by FP64 LDS
// atomics), one global atomic per block and non-empty plane.  A plane outside
// the table raises ST_PLANE.  wstack2048 (2e6 visibilities, 65 planes):
// 19 us for both, bound by the strided reads of w, where a global-atomic
// weighted histogram took 4.05 ms (every wavefront's FP64 adds fall on the
// same few lines of L2).
constexpr int PLANES_LDS = 4096;  // 48 KiB of LDS

template <bool LDS>
__global__ __launch_bounds__(512) void k_wplane_sums(const double *__restrict__ uvw, int64_t nv,
                                                     int64_t stride, double wstep,
                                                     int64_t plane0, int ntab,
                                                     unsigned long long *__restrict__ count,
                                                     double *__restrict__ sum, uint32_t *status) {
  __shared__ double s_sum[LDS ? PLANES_LDS : 1];
  __shared__ unsigned int s_n[LDS ? PLANES_LDS : 1];
  if (LDS) {
    for (int t = threadIdx.x; t < ntab; t += blockDim.x) {
      s_sum[t] = 0.0;
      s_n[t] = 0u;
    }
    __syncthreads();
  }
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nv; i += step) {
    const double w = uvw[i * stride + 2];
    const int64_t t = wbin_dev(w, wstep) - plane0;
    if (t < 0 || t >= ntab) {
      atomicOr(status, (uint32_t)ST_PLANE);
      continue;
    }
    if (LDS) {
      unsafeAtomicAdd(&s_sum[t], w);
      atomicAdd(&s_n[t], 1u);
    } else {
      unsafeAtomicAdd(&sum[t], w);
      atomicAdd(&count[t], 1ull);
    }
  }
  if (LDS) {
    barrier_after_lds_atomics();
    for (int t = threadIdx.x; t < ntab; t += blockDim.x) {
      if (s_n[t]) {
        unsafeAtomicAdd(&sum[t], s_sum[t]);
        atomicAdd(&count[t], (unsigned long long)s_n[t]);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// The planes' inverse transforms for power-of-two grids, the sum over planes
// fused into the column pass.
//
// A transform of N = 2^L points is Stockham radix-8 passes and a last pass of
// radix N / 8^k, eight elements per thread in registers (j + s N / 8, s = 0 ..
// 7, before and after), exchanged through LDS between passes; N / 8 threads to
// a line.  Rows are transformed in place (k_wst_rows).  The column pass
// (k_wst_cols_add) holds a tile of columns, walks the planes, and leaves
// each plane's transform in registers, where the Fresnel phase is applied and
// the sum kept in FP64: the transformed planes never go back to memory.
// Memory traffic is one read and one write of the stack for the rows and
// one read for the columns, against four of each (two transposes), a copy
// and k_wstack_add's read.  Twiddles come from an FP64-rounded table in LDS, so
// rounding matches a plain FP32 FFT.
//
// wstack2048 (65 planes): 957 + 1384 us, where the library transform, its
// input copy and k_wstack_add took 4.67 ms.  The rows are bound by that traffic
// (4.56 TB/s, a large copy 4.79); the columns move 1.86 TB/s and issue VALU
// instructions for 614 us, the rest exposed between the barriers of the one
// workgroup per compute unit.
template <int L>
struct WstFft {
  static constexpr int N = 1 << L;
  static constexpr int T = N / 8;               // threads per line
  static constexpr int FULL = (L - 1) / 3;      // radix-8 passes before the last
  static constexpr int NS = 1 << (3 * FULL);    // points already combined
  static constexpr int RL = N / NS;             // last radix: 2, 4 or 8
  static_assert(RL == 2 || RL == 4 || RL == 8, "last radix");
};

// v[r] twiddled by W_N^(e r), r = 1 .. R - 1 (inverse sign).
template <int R>
__device__ __forceinline__ void wst_twiddle(float2 *v, int stride, const float2 *tw, int e) {
#pragma unroll
  for (int r = 1; r < R; r++) v[r * stride] = cmul(v[r * stride], tw[e * r]);
}

// One line's transform: v holds elements j + s N / 8 and receives the
// outputs of the same indices.  at(i) is the LDS slot of element i; barriers
// are the workgroup's (every thread takes part).
template <int L, class At>
__device__ __forceinline__ void wst_line(float2 (&v)[8], int j, float2 *lds, const float2 *tw,
                                         At at) {
  using F = WstFft<L>;
  constexpr float sgn = 1.0f;
  int ns = 1;
#pragma unroll
  for (int p = 0; p < F::FULL; p++) {
    const int k = j & (ns - 1);
    if (p) wst_twiddle<8>(v, 1, tw, k * (F::N / (8 * ns)));
    fft_reg<8>(v, sgn);
    const int d = (j - k) * 8 + k;
    __syncthreads();  // the previous pass's reads are done
#pragma unroll
    for (int r = 0; r < 8; r++) lds[at(d + r * ns)] = v[r];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < 8; s++) v[s] = lds[at(j + s * F::T)];
    ns *= 8;
  }
  // last pass: outputs fall on the elements read
  constexpr int U = 8 / F::RL;
#pragma unroll
  for (int u = 0; u < U; u++) {
    wst_twiddle<F::RL>(v + u, U, tw, j + u * F::T);
    if constexpr (F::RL == 8) {
      fft_reg<8>(v, sgn);
    } else if constexpr (F::RL == 4) {
      fft_reg4(v[u], v[u + U], v[u + 2 * U], v[u + 3 * U], sgn);
    } else {
      const float2 a = v[u], b = v[u + U];
      v[u] = cadd(a, b);
      v[u + U] = csub(a, b);
    }
  }
}

__global__ void k_wst_twiddles(int N, float2 *__restrict__ tw) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= N) return;
  double s, c;
  sincospi(2.0 * (double)k / (double)N, &s, &c);
  tw[k] = make_float2((float)c, (float)s);
}

// Rows in place: persistent workgroups, 4096 / N rows (512 threads) at a
// time, the next rows loaded during the current ones' passes.
constexpr int WST_ROW_NT = 512;
template <int L>
__global__ __launch_bounds__(WST_ROW_NT) void k_wst_rows(float2 *__restrict__ stack,
                                                        int64_t nrows,
                                                        const float2 *__restrict__ twg) {
  using F = WstFft<L>;
  constexpr int LINES = WST_ROW_NT / F::T;
  __shared__ float2 lds[LINES * F::N + LINES * F::N / 32];
  __shared__ float2 tw[F::N];
  const int tid = threadIdx.x, line = tid / F::T, j = tid % F::T;
  for (int k = tid; k < F::N; k += WST_ROW_NT) tw[k] = twg[k];
  auto at = [&](int i) {
    const int e = line * F::N + i;
    return e + (e >> 5);
  };
  const int64_t ngroups = nrows / LINES;  // N is a multiple of LINES
  float2 nxt[8];
  int64_t g = blockIdx.x;
  auto load = [&](int64_t q) {
    const float2 *row = stack + (q * LINES + line) * F::N + j;
#pragma unroll
    for (int s = 0; s < 8; s++) nxt[s] = row[s * F::T];
  };
  if (g < ngroups) load(g);
  __syncthreads();  // table written
  for (; g < ngroups; g += gridDim.x) {
    float2 v[8];
#pragma unroll
    for (int s = 0; s < 8; s++) v[s] = nxt[s];
    if (g + gridDim.x < ngroups) load(g + gridDim.x);
    wst_line<L>(v, j, lds, tw, at);
    float2 *row = stack + (g * LINES + line) * F::N + j;
#pragma unroll
    for (int s = 0; s < 8; s++) row[s * F::T] = v[s];
  }
}

// Columns of every plane and the phase-weighted sum: image[y][x] += sign
// sum_p column transform of plane p at (y, x) times exp(-2 pi i midw[p] n1),
// as k_wstack_add.  8192 / N columns (1024 threads) per workgroup and the
// planes [p0, p1) of its plane group (blockIdx.y); workgroups of one XCD take
// neighbouring columns, which share cache lines.  With one plane group the sum
// is added without atomics.
constexpr int WST_COL_NT = 1024;
template <int L>
__global__ __launch_bounds__(WST_COL_NT) void k_wst_cols_add(
    double2 *__restrict__ image, const float2 *__restrict__ stack, int P, double theta,
    const double *__restrict__ midw, const float2 *__restrict__ twg) {
#pragma clang fp contract(off)
  using F = WstFft<L>;
  constexpr int TC = WST_COL_NT / F::T;  // columns of the tile
  constexpr int E = TC * F::N;
  __shared__ float2 lds[E + E / 8];
  __shared__ float2 tw[F::N];
  const int tid = threadIdx.x, c = tid % TC, j = tid / TC;
  for (int k = tid; k < F::N; k += WST_COL_NT) tw[k] = twg[k];
  constexpr int TILES = F::N / TC;
  const int b = blockIdx.x;
  const int tile = TILES % XCD_QUEUES == 0 ? (b % XCD_QUEUES) * (TILES / XCD_QUEUES) + b / XCD_QUEUES
                                           : b;
  const int x = tile * TC + c;
  const int p0 = (int)((int64_t)P * blockIdx.y / gridDim.y);
  const int p1 = (int)((int64_t)P * (blockIdx.y + 1) / gridDim.y);
  auto at = [&](int i) {
    const int e = i * TC + c;
    return e + 4 * (e >> 5);
  };
  const int64_t NN = (int64_t)F::N * F::N;
  const double l = theta * ((double)(x - F::N / 2) / (double)F::N);
  double n1[8];
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int y = j + s * F::T;
    const double m = theta * ((double)(y - F::N / 2) / (double)F::N);
    n1[s] = 1.0 - sqrt(1.0 - (l * l + m * m));
  }
  double ax[8], ay[8];
#pragma unroll
  for (int s = 0; s < 8; s++) ax[s] = ay[s] = 0.0;
  float2 nxt[8];
  auto load = [&](int p) {
    const float2 *col = stack + p * NN + (int64_t)j * F::N + x;
#pragma unroll
    for (int s = 0; s < 8; s++) nxt[s] = col[(int64_t)s * F::T * F::N];
  };
  if (p0 < p1) load(p0);
  __syncthreads();  // table written
  for (int p = p0; p < p1; p++) {
    float2 v[8];
#pragma unroll
    for (int s = 0; s < 8; s++) v[s] = nxt[s];
    if (p + 1 < p1) load(p + 1);
    wst_line<L>(v, j, lds, tw, at);
    const double mw = midw[p];
#pragma unroll
    for (int s = 0; s < 8; s++) {
      // turns reduced in FP64, then k_wstack_add's sincospif (the hardware sine
      // and cosine, 1.24e-7 off, would save 2 % of wstack2048); products and
      // sum in FP64
      const double t = mw * n1[s];
      float c, d;
      sincospif((float)(2.0 * (t - rint(t))), &d, &c);
      const double cs = (double)c, sn = (double)d;
      const double vx = (double)v[s].x, vy = (double)v[s].y;
      ax[s] = fma(vx, cs, fma(vy, sn, ax[s]));
      ay[s] = fma(vy, cs, fma(-vx, sn, ay[s]));
    }
  }
#pragma unroll
  for (int s = 0; s < 8; s++) {
    const int y = j + s * F::T;
    const double sg = ((x + y) & 1) ? -1.0 : 1.0;
    double2 *o = image + (int64_t)y * F::N + x;
    if (gridDim.y == 1) {
      const double2 i = *o;
      *o = make_double2(i.x + sg * ax[s], i.y + sg * ay[s]);
    } else {
      unsafeAtomicAdd(&o->x, sg * ax[s]);
      unsafeAtomicAdd(&o->y, sg * ay[s]);
    }
  }
}

template <int L>
void wst_image(croc_ctx *ctx, double2 *image, float2 *stack, int P, double theta,
               const double *midw, float2 *tw) {
  constexpr int N = 1 << L;
  hipStream_t s = ctx->stream;
  k_wst_twiddles<<<(N + 255) / 256, 256, 0, s>>>(N, tw);
  const int64_t nrows = (int64_t)P * N, groups = nrows * N / (8 * WST_ROW_NT);
  k_wst_rows<L><<<(unsigned)std::min<int64_t>(groups, 3 * (int64_t)ctx->num_cu), WST_ROW_NT, 0,
                  s>>>(stack, nrows, tw);
  // plane groups where the columns alone would not fill the chip
  const int tiles = N / (8 * WST_COL_NT / N);
  const int ng = std::max(1, std::min(P, 2 * ctx->num_cu / tiles));
  k_wst_cols_add<L><<<dim3((unsigned)tiles, (unsigned)ng), WST_COL_NT, 0, s>>>(
      image, stack, P, theta, midw, tw);
}

}  // namespace

extern "C" int croc_wstack_image(croc_ctx *ctx, void *image, void *stack, int P, int N,
                                 double theta, const double *midw) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(image && stack && midw && P >= 1 && theta > 0, CROC_EINVAL, "bad arguments");
  CROC_REQUIRE(N == 256 || N == 512 || N == 1024 || N == 2048, CROC_EINVAL,
               "N must be 256, 512, 1024 or 2048");
  const double c = theta * ((double)(0 - N / 2) / (double)N);
  CROC_REQUIRE(c * c + c * c < 1.0, CROC_EDOMAIN, "Error in image coordinate system");
  float2 *tw = (float2 *)ws_get(ctx, WS_TMP, sizeof(float2) * N);
  if (!tw) return CROC_ENOMEM;
  double2 *im = (double2 *)image;
  float2 *st = (float2 *)stack;
  if (N == 256)
    wst_image<8>(ctx, im, st, P, theta, midw, tw);
  else if (N == 512)
    wst_image<9>(ctx, im, st, P, theta, midw, tw);
  else if (N == 1024)
    wst_image<10>(ctx, im, st, P, theta, midw, tw);
  else
    wst_image<11>(ctx, im, st, P, theta, midw, tw);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}

extern "C" int croc_w_bins(croc_ctx *ctx, const double *w, int64_t nv, int64_t stride,
                           double wstep, int64_t *bin) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(nv >= 0 && stride >= 1, CROC_EINVAL, "bad arguments");
  if (nv == 0) return CROC_OK;
  CROC_REQUIRE(w && bin, CROC_EINVAL, "null array");
  const unsigned nb = (unsigned)std::min<int64_t>((nv + 255) / 256, 1 << 20);
  k_w_bins<<<nb, 256, 0, ctx->stream>>>(w, nv, stride, wstep, bin);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}

extern "C" int croc_wplane_sums(croc_ctx *ctx, const double *uvw, int64_t nv, int64_t stride,
                                double wstep, int64_t plane0, int ntab, int64_t *count,
                                double *sum) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(nv >= 0 && stride >= 3 && wstep != 0 && ntab >= 1, CROC_EINVAL,
               "bad arguments");
  CROC_REQUIRE(count && sum && (nv == 0 || uvw), CROC_EINVAL, "null array");
  if ((rc = zero_u32_async(ctx, (uint32_t *)count, 2 * (int64_t)ntab))) return rc;
  if ((rc = zero_u32_async(ctx, (uint32_t *)sum, 2 * (int64_t)ntab))) return rc;
  if (nv == 0) return CROC_OK;
  uint32_t *st;
  if ((rc = small_status(ctx, &st))) return rc;
  const unsigned nb = (unsigned)std::min<int64_t>((nv + 511) / 512, 2 * (int64_t)ctx->num_cu);
  if (ntab <= PLANES_LDS)
    k_wplane_sums<true><<<nb, 512, 0, ctx->stream>>>(
        uvw, nv, stride, wstep, plane0, ntab, (unsigned long long *)count, sum, st);
  else
    k_wplane_sums<false><<<nb, 512, 0, ctx->stream>>>(
        uvw, nv, stride, wstep, plane0, ntab, (unsigned long long *)count, sum, st);
  CROC_HIP(hipGetLastError());
  return finish_status(ctx, st);
}

extern "C" int croc_wstack_grid(croc_ctx *ctx, void *stack, int P, int N,
                                const double *uvw, int64_t nv, int64_t stride,
                                double lam, double wstep, int64_t plane0,
                                int ntab, const int32_t *slot_of,
                                const void *vis, int centred) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(N >= 1 && P >= 1 && stride >= 3 && lam > 0 && wstep > 0 && ntab >= 1,
               CROC_EINVAL, "bad arguments");
  CROC_REQUIRE(!centred || N % 2 == 0, CROC_EINVAL,
               "the folded centring sign needs an even grid");
  CROC_REQUIRE((int64_t)P * N * N < ((int64_t)1 << 46), CROC_EINVAL, "stack too large");
  if (nv == 0) return CROC_OK;
  CROC_REQUIRE(stack && uvw && vis && slot_of, CROC_EINVAL, "null array");
  uint32_t *st;
  if ((rc = small_status(ctx, &st))) return rc;
  const unsigned nb = (unsigned)((nv + 255) / 256);
  // Validate everything first so that an error leaves the stack untouched.
  k_wstack_grid<<<nb, 256, 0, ctx->stream>>>((float2 *)stack, N, uvw, nv, stride, lam,
                                             wstep, plane0, ntab, slot_of,
                                             (const float2 *)vis, centred, 0, st);
  CROC_HIP(hipGetLastError());
  if ((rc = finish_status(ctx, st))) return rc;
  k_wstack_grid<<<nb, 256, 0, ctx->stream>>>((float2 *)stack, N, uvw, nv, stride, lam,
                                             wstep, plane0, ntab, slot_of,
                                             (const float2 *)vis, centred, 1, st);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}

extern "C" int croc_wstack_add(croc_ctx *ctx, void *image, const void *stack, int P,
                               int N, double theta, const double *midw, int centred) {
  int rc = ctx_enter(ctx);
  if (rc) return rc;
  CROC_REQUIRE(image && stack && midw && N >= 1 && P >= 1 && theta > 0, CROC_EINVAL,
               "bad arguments");
  CROC_REQUIRE(!centred || N % 2 == 0, CROC_EINVAL,
               "the folded centring sign needs an even grid");
  // synthesis.py:290: the corner of the image (the most negative l and m)
  // must lie inside the unit circle.
  const double c = theta * ((double)(0 - N / 2) / (double)N);
  CROC_REQUIRE(c * c + c * c < 1.0, CROC_EDOMAIN, "Error in image coordinate system");
  const int64_t NN = (int64_t)N * N;
  k_wstack_add<<<(unsigned)((NN + 255) / 256), 256, 0, ctx->stream>>>(
      (double2 *)image, (const float2 *)stack, P, N, theta, midw, centred);
  CROC_HIP(hipGetLastError());
  return CROC_OK;
}
