// Direct gridding and degridding of small one-shot calls: crocodile/
// synthesis.py:464-503 without binning.
//
// croc_convgrid and croc_convdegrid bin their visibilities by tile so that
// the taps land in LDS.  For a few thousand visibilities the binning's ten
// launches, and not the taps, are the call's time.  Here one wavefront takes
// a few visibilities at a time, locates them (locate.h) and walks their taps
// straight over the grid (gridding: over the int64 accumulator), three
// launches for gridding and two for degridding, one host wait.  The tap
// walks, the fixed-point scale and, in degridding, every lane's order of
// summation are the tile kernels', so the results are theirs bit for bit.
//
// The status word is zero between calls (cleared again after an error), so
// no launch clears it; the last kernel of a call writes status and flags to
// pinned host memory, so no copy fetches them.
#include <algorithm>

#include "locate.h"
#include "taps.h"

namespace {

constexpr int DIR_NT = 256;
constexpr int DIR_WAVES = DIR_NT / 64;
constexpr int DIR_PARTS = 256;  // blocks of the maxima pass
constexpr int DIR_WAVES_CU = 32;  // wavefronts per compute unit a launch aims at

struct DirectState {
  uint32_t status;  // zero between calls
  uint32_t pad[3];
  double inv_scale;
  // per block of the maxima pass: max |re|, |im| of the visibilities and of
  // the kernel bank (float bits), non-finite flags
  uint32_t vmax[DIR_PARTS], kmax[DIR_PARTS], flags[DIR_PARTS];
  uint32_t nonfinite;  // their union, for k_grid_nonfinite
};

// Largest of the block's values in every thread (blockDim DIR_NT).
__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t *s) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, off, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  v = s[0];
#pragma unroll
  for (int w = 1; w < DIR_WAVES; w++) v = max(v, s[w]);
  return v;
}

// Accumulator cleared, and the block's maxima of the finite visibility and
// kernel components (non-negative floats order like their bits).
__global__ __launch_bounds__(DIR_NT) void k_direct_prep(
    ulonglong2 *__restrict__ acc, int64_t cells, const float2 *__restrict__ vis, int64_t nv,
    const float2 *__restrict__ kern, const int64_t *__restrict__ plane_off,
    const int32_t *__restrict__ plane_s, int nplanes, int Q, int separable,
    DirectState *__restrict__ st) {
  __shared__ unsigned long long s_ext;
  __shared__ uint32_t s[DIR_WAVES];
  const int64_t stride = (int64_t)gridDim.x * DIR_NT;
  const int64_t i0 = (int64_t)blockIdx.x * DIR_NT + threadIdx.x;
  for (int64_t i = i0; i < cells; i += stride) acc[i] = make_ulonglong2(0ull, 0ull);
  const int64_t nk = bank_extent(plane_off, plane_s, nplanes, Q, separable, &s_ext);
  bool bv = false, bk = false;
  const float mv = array_max(vis, nv, i0, stride, bv);
  const float mk = array_max(kern, nk, i0, stride, bk);
  const uint32_t v = block_max_u32(__float_as_uint(mv), s);
  const uint32_t k = block_max_u32(__float_as_uint(mk), s);
  const uint32_t f = (__syncthreads_or(bv) ? 1u : 0u) | (__syncthreads_or(bk) ? 2u : 0u);
  if (threadIdx.x == 0) {
    st->vmax[blockIdx.x] = v;
    st->kmax[blockIdx.x] = k;
    st->flags[blockIdx.x] = f;
  }
}

// The wavefront's `per` visibilities located, one per lane; records kept for
// the marking of non-finite cells (gridding) or the degridding pass.
__device__ __forceinline__ uint4 direct_locate(const BinArgs &a, int per, int64_t *first, int *n,
                                               uint4 *__restrict__ rec, uint32_t *status) {
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * DIR_WAVES +
                    __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  *first = w * per;
  *n = (int)max((int64_t)0, min((int64_t)per, a.nv - *first));
  uint4 r = make_uint4(0u, 0u, 0u, LOC_INVALID);
  if (lane < *n) {
    const BinGeom g{a.N, 1, 1, 1};  // one tile, one group
    uint32_t st = 0;
    r = locate(a, g, *first + lane, &st);
    if (st) atomicOr(status, st);
    // an invalid visibility (the call fails) leaves an empty window
    if (r.w == LOC_INVALID) r = make_uint4(0u, 0u, 0u, LOC_INVALID);
    rec[*first + lane] = make_uint4(r.x, r.y, r.z, (uint32_t)(*first + lane));
  }
  return r;
}

template <bool SEPARABLE>
__global__ __launch_bounds__(DIR_NT) void k_direct_grid(
    BinArgs a, int per, unsigned long long *__restrict__ acc, const float2 *__restrict__ vis,
    const float2 *__restrict__ kern, int nparts, uint4 *__restrict__ rec,
    DirectState *__restrict__ st) {
  __shared__ uint32_t s[DIR_WAVES];
  const int t = threadIdx.x, lane = t & 63;
  const uint32_t v = block_max_u32(t < nparts ? st->vmax[t] : 0u, s);
  const uint32_t k = block_max_u32(t < nparts ? st->kmax[t] : 0u, s);
  const int e = fixed_exponent(__uint_as_float(v), __uint_as_float(k), a.nv, SEPARABLE);
  const double scale = ldexp(1.0, e);
  if (blockIdx.x == 0 && t == 0) st->inv_scale = ldexp(1.0, -e);
  int64_t first;
  int n;
  const uint4 rl = direct_locate(a, per, &first, &n, rec, &st->status);
  const float2 vl = lane < n ? vis[first + lane] : make_float2(0.f, 0.f);
  for (int it = 0; it < n; it++) {
    const uint4 r = lane_u4(rl, it);
    if (r.w == LOC_INVALID) continue;
    const float2 x = lane_f2(vl, it);
    const int S = (int)(r.y & 0xffu);
    const int xf = (int)((r.y >> 8) & 0xfffu), yf = (int)(r.y >> 20);
    const float2 *kp = kern + r.z, *ky = kp + yf * S, *kx = kp + xf * S;
    unsigned long long *cell = acc + 2 * ((int64_t)(r.x >> 16) * a.N + (int64_t)(r.x & 0xffffu));
    spread_range<SEPARABLE>(cell, 0, a.N, S, 0, S * S, lane, kp, ky, kx, (double)x.x * scale,
                            (double)x.y * scale);
  }
}

// grid[c] += acc[c] / 2^e unless the call failed; status and flags to the
// host words.
__global__ __launch_bounds__(DIR_NT) void k_direct_finish(
    float2 *__restrict__ grid, const longlong2 *__restrict__ acc, int64_t cells, int nparts,
    DirectState *__restrict__ st, uint32_t *__restrict__ host, float sign) {
  __shared__ uint32_t s[DIR_WAVES];
  const uint32_t status = st->status;
  if (blockIdx.x == 0) {
    uint32_t f = 0u;  // two one-bit flags: their union by two maxima
    const uint32_t mine = (int)threadIdx.x < nparts ? st->flags[threadIdx.x] : 0u;
    f = block_max_u32(mine & 1u, s) | block_max_u32(mine & 2u, s);
    if (threadIdx.x == 0) {
      st->nonfinite = f;
      __hip_atomic_store(host, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(host + 1, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
  if (status) return;
  const double inv = st->inv_scale;
  const int64_t stride = (int64_t)gridDim.x * DIR_NT;
  for (int64_t i = (int64_t)blockIdx.x * DIR_NT + threadIdx.x; i < cells; i += stride) {
    const longlong2 c = acc[i];
    if (c.x | c.y) {
      float2 g = grid[i];
      g.x += (float)((double)c.x * inv);
      g.y = sign * (sign * g.y + (float)((double)c.y * inv));
      grid[i] = g;
    }
  }
}

__global__ __launch_bounds__(DIR_NT) void k_direct_locate(BinArgs a, uint4 *__restrict__ rec,
                                                         DirectState *__restrict__ st) {
  int64_t first;
  int n;
  direct_locate(a, 64, &first, &n, rec, &st->status);
}

template <bool SEPARABLE>
__global__ __launch_bounds__(DIR_NT) void k_direct_degrid(
    int64_t nv, int N, int per, const uint4 *__restrict__ rec,
    const float2 *__restrict__ grid, const float2 *__restrict__ kern,
    float2 *__restrict__ vis_out, const DirectState *__restrict__ st,
    uint32_t *__restrict__ host) {
  const int lane = threadIdx.x & 63;
  const uint32_t status = st->status;
  if (blockIdx.x == 0 && threadIdx.x == 0)
    __hip_atomic_store(host, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  if (status) return;
  const int64_t first = ((int64_t)blockIdx.x * DIR_WAVES +
                         __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) *
                        per;
  const int n = (int)max((int64_t)0, min((int64_t)per, nv - first));
  const uint4 rl = lane < n ? rec[first + lane] : make_uint4(0u, 0u, 0u, 0u);
  float2 res = make_float2(0.f, 0.f);
  for (int it = 0; it < n; it++) {
    const uint4 r = lane_u4(rl, it);
    const int S = (int)(r.y & 0xffu);
    const int xf = (int)((r.y >> 8) & 0xfffu), yf = (int)(r.y >> 20);
    const float2 *kp = kern + r.z, *ky = kp + yf * S, *kx = kp + xf * S;
    const float2 *cell = grid + (int64_t)(r.x >> 16) * N + (int64_t)(r.x & 0xffffu);
    float ar = 0.f, ai = 0.f;
    gather_range<SEPARABLE, false>(cell, 0, N, S, 0, S * S, lane, kp, ky, kx, ar, ai);
    ar = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wave_sum_to_63(ar)), 63));
    ai = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wave_sum_to_63(ai)), 63));
    if (lane == it) res = make_float2(ar, ai);
  }
  if (lane < n) vis_out[first + lane] = res;
}

// Visibilities per wavefront: as few as still fill the chip.
int per_wave(croc_ctx *ctx, int64_t nv) {
  const int64_t waves = (int64_t)ctx->num_cu * DIR_WAVES_CU;
  return (int)std::min<int64_t>(64, std::max<int64_t>(1, (nv + waves - 1) / waves));
}

unsigned blocks_of(int64_t nv, int per) {
  const int64_t waves = (nv + per - 1) / per;
  return (unsigned)((waves + DIR_WAVES - 1) / DIR_WAVES);
}

int direct_begin(croc_ctx *ctx, const BinArgs &a, DirectState **st, uint4 **rec) {
  *st = (DirectState *)ws_get(ctx, WS_DIRECT, sizeof(DirectState));
  *rec = (uint4 *)ws_get(ctx, WS_REC, sizeof(uint4) * (size_t)a.nv);
  if (!*st || !*rec) return CROC_ENOMEM;
  if (!ctx->direct_clean) {
    int rc = zero_u32_async(ctx, &(*st)->status, 1);
    if (rc) return rc;
  }
  ctx->direct_clean = false;  // until the call's status is known to be zero
  return CROC_OK;
}

int direct_end(croc_ctx *ctx, volatile uint32_t *host) {
  CROC_HIP(hipStreamSynchronize(ctx->stream));
  const uint32_t status = host[0];
  ctx->direct_clean = status == 0;
  return croc_status_to_code(status);
}

}  // namespace

// Where the direct path is the faster one, measured per call against the tile
// path (us, direct / tile; one plane unless said otherwise).
//
// Gridding is bound by the 64-bit atomics into the accumulator, and by how many
// of them fall on one cell, which the tile path adds up in LDS: 24 ns per
// visibility (S = 8) when all share one window.  So the line is not drawn where
// spread visibilities break even (1e4 to 2e5) but where those of a core do,
// normal with a sigma of 4 cells; there nv S is about the same at every S from
// 4 to 32.  N = 256, S = 8, 5120 visibilities: spread 57 / 101, core 124 / 114,
// one window 169 / 115 (at 49152: 149 / 113, 734 / 110, 1227 / 107); N = 2048,
// S = 15, 2730: 90 / 229 with 100 planes (at 13981 with one: 157 / 199, core
// 565 / 151).  Below S = 8 the count is bounded (S = 1, 196608, core: 238 / 137).
// N = 8192 and 30000 lie on the same side (433 / 596, 5304 / 5449), and so does a
// bank of 197 MB (115 / 198).
constexpr int64_t DIRECT_GRID_ROWS = 40960;  // visibilities times max(S, 8)
//
// Degridding is bound by the visibilities (0.15 ns each up to S = 8) and then by
// L2 reads of grid and taps: taps (visibilities times S^2) set the line, twice
// as far out with kernel banks that crowd an L2 of 4 MiB, which the tile path
// reads plane group by plane group.
//   Small banks, N = 2048: S = 15, 149130 128 / 141, 298260 212 / 184; S = 32,
//     32768 86 / 151, 65536 133 / 163, 1.3e5 211 / 200; S = 8, 524288 154 / 222;
//     S = 1, 1.7e7 2472 / 3069.  N = 8192 and 30000, S = 8, 524288: 185 / 513 and
//     228 / 3654.
//   100 planes, Q = 8, N = 2048: S = 8 (3 MiB), 1048576 291 / 332; S = 15 (11
//     MiB), 298260 273 / 413; 150 planes, S = 31, 69832: 211 / 554.
constexpr int64_t DIRECT_DEGRID_TAPS = 32 << 20;
constexpr int64_t DIRECT_BANK_BYTES = 2 << 20;

bool direct_grid_wins(const BinArgs &a, int max_support) {
  return max_support >= 1 && max_support <= 64 && a.nv > 0 &&
         a.nv <= DIRECT_GRID_ROWS / std::max(max_support, 8);
}

bool direct_degrid_wins(const BinArgs &a, int max_support) {
  if (max_support < 1 || max_support > 64 || a.nv <= 0) return false;
  const int64_t row = (int64_t)a.Q * max_support;
  const double bank = 8.0 * (double)a.nplanes * (a.separable ? (double)row : (double)row * row);
  const int64_t taps = DIRECT_DEGRID_TAPS * (bank > DIRECT_BANK_BYTES ? 2 : 1);
  return a.nv <= taps / ((int64_t)max_support * max_support);
}

int direct_grid(croc_ctx *ctx, const BinArgs &a, void *grid, const void *vis, const void *kern,
                float sign) {
  const int64_t cells = (int64_t)a.N * a.N;
  ulonglong2 *acc = (ulonglong2 *)ws_get(ctx, WS_ACC, sizeof(ulonglong2) * cells);
  if (!acc) return CROC_ENOMEM;
  DirectState *st;
  uint4 *rec;
  int rc = direct_begin(ctx, a, &st, &rec);
  if (rc) return rc;
  uint32_t *host = ctx->host_status + 2;
  hipStream_t s = ctx->stream;
  const float2 *v = (const float2 *)vis, *k = (const float2 *)kern;
  k_direct_prep<<<DIR_PARTS, DIR_NT, 0, s>>>(acc, cells, v, a.nv, k, a.plane_off, a.plane_s,
                                             a.nplanes, a.Q, a.separable, st);
  const int per = per_wave(ctx, a.nv);
  const unsigned nb = blocks_of(a.nv, per);
  tap_timer_reset(ctx, 0);
  CROC_HIP(hipEventRecord(ctx->ev[0], s));
  if (a.separable)
    k_direct_grid<true><<<nb, DIR_NT, 0, s>>>(a, per, (unsigned long long *)acc, v, k, DIR_PARTS,
                                              rec, st);
  else
    k_direct_grid<false><<<nb, DIR_NT, 0, s>>>(a, per, (unsigned long long *)acc, v, k,
                                               DIR_PARTS, rec, st);
  CROC_HIP(hipEventRecord(ctx->ev[1], s));
  ctx->ev_grid = ctx->tap_is_ev[0] = true;
  k_direct_finish<<<(unsigned)std::min<int64_t>((cells + DIR_NT - 1) / DIR_NT, 8192), DIR_NT, 0,
                    s>>>((float2 *)grid, (const longlong2 *)acc, cells, DIR_PARTS, st, host,
                          sign);
  CROC_HIP(hipGetLastError());
  if ((rc = direct_end(ctx, host))) return rc;
  if (host[1])  // non-finite values: their cells, on the stream
    return grid_mark_nonfinite(ctx, grid, a.N, rec, a.nv, vis, kern, a.separable,
                               &st->nonfinite);
  return CROC_OK;
}

int direct_degrid(croc_ctx *ctx, const BinArgs &a, const void *grid, void *vis_out,
                  const void *kern) {
  DirectState *st;
  uint4 *rec;
  int rc = direct_begin(ctx, a, &st, &rec);
  if (rc) return rc;
  uint32_t *host = ctx->host_status + 2;
  hipStream_t s = ctx->stream;
  const float2 *g = (const float2 *)grid, *k = (const float2 *)kern;
  float2 *out = (float2 *)vis_out;
  k_direct_locate<<<blocks_of(a.nv, 64), DIR_NT, 0, s>>>(a, rec, st);
  const int per = per_wave(ctx, a.nv);
  const unsigned nb = blocks_of(a.nv, per);
  tap_timer_reset(ctx, 1);
  CROC_HIP(hipEventRecord(ctx->ev[2], s));
  if (a.separable)
    k_direct_degrid<true><<<nb, DIR_NT, 0, s>>>(a.nv, a.N, per, rec, g, k, out, st, host);
  else
    k_direct_degrid<false><<<nb, DIR_NT, 0, s>>>(a.nv, a.N, per, rec, g, k, out, st, host);
  CROC_HIP(hipEventRecord(ctx->ev[3], s));
  ctx->ev_degrid = ctx->tap_is_ev[1] = true;
  CROC_HIP(hipGetLastError());
  return direct_end(ctx, host);
}
