// The 128-point building blocks of the batched 128 x 128 sub-grid FFT
// (fft.hip) shared with the kernels that transform a sub-grid in LDS and
// use it there (the w-towers predict).  Each 1D transform of 128 points is
// split as 128 = 16 x 8 (j = 8 j1 + j2, k = k1 + 16 k2):
//   pass A: for each j2, a 16-point DFT over j1 in registers, times the
//           twiddle W128^(j2 k1), written back in place;
//   pass B: for each k1, an 8-point DFT over j2 in registers, written to
//           the natural position k1 + 16 k2.
// LDS rows are padded to FP = 129 elements so that row- and column-wise
// accesses spread over the banks.
#pragma once

#include "internal.h"

namespace {

constexpr int FN = 128;
constexpr int FP = FN + 1;  // padded LDS row
constexpr int FFT_NT = 1024;
constexpr int PASS_A = FN * 8 / FFT_NT;   // pass-A items (line, j2) per thread
constexpr int PASS_B = FN * 16 / FFT_NT;  // pass-B items (line, k1) per thread
static_assert(PASS_A * FFT_NT == FN * 8 && PASS_B * FFT_NT == FN * 16, "item split");

struct FModArgs {
  const double *phi;
  const int32_t *kplane;
  int sign;
};

// v * exp(i kf phi), kf = s k (the plane multiplier times the sign): the
// angle in turns, reduced to [-1/2, 1/2] in FP64, then the hardware sine
// and cosine of turns (v_sin_f32 / v_cos_f32: 1.24e-7 largest absolute
// error on [-1/2, 1/2], measured against FP64 over 2^20 points; a library
// sincosf of the FP32 angle in radians is 2.1e-7 there and several times
// the instructions).
__device__ __forceinline__ float2 rotation(double kf, double phi) {  // {cos, sin}
  const double t = kf * phi * 0.15915494309189535;
  const float f = (float)(t - rint(t));
  const float s = __builtin_amdgcn_sinf(f), c = __builtin_amdgcn_cosf(f);
  return make_float2(c, s);
}
__device__ __forceinline__ float2 rotate_by(float2 v, float2 r) {
  return make_float2(v.x * r.x - v.y * r.y, v.x * r.y + v.y * r.x);
}
__device__ __forceinline__ float2 rotate(float2 v, double kf, double phi) {
  return rotate_by(v, rotation(kf, phi));
}

// The rotations of one w-plane, each taken once: phi depends on the pixel's
// distances u, w from the middle row and column only, and not on their order
// (to the bit: its l^2 + m^2 is formed symmetrically), so 2145 of the 16384
// pixels' rotations differ.  Entry (hi, lo) = (max, min)(u, w), 0 <= lo <= hi
// <= 64, sits at |hi - 32| ROT_P + (hi > 32 ? lo : 66 - lo): rows hi and
// 64 - hi share a line, and with the odd pitch a half-wavefront along a row or
// a column of pixels takes 1.6 passes over the banks on average.
constexpr int ROT_P = 67;
constexpr int ROT_N = 33 * ROT_P;

__device__ __forceinline__ int rot_index(int y, int x) {
  const int u = abs(x - FN / 2), w = abs(y - FN / 2);
  const int hi = max(u, w), lo = min(u, w);
  return abs(hi - 32) * ROT_P + (hi > 32 ? lo : 66 - lo);
}

// rot[e] = rotation(kf, phic[e]), by the whole workgroup; phic in the layout
// above.
__device__ __forceinline__ void rot_table(float2 *rot, const double *__restrict__ phic,
                                          double kf) {
  for (int e = threadIdx.x; e < ROT_N; e += FFT_NT) rot[e] = rotation(kf, phic[e]);
}

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }

// v sqrt(1/2) (1 + s i) and v sqrt(1/2) (-1 + s i): the odd eighths of a turn.
__device__ __forceinline__ float2 rot45(float2 v, float s) {
  constexpr float H = 0.70710678118654757f;
  return make_float2(H * fmaf(-s, v.y, v.x), H * fmaf(s, v.x, v.y));
}
__device__ __forceinline__ float2 rot135(float2 v, float s) {
  constexpr float H = 0.70710678118654757f;
  return make_float2(-H * fmaf(s, v.y, v.x), H * fmaf(s, v.x, -v.y));
}

// Four-point DFT in place, W_4 = s i (s = sgn).
__device__ __forceinline__ void fft_reg4(float2 &a, float2 &b, float2 &c, float2 &d, float s) {
  const float2 p = cadd(a, c), q = csub(a, c), r = cadd(b, d), t = csub(b, d);
  a = cadd(p, r);
  c = csub(p, r);
  b = make_float2(fmaf(-s, t.y, q.x), fmaf(s, t.x, q.y));
  d = make_float2(fmaf(s, t.y, q.x), fmaf(-s, t.x, q.y));
}

// In-register DFT of N = 8 or 16 points: v[k] = sum_j v[j] W_N^(jk), W_N =
// exp(sgn 2 pi i / N).  Radix 4 (8 = 2 x 4, 16 = 4 x 4) with the quarter and
// eighth turns written out: 56 and 162 instructions, where a radix-2 recursion
// that multiplies by every twiddle takes 96 and 256.
template <int N>
__device__ __forceinline__ void fft_reg(float2 *v, float sgn) {
  static_assert(N == 8 || N == 16, "8 or 16 points");
  if constexpr (N == 8) {
    float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    fft_reg4(e0, e1, e2, e3, sgn);
    fft_reg4(o0, o1, o2, o3, sgn);
    o1 = rot45(o1, sgn);
    o2 = make_float2(-sgn * o2.y, sgn * o2.x);
    o3 = rot135(o3, sgn);
    v[0] = cadd(e0, o0);
    v[4] = csub(e0, o0);
    v[1] = cadd(e1, o1);
    v[5] = csub(e1, o1);
    v[2] = cadd(e2, o2);
    v[6] = csub(e2, o2);
    v[3] = cadd(e3, o3);
    v[7] = csub(e3, o3);
  } else {
    // cos, sin of an eighth of pi
    constexpr float C = 0.92387953251128674f, S = 0.38268343236508978f;
    // column b holds elements 4 a + b; after its DFT entry k1 takes W16^(b k1)
#pragma unroll
    for (int b = 0; b < 4; b++) fft_reg4(v[b], v[4 + b], v[8 + b], v[12 + b], sgn);
    v[5] = cmul(v[5], make_float2(C, sgn * S));
    v[9] = rot45(v[9], sgn);
    v[13] = cmul(v[13], make_float2(S, sgn * C));
    v[6] = rot45(v[6], sgn);
    v[10] = make_float2(-sgn * v[10].y, sgn * v[10].x);
    v[14] = rot135(v[14], sgn);
    v[7] = cmul(v[7], make_float2(S, sgn * C));
    v[11] = rot135(v[11], sgn);
    v[15] = cmul(v[15], make_float2(-C, -sgn * S));
    // row k1 (v[4 k1 ..]) gives outputs k1 + 4 k2
#pragma unroll
    for (int k = 0; k < 4; k++) fft_reg4(v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3], sgn);
    // transpose to natural order
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = i + 1; j < 4; j++) {
        const float2 t = v[4 * i + j];
        v[4 * i + j] = v[4 * j + i];
        v[4 * j + i] = t;
      }
  }
}

// Column passes of all 128 columns of a sub-grid in LDS (element (y, x) at
// y FP + x), consecutive lanes on consecutive columns (consecutive
// addresses: distinct banks).  Pass A on items (column x, j2), in place;
// tw[m] = W128^m.
__device__ __forceinline__ void cols_pass_a(float2 *lds, const float2 *tw, float sgn) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int r = 0; r < PASS_A; r++) {
    const int it = tid + r * FFT_NT;
    const int x = it & 127, j2 = it >> 7;
    float2 *p = lds + x + j2 * FP;
    float2 v[16];
#pragma unroll
    for (int j1 = 0; j1 < 16; j1++) v[j1] = p[8 * j1 * FP];
    fft_reg<16>(v, sgn);
#pragma unroll
    for (int k1 = 0; k1 < 16; k1++) {
      const float2 w = tw[(j2 * k1) & 127];
      p[8 * k1 * FP] = cmul(v[k1], make_float2(w.x, sgn * w.y));
    }
  }
}

// Column pass-B item r of the thread: (column x, k1).
__device__ __forceinline__ void cols_pass_b_item(int r, int &x, int &k1) {
  const int it = threadIdx.x + r * FFT_NT;
  x = it & 127;
  k1 = it >> 7;
}

// Column pass B on items (x, k1): v[r][k2] = output row k1 + 16 k2 of the
// thread's r-th column, read from LDS; the caller stores it.
__device__ __forceinline__ void cols_pass_b(const float2 *lds, float sgn,
                                            float2 (&v)[PASS_B][8]) {
#pragma unroll
  for (int r = 0; r < PASS_B; r++) {
    int x, k1;
    cols_pass_b_item(r, x, k1);
    const float2 *p = lds + x + 8 * k1 * FP;
#pragma unroll
    for (int j2 = 0; j2 < 8; j2++) v[r][j2] = p[j2 * FP];
    fft_reg<8>(v[r], sgn);
  }
}

// Row passes over the rows rows[0 .. nrows - 1] (rows == nullptr: row k
// is k) of a sub-grid in LDS, with 32 consecutive lanes on 32 rows at the
// same element offset: with the odd pitch FP they fall on distinct banks
// (a lane per row segment, 8 lanes to a row, puts 16 lanes of a pass-B
// read on 4 banks).  Items of pass A: (k, j2), k = 32 (t >> 8) +
// (t & 31), j2 = (t >> 5) & 7; of pass B: (k, k1) for it = t + r FFT_NT,
// k = 32 (it >> 9) + (it & 31), k1 = (it >> 5) & 15.  Wavefronts whose 32
// rows lie past nrows skip as a whole.
__device__ __forceinline__ int rowlist_line(const int *rows, int k) { return rows ? rows[k] : k; }

__device__ __forceinline__ void rows_pass_a(float2 *lds, const int *rows, int nrows,
                                            const float2 *tw, float sgn) {
  const int t = threadIdx.x;
  const int k = 32 * (t >> 8) + (t & 31), j2 = (t >> 5) & 7;
  if (__builtin_amdgcn_readfirstlane(32 * (t >> 8)) >= nrows || k >= nrows) return;
  float2 *p = lds + rowlist_line(rows, k) * FP + j2;
  float2 v[16];
#pragma unroll
  for (int j1 = 0; j1 < 16; j1++) v[j1] = p[8 * j1];
  fft_reg<16>(v, sgn);
#pragma unroll
  for (int k1 = 0; k1 < 16; k1++) {
    const float2 w = tw[(j2 * k1) & 127];
    p[8 * k1] = cmul(v[k1], make_float2(w.x, sgn * w.y));
  }
}

// Pass B item r of the thread: list entry k and k1 (k past nrows: none).
__device__ __forceinline__ void rows_pass_b_item(int r, int &k, int &k1) {
  const int it = threadIdx.x + r * FFT_NT;
  k = 32 * (it >> 9) + (it & 31);
  k1 = (it >> 5) & 15;
}

// Pass B reads: v[r][k2] = output k1 + 16 k2 of the thread's r-th item
// (zeros for wavefronts past the list); the caller writes them back after a
// barrier.
__device__ __forceinline__ void rows_pass_b(const float2 *lds, const int *rows, int nrows,
                                            float sgn, float2 (&v)[PASS_B][8]) {
#pragma unroll
  for (int r = 0; r < PASS_B; r++) {
    int k, k1;
    rows_pass_b_item(r, k, k1);
    const int kw = __builtin_amdgcn_readfirstlane(32 * ((threadIdx.x + r * FFT_NT) >> 9));
    if (kw < nrows) {
      const float2 *p = lds + rowlist_line(rows, min(k, nrows - 1)) * FP + 8 * k1;
#pragma unroll
      for (int j2 = 0; j2 < 8; j2++) v[r][j2] = p[j2];
      fft_reg<8>(v[r], sgn);
    } else {
#pragma unroll
      for (int j2 = 0; j2 < 8; j2++) v[r][j2] = make_float2(0.f, 0.f);
    }
  }
}

// W128^m = exp(2 pi i m / 128), m = 0..127, rounded from FP64 (the caller
// applies the sign of the transform to the imaginary part).
__device__ __forceinline__ void fft128_twiddles(float2 *tw) {
  if (threadIdx.x < FN) {
    double s, c;
    sincospi((double)threadIdx.x / 64.0, &s, &c);
    tw[threadIdx.x] = make_float2((float)c, (float)s);
  }
}

}  // namespace
