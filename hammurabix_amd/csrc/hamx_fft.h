// The LDS line-transform engine: a workgroup holds C lines of n complex128
// points in LDS and transforms them in place (forward or backward,
// unnormalised).  Used by the 3D transform (hamx_fft.hip) and by the
// random-field kernels that fuse their elementwise steps into an axis pass
// (hamx_rnd.hip).
//
// * n = 2^a 3^b 5^c 7^d <= 8192: mixed-radix Stockham autosort passes (the
//   power of two in radix 8 and 4, then 3, 5, 7).  A pass of radix R
//   stages its inputs in registers, synchronises, then writes its outputs, so
//   one LDS buffer suffices.
// * any other n <= 4096: Bluestein's algorithm.  With c_j = exp(sign i pi j^2 / n),
//   X_k = c_k sum_j (x_j c_j) conj(c_{k-j}): the line times the chirp, zero
//   padded to a power of two M >= 2n - 1, is convolved with conj(c) by an
//   M-point forward transform, a product with the transform of conj(c), and
//   an M-point inverse transform; the outputs are multiplied by the chirp
//   and 1/M.
//
// A pass over memory is bound by HBM only while the LDS passes hide behind
// it, so there are few of them: with radix 8 (and the odd radices in their
// real-factor form, fused multiply-adds throughout) the axis passes of es
// 256x256x64 took 5 to 12% less time than with radix 4 and 2, te 800x800x160's
// 12 to 20% less.
//
// Layout: point t of line c at lds[t P + c].  C is a power of two and
// consecutive threads take consecutive lines, so a pass's reads are
// contiguous runs of LDS.  A kernel whose lines are columns of memory takes
// P = C (its rows of C columns are contiguous on both sides); one whose lines
// are runs of memory takes P = C + 1, so that consecutive points of a run
// fall in different banks.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "hamx_internal.h"

namespace hamx {

constexpr uint32_t kMaxPass = 16;
constexpr uint32_t kTileMax = 8192; // complex128 values: 128 KB of LDS

struct FftPass {
  uint16_t radix, p; // p: product of the radices of the earlier passes
  uint16_t q, tstep; // n / radix and n / (radix p)
  float inv_p;
};

struct FftPlan {
  uint32_t n, npass;
  FftPass pass[kMaxPass];
};

enum FftMode { kFftPow2 = 0, kFftMixed = 1, kFftBlue = 2 };

// One line length: n points, held as len LDS points (n, or Bluestein's M),
// with the plan and twiddle table (exp(2 pi i m / len)) of len.  chirp
// (exp(i pi j^2 / n), n values) and bhat (the forward transform of
// conj(chirp) laid out circularly, len values) serve exponent +1; both are
// conjugated for exponent -1 (bhat is even because conj(chirp) is).
struct FftLine {
  uint32_t n, len;
  int mode;
  FftPlan plan;
  const double2 *tw, *chirp, *bhat;
};

// Quotients by a launch constant without the software division: exact for
// e d < 2^32, d >= 2.
struct FastDiv {
  uint32_t d, m;
};
inline FastDiv fast_div(uint32_t d) {
  return FastDiv{d, static_cast<uint32_t>((1ull << 32) / d + 1)};
}
__device__ inline uint32_t fast_quot(const FastDiv &f, uint32_t e) { return __umulhi(e, f.m); }

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
__device__ inline double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// w or conj(w): the exponent's sign applied to a table value
template <int SIGN>
__device__ inline double2 with_sign(double2 w) {
  if (SIGN < 0)
    w.y = -w.y;
  return w;
}
// SIGN * i * v
template <int SIGN>
__device__ inline double2 times_i(double2 v) {
  return SIGN > 0 ? make_double2(-v.y, v.x) : make_double2(v.y, -v.x);
}

// cos and sin of 2 pi t m / R for the odd radices
template <int R>
__device__ constexpr double odd_cos(int j) {
  constexpr double c3[2] = {1., -0.5};
  constexpr double c5[3] = {1., 0.30901699437494742410, -0.80901699437494742410};
  constexpr double c7[4] = {1., 0.62348980185873353053, -0.22252093395631440429,
                            -0.90096886790241912624};
  const int k = j % R, h = 2 * k > R ? R - k : k;
  return R == 3 ? c3[h] : R == 5 ? c5[h] : c7[h];
}
template <int R>
__device__ constexpr double odd_sin(int j) {
  constexpr double s3[2] = {0., 0.86602540378443864676};
  constexpr double s5[3] = {0., 0.95105651629515357212, 0.58778525229247312917};
  constexpr double s7[4] = {0., 0.78183148246802980871, 0.97492791218182360702,
                            0.43388373911755812048};
  const int k = j % R, h = 2 * k > R ? R - k : k;
  const double s = R == 3 ? s3[h] : R == 5 ? s5[h] : s7[h];
  return 2 * k > R ? -s : s;
}

template <int SIGN>
__device__ inline void dft4(double2 x0, double2 x1, double2 x2, double2 x3, double2 &y0,
                            double2 &y1, double2 &y2, double2 &y3) {
  const double2 a0 = cadd(x0, x2), a1 = csub(x0, x2), a2 = cadd(x1, x3);
  const double2 a3 = times_i<SIGN>(csub(x1, x3));
  y0 = cadd(a0, a2);
  y1 = cadd(a1, a3);
  y2 = csub(a0, a2);
  y3 = csub(a1, a3);
}

// y_t = sum_m x_m W^(t m), W = exp(SIGN 2 pi i / R).  Odd R by the pairs
// x_m + x_{R-m}, x_m - x_{R-m}: real factors only.
template <int R, int SIGN>
__device__ inline void small_dft(const double2 (&x)[R], double2 (&y)[R]) {
  if constexpr (R == 2) {
    y[0] = cadd(x[0], x[1]);
    y[1] = csub(x[0], x[1]);
  } else if constexpr (R == 4) {
    dft4<SIGN>(x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]);
  } else if constexpr (R == 8) {
    // even and odd points by dft4, the odd ones times W^t
    constexpr double h = 0.70710678118654752440;
    double2 e[4], o[4];
    dft4<SIGN>(x[0], x[2], x[4], x[6], e[0], e[1], e[2], e[3]);
    dft4<SIGN>(x[1], x[3], x[5], x[7], o[0], o[1], o[2], o[3]);
    const double2 i1 = times_i<SIGN>(o[1]), i3 = times_i<SIGN>(o[3]);
    o[1] = make_double2(h * (o[1].x + i1.x), h * (o[1].y + i1.y));
    o[2] = times_i<SIGN>(o[2]);
    o[3] = make_double2(h * (i3.x - o[3].x), h * (i3.y - o[3].y));
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      y[t] = cadd(e[t], o[t]);
      y[t + 4] = csub(e[t], o[t]);
    }
  } else {
    constexpr int H = R / 2;
    double2 s[H], d[H];
    y[0] = x[0];
#pragma unroll
    for (int m = 0; m < H; ++m) {
      s[m] = cadd(x[m + 1], x[R - 1 - m]);
      d[m] = csub(x[m + 1], x[R - 1 - m]);
      y[0] = cadd(y[0], s[m]);
    }
#pragma unroll
    for (int t = 1; t <= H; ++t) {
      double2 a = x[0], b = make_double2(0., 0.);
#pragma unroll
      for (int m = 0; m < H; ++m) {
        const double c = odd_cos<R>(t * (m + 1)), q = odd_sin<R>(t * (m + 1));
        a = make_double2(fma(c, s[m].x, a.x), fma(c, s[m].y, a.y));
        b = make_double2(fma(q, d[m].x, b.x), fma(q, d[m].y, b.y));
      }
      b = times_i<SIGN>(b);
      y[t] = cadd(a, b);
      y[R - t] = csub(a, b);
    }
  }
}

// One radix-R pass over C = 2^cshift lines of length n, TILE >= C n.
template <int R, int SIGN, uint32_t TILE, uint32_t NT, bool POW2>
__device__ inline void stockham_pass(double2 *lds, uint32_t n, uint32_t cshift, uint32_t P,
                                     const FftPass &ps, const double2 *tw) {
  constexpr uint32_t NB = (TILE / R + NT - 1) / NT; // butterflies per thread
  const uint32_t q = ps.q, nbf = q << cshift, cmask = (1u << cshift) - 1;
  double2 x[NB][R];
#pragma unroll
  for (uint32_t u = 0; u < NB; ++u) {
    const uint32_t b = threadIdx.x + u * NT;
    if (b < nbf) {
      const double2 *at = lds + (b >> cshift) * P + (b & cmask);
#pragma unroll
      for (int m = 0; m < R; ++m)
        x[u][m] = at[m * q * P];
    }
  }
  __syncthreads();
  const uint32_t p = ps.p;
#pragma unroll
  for (uint32_t u = 0; u < NB; ++u) {
    const uint32_t b = threadIdx.x + u * NT;
    if (b < nbf) {
      const uint32_t i = b >> cshift;
      // i mod p (i < 8192: the float quotient of i + 1/2 truncates exactly)
      const uint32_t k =
          POW2 ? (i & (p - 1))
               : i - p * static_cast<uint32_t>((static_cast<float>(i) + 0.5f) * ps.inv_p);
      double2 y[R];
      if (p > 1) { // uniform; the first pass's twiddles are all 1
#pragma unroll
        for (int m = 1; m < R; ++m)
          x[u][m] = cmul(x[u][m], with_sign<SIGN>(tw[m * k * ps.tstep]));
      }
      small_dft<R, SIGN>(x[u], y);
      double2 *at = lds + ((i - k) * R + k) * P + (b & cmask);
#pragma unroll
      for (int m = 0; m < R; ++m)
        at[m * p * P] = y[m];
    }
  }
  __syncthreads();
}

// Every pass of a plan, in order.  Entered and left with LDS synchronised.
// POW2 instances (plans of radix 8, 4 and 2) leave the odd radices out, whose
// register staging is larger.
template <int SIGN, uint32_t TILE, uint32_t NT, bool POW2>
__device__ inline void run_plan(double2 *lds, const FftPlan &pl, uint32_t cshift, uint32_t P,
                                const double2 *tw) {
  for (uint32_t s = 0; s < pl.npass; ++s) {
    const FftPass ps = pl.pass[s];
    if (ps.radix == 8) {
      stockham_pass<8, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
    } else if (ps.radix == 4) {
      stockham_pass<4, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
    } else if (ps.radix == 2) {
      stockham_pass<2, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
    } else if constexpr (!POW2) {
      if (ps.radix == 3)
        stockham_pass<3, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
      else if (ps.radix == 5)
        stockham_pass<5, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
      else
        stockham_pass<7, SIGN, TILE, NT, POW2>(lds, pl.n, cshift, P, ps, tw);
    }
  }
}

// Power-of-two kernels copy the twiddle table into LDS behind the tile (the
// mixed-radix and Bluestein kernels keep it in memory).
template <uint32_t TILE, int MODE>
constexpr bool fft_lds_tw() {
  return MODE == kFftPow2 && TILE <= 4096;
}

// LDS bytes of a kernel holding `lines` lines at pitch P.
inline uint32_t fft_lds_bytes(const FftLine &L, uint32_t P, uint32_t tile) {
  const uint32_t tw = L.mode == kFftPow2 && tile <= 4096 ? L.len : 0;
  return (L.len * P + tw) * static_cast<uint32_t>(sizeof(double2));
}

// The table the passes read: loaded into LDS behind the tile where the
// kernel keeps it there (the caller synchronises before the first pass).
template <uint32_t TILE, uint32_t NT, int MODE>
__device__ inline const double2 *fft_tables(double2 *lds, const FftLine &L, uint32_t P) {
  if constexpr (fft_lds_tw<TILE, MODE>()) {
    double2 *t = lds + L.len * P;
    for (uint32_t e = threadIdx.x; e < L.len; e += NT)
      t[e] = L.tw[e];
    return t;
  } else {
    return L.tw;
  }
}

// Transforms 2^cshift lines, entered and left with LDS synchronised; points
// t >= n of a line (Bluestein) need not be set.
template <int SIGN, uint32_t TILE, uint32_t NT, int MODE>
__device__ inline void fft_lines(double2 *lds, const double2 *twl, const FftLine &L,
                                 uint32_t cshift, uint32_t P) {
  if constexpr (MODE != kFftBlue) {
    run_plan<SIGN, TILE, NT, MODE == kFftPow2>(lds, L.plan, cshift, P, twl);
  } else {
    const uint32_t cmask = (1u << cshift) - 1, total = L.len << cshift;
    for (uint32_t e = threadIdx.x; e < total; e += NT) {
      const uint32_t t = e >> cshift;
      double2 *at = lds + t * P + (e & cmask);
      *at = t < L.n ? cmul(*at, with_sign<SIGN>(L.chirp[t])) : make_double2(0., 0.);
    }
    __syncthreads();
    run_plan<-1, TILE, NT, true>(lds, L.plan, cshift, P, twl);
    for (uint32_t e = threadIdx.x; e < total; e += NT) {
      const uint32_t t = e >> cshift;
      double2 *at = lds + t * P + (e & cmask);
      *at = cmul(*at, with_sign<SIGN>(L.bhat[t]));
    }
    __syncthreads();
    run_plan<1, TILE, NT, true>(lds, L.plan, cshift, P, twl);
    const double inv_m = 1.0 / static_cast<double>(L.len);
    for (uint32_t e = threadIdx.x; e < (L.n << cshift); e += NT) {
      const uint32_t t = e >> cshift;
      double2 *at = lds + t * P + (e & cmask);
      const double2 v = cmul(*at, with_sign<SIGN>(L.chirp[t]));
      *at = make_double2(v.x * inv_m, v.y * inv_m);
    }
    __syncthreads();
  }
}

// Lines along one axis of an array: `lines` of them, consecutive ones
// `inner` at a time at consecutive addresses, `outer` apart between such
// groups, points s apart; C = 2^cshift of them per workgroup.
struct FftAxis {
  uint64_t s, inner, outer, lines;
  uint32_t cshift, P;
};

// The tile of workgroup b of g (g a multiple of 8): the eight XCDs take
// workgroups in turn, and this gives each of them a contiguous run of tiles,
// so that neighbouring columns meet in one L2.  Columns rarely start on a
// cache line (H's rows are nz/2 + 1 long), and a tile's rows are a line or
// less: both tiles that touch a line then read it from memory once (y passes
// of es 512x512x128: 280 -> 204 us; with eight columns a tile, 172 us).
__device__ inline uint32_t xcd_tile(uint32_t b, uint32_t g) { return (b & 7) * (g >> 3) + (b >> 3); }
inline unsigned xcd_grid(uint64_t tiles) { return static_cast<unsigned>((tiles + 7) / 8 * 8); }

__device__ inline uint64_t line_base(const FftAxis &ax, uint64_t L) {
  if (ax.lines <= 0xffffffffull) { // uniform: 32-bit software division
    const uint32_t l = static_cast<uint32_t>(L), in = static_cast<uint32_t>(ax.inner);
    const uint32_t g = l / in;
    return static_cast<uint64_t>(g) * ax.outer + (l - g * in);
  }
  return (L / ax.inner) * ax.outer + (L % ax.inner);
}

// ------------------------------------------------------------------ host --
// The line description of length n (n >= 2, fft_length_ok), its tables
// cached in the context.
int fft_line(hamx_ctx *ctx, uint64_t n, FftLine *out);
// One strided axis pass of up to three arrays of one shape, in place: the
// lines of `n` points ax.s apart.
int fft_strided(hamx_ctx *ctx, double2 *const data[3], unsigned arrays, const FftLine &L,
                FftAxis ax, int sign);
// fft_strided of exponent +1 that also leaves the partial sums of the first
// array's variance: *np groups of four doubles at *part (hamx_rnd_half.h).
int fft_strided_var(hamx_ctx *ctx, double2 *const data[3], unsigned arrays, const FftLine &L,
                    FftAxis ax, uint64_t nfull, double **part, uint32_t *np);
// cshift of the largest power of two of lines of `len` points in `tile`
// values, at most 2^most and `lines` (rounded up to a power of two).
uint32_t fft_cshift(uint32_t tile, uint32_t len, uint32_t most, uint64_t lines);

} // namespace hamx
