// Half-space passes of the random-field generators (included by
// hamx_rnd.hip).
//
// The generators' transforms carry far less than the complex arrays they are
// written with.  In Brnd_es, Gram-Schmidt reads 0.5 (Re c(k) + Re c(-k)) of
// the forward transform of c0 = bx + i by, c1 = by + i bz, and the
// extraction 0.5 (Re c(r) + Re c(-r)) of the last one: with E f = (f(r) +
// f(-r)) / 2, both are the transform of the real even field E bx (E by, E bz)
// alone, which is real and even again.  (The imaginary part of c0, the
// second copy of by, enters neither.)  A real even array is held by half of
// its x planes, and after its z transform by half of its kz as well, since
//   G(-x, -y, kz) = conj G(x, y, kz)   after z,
//   G(-x, ky, kz) = conj G(x, ky, kz)  after z and y (so x is complex to real),
// and the same in reverse on the way back.  Three fields cost 12 bytes per
// vertex per read or write this way instead of 32:
//
//   es: k_draw_axis   draw + x(+)                                write 32 B
//       fft_strided   y(+), and the variance's partial sums      64 B
//       k_es_mid      z(+), rescale, even part, z(-)             read 32, write 12
//       fft_strided   y(-)                                       24 B
//       k_es_gs_x     x(-), Gram-Schmidt and even part, x(+)     24 B
//       fft_strided   y(+)                                       24 B
//       k_half_out    z(+), the three fields                     read 12, write 24
//   mhd: k_mhd_x (draw, even part, x(+)), fft_strided y(+), k_half_out
//   te: k_draw_axis, fft_strided with the variance sums, k_te_out (z(+), rescale)
//
// 248 bytes per vertex for es instead of 808 (one elementwise or axis pass
// at a time over two complex arrays), 72 instead of 280 for mhd, 72 instead of
// 144 for te.  Measured per realisation, whole-array steps -> these (with the
// engine and table work below): es 256x256x64 726 -> 304 us, es 512x512x128
// 7.05 -> 2.23 ms, te 800x800x160 7.90 -> 2.69 ms, mhd 135x121x98 344 -> 125 us.
//
// Half arrays: H[i][j][k], i <= nx/2, all j, k <= nz/2.  Two real lines share
// one complex transform: X + i U in one, V in the other.
#pragma once

#include <type_traits>

namespace hamx {

struct HalfArgs {
  uint32_t nx, ny, nz; // the box
  uint32_t nx2, nh;    // nx/2 + 1, nz/2 + 1
  uint32_t lines;      // nx2 * ny stored z lines
  uint32_t ncol;       // columns of the strided pass
  FastDiv dz, dh;      // by nz, nh
};

struct HalfArrays {
  double2 *x, *u, *v;
};

// X(k), U(k) of two real lines from Z = FFT(x + i u) at k and -k.
__device__ inline void split_pair(const double2 &zk, const double2 &zm, double2 &X, double2 &U) {
  X = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
  U = make_double2(0.5 * (zk.y + zm.y), 0.5 * (zm.x - zk.x));
}

// Z at k and n - k of the Hermitian lines X, U, V (their points k <= n/2):
// X + i U on one line, V on the line voff values after it.  The points that
// are their own mirror are real.
__device__ inline void join_lines(double2 *at, uint32_t k, uint32_t n, uint32_t P, uint32_t voff,
                                  const double2 &X, const double2 &U, const double2 &V) {
  if (k == 0 || 2 * k == n) {
    at[k * P] = make_double2(X.x, U.x);
    at[k * P + voff] = make_double2(V.x, 0.);
    return;
  }
  at[k * P] = make_double2(X.x - U.y, X.y + U.x);
  at[k * P + voff] = V;
  at[(n - k) * P] = make_double2(X.x + U.y, U.x - X.y);
  at[(n - k) * P + voff] = make_double2(V.x, -V.y);
}

__device__ inline uint32_t mirror_of(uint32_t i, uint32_t n) { return i == 0 ? 0 : n - i; }

// ------------------------------------------------------------ draw + x(+) --
// Brnd_es (two complex values per mode) and TErnd_dft (one).
struct EsDraw {
  static constexpr int NL = 2;
  EsArgs a;
  __device__ void operator()(double k2, uint64_t idx, uint64_t seed, double2 (&v)[NL]) const {
    const double sigma = es_sigma(a, k2);
    double g0, g1, g2, g3;
    gauss_pair(seed, 0, 2 * idx, g0, g1);
    gauss_pair(seed, 0, 2 * idx + 1, g2, g3);
    v[0] = make_double2(sigma * g0, sigma * g1);
    v[1] = make_double2(sigma * g2, sigma * g3);
  }
};

struct DftDraw {
  static constexpr int NL = 1;
  DftArgs a;
  __device__ void operator()(double k2, uint64_t idx, uint64_t seed, double2 (&v)[NL]) const {
    const double sigma = dft_sigma(a, k2);
    double g0, g1;
    gauss_pair(seed, 1, idx, g0, g1);
    v[0] = make_double2(sigma * g0, sigma * g1);
  }
};

// A tile of C columns (j, l): the modes (0..nx-1, j, l) drawn into LDS,
// transformed along x and stored.  The wave numbers of j and l are formed
// once per thread, the squares of x's once per workgroup in LDS (behind the
// engine's tables).  Bound by the FP64 and integer instructions of the draws:
// with the band decided on |k|^2, the spectrum as one power of it and the
// square roots and angles without the library's special cases, te 800x800x160
// 2633 -> 1416 us, es 256x256x64 94 -> 82 us (1207 and 78 with radix 8).
template <typename Draw, uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_draw_axis(double2 *__restrict__ o0,
                                                  double2 *__restrict__ o1, Draw dr,
                                                  uint64_t seed, HalfArgs h, FftLine L,
                                                  uint32_t cs) {
  extern __shared__ double2 lds[];
  constexpr int NL = Draw::NL;
  const BoxArgs &b = dr.a.b;
  const uint32_t n = L.n, C = 1u << cs, P = C * NL;
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint32_t c = threadIdx.x & (C - 1), t0 = threadIdx.x >> cs, dt = NT >> cs;
  const uint32_t col = (blockIdx.x << cs) + c;
  const bool on = col < h.ncol;
  const uint32_t j = col / h.nz, l = col - j * h.nz;
  const double ky = wavenum(j, b.ny, b.ly), kz = wavenum(l, b.nz, b.lz);
  double *kx2 = reinterpret_cast<double *>(lds) +
                2 * (L.len * P + (fft_lds_tw<TILE, MODE>() ? L.len : 0));
  for (uint32_t t = threadIdx.x; t < n; t += NT) {
    const double kx = wavenum(t, b.nx, b.lx);
    kx2[t] = kx * kx;
  }
  __syncthreads();
#pragma unroll 1
  for (uint32_t t = t0; t < n; t += dt) {
    const uint64_t idx = static_cast<uint64_t>(t) * h.ncol + col;
    double2 v[NL];
#pragma unroll
    for (int m = 0; m < NL; ++m)
      v[m] = make_double2(0., 0.);
    if (on && idx != 0)
      dr(mode_k2(kx2[t], ky, kz), idx, seed, v);
#pragma unroll
    for (int m = 0; m < NL; ++m)
      lds[t * P + m * C + c] = v[m];
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cs + (NL - 1), P);
  if (!on)
    return;
  for (uint32_t t = t0; t < n; t += dt) {
    const uint64_t idx = static_cast<uint64_t>(t) * h.ncol + col;
    o0[idx] = lds[t * P + c];
    if constexpr (NL == 2)
      o1[idx] = lds[t * P + C + c];
  }
}

// ---------------------------------------------------- variance, from y(+) --
// toolkit::variance over the first n doubles of c0 (toolkit.h:48-78) from
// its y-transformed lines: a z line's doubles sum to nz (Re G_0 + Im G_0) and
// their squared deviations from m to nz (sum_{k>0} |G_k|^2 + |G_0 - m (1 + i)|^2)
// by Parseval.  part holds, per workgroup of the y pass, the mean of the
// k = 0 components it saw, their count, their squared deviations from that
// mean, and the sum of the other |G_k|^2 (fft_strided_var).  With an odd
// number of z lines the first n doubles end inside one: that line (`rest`) is
// transformed here and its first nz doubles are taken as they are.
template <int MODE>
__global__ __launch_bounds__(1024) void k_var_half(const double *part, uint32_t np,
                                                   const double2 *rest, FftLine L, double n,
                                                   double *out) {
  extern __shared__ double2 lds[];
  constexpr uint32_t NT = 1024;
  const uint32_t nz = L.n;
  const double nzd = static_cast<double>(nz);
  double own = 0.; // this thread's double of the rest line (nz <= 1024)
  const bool has = rest && threadIdx.x < nz;
  if (rest) {
    const double2 *twl = fft_tables<NT, NT, MODE>(lds, L, 1);
    if (threadIdx.x < nz)
      lds[threadIdx.x] = rest[threadIdx.x];
    __syncthreads();
    fft_lines<1, NT, NT, MODE>(lds, twl, L, 0, 1);
    if (has) {
      const double2 v = lds[threadIdx.x >> 1];
      own = threadIdx.x & 1 ? v.y : v.x;
    }
  }
  double s = 0.;
  for (uint32_t i = threadIdx.x; i < np; i += NT)
    s += part[4 * i] * part[4 * i + 1];
  const double mean = block_sum<NT>(nzd * s + own) / n;
  double e = 0.;
  for (uint32_t i = threadIdx.x; i < np; i += NT) {
    const double d = part[4 * i] - mean;
    e += part[4 * i + 2] + part[4 * i + 1] * (d * d) + part[4 * i + 3];
  }
  const double d = has ? own - mean : 0.;
  const double var = block_sum<NT>(nzd * e + d * d) / n;
  if (threadIdx.x == 0) {
    out[0] = mean;
    out[1] = var;
  }
}

// ------------------------------------- z(+), rescale, even part, z(-) --
// CL stored z lines (i, j) and their mirrors (-i, -j): lines c0 and c1 of
// the former in LDS, then those of the latter.  A thread's vertex l of a
// line and vertex -l of its mirror are read by no other thread, so the even
// parts go straight back into the two lines' places.  SPLIT takes the
// rescale's factors from tables of the tile's 2 CL lines and of z in LDS: the
// kernel was bound by the per-vertex models (es 256x256x64 106 -> 62 us, 55 with radix 8).
template <bool SPLIT, uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_es_mid(const double2 *__restrict__ c0,
                                               const double2 *__restrict__ c1, HalfArrays H,
                                               EsArgs a, const double *__restrict__ var,
                                               HalfArgs h, FftLine L, uint32_t cl) {
  extern __shared__ double2 lds[];
  constexpr uint32_t K = TILE / 4 / NT; // a thread's points of each of the four line sets
  const uint32_t n = h.nz, CL = 1u << cl, P = 4 * CL + 1;
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint32_t L0 = blockIdx.x << cl;
  const uint32_t nl = h.lines - L0 < CL ? h.lines - L0 : CL;
  double2 r[K][4];
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t e = threadIdx.x + NT * k, q = fast_quot(h.dz, e);
#pragma unroll
    for (int m = 0; m < 4; ++m)
      r[k][m] = make_double2(0., 0.);
    if (q < nl) {
      const uint32_t line = L0 + q, i = line / h.ny, j = line - i * h.ny;
      const uint64_t own = static_cast<uint64_t>(line) * n + (e - q * n);
      const uint64_t mir = (static_cast<uint64_t>(mirror_of(i, h.nx)) * h.ny +
                            mirror_of(j, h.ny)) * n + (e - q * n);
      r[k][0] = c0[own];
      r[k][1] = c1[own];
      r[k][2] = c0[mir];
      r[k][3] = c1[mir];
    }
  }
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t e = threadIdx.x + NT * k, q = fast_quot(h.dz, e);
    if (q < CL) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        lds[(e - q * n) * P + m * CL + q] = r[k][m];
    }
  }
  const EsScale sc = es_scale(a, var);
  EsZ *zt = reinterpret_cast<EsZ *>(lds + L.len * P + (fft_lds_tw<TILE, MODE>() ? L.len : 0));
  EsLine *lt = reinterpret_cast<EsLine *>(zt + n);
  if constexpr (SPLIT) {
    for (uint32_t e = threadIdx.x; e < n + 2 * nl; e += NT) {
      if (e < n) {
        zt[e] = es_z(a, e);
      } else {
        const bool mir = e - n >= nl;
        const uint32_t q = e - n - (mir ? nl : 0), line = L0 + q;
        const uint32_t i = line / h.ny, j = line - i * h.ny;
        lt[mir ? CL + q : q] = mir ? es_line(a, sc, mirror_of(i, h.nx), mirror_of(j, h.ny))
                                   : es_line(a, sc, i, j);
      }
    }
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cl + 2, P);
#pragma unroll 1
  for (uint32_t e = threadIdx.x; e < nl * n; e += NT) {
    const uint32_t q = fast_quot(h.dz, e), l = e - q * n, lm = mirror_of(l, n);
    Vec3 f{0., 0., 0.};
    if constexpr (SPLIT) {
      const Vec3 b = es_rescale_split(lt[q], zt[l], sc, lds[l * P + q], lds[l * P + CL + q]);
      const Vec3 m = es_rescale_split(lt[CL + q], zt[lm], sc, lds[lm * P + 2 * CL + q],
                                      lds[lm * P + 3 * CL + q]);
      f = Vec3{b.x + m.x, b.y + m.y, b.z + m.z};
    } else {
      const uint32_t line = L0 + q, i = line / h.ny, j = line - i * h.ny;
#pragma unroll 1
      for (int m = 0; m < 2; ++m) {
        const uint32_t vi = m ? mirror_of(i, h.nx) : i, vj = m ? mirror_of(j, h.ny) : j;
        const uint32_t vl = m ? lm : l;
        const double2 v0 = lds[vl * P + 2 * m * CL + q], v1 = lds[vl * P + (2 * m + 1) * CL + q];
        Vec3 b;
        if (!es_rescale_at<true>(a, sc, vi, vj, vl, v0, v1, b))
          b = Vec3{v0.x, v1.x, v1.y};
        f.x += b.x;
        f.y += b.y;
        f.z += b.z;
      }
    }
    lds[l * P + q] = make_double2(0.5 * f.x, 0.5 * f.y);
    lds[l * P + CL + q] = make_double2(0.5 * f.z, 0.);
  }
  __syncthreads();
  fft_lines<-1, TILE, NT, MODE>(lds, twl, L, cl + 1, P);
  const uint64_t out0 = static_cast<uint64_t>(L0) * h.nh;
  for (uint32_t e = threadIdx.x; e < nl * h.nh; e += NT) {
    const uint32_t q = fast_quot(h.dh, e), k = e - q * h.nh;
    double2 X, U;
    split_pair(lds[k * P + q], lds[mirror_of(k, n) * P + q], X, U);
    H.x[out0 + e] = X;
    H.u[out0 + e] = U;
    H.v[out0 + e] = lds[k * P + CL + q];
  }
}

// -------------------------------------------------- columns along x (half) --
// The Hermitian lines of a column into LDS, and back from it.
template <uint32_t TILE, uint32_t NT>
__device__ inline void load_half_columns(double2 *lds, const HalfArrays &H, const HalfArgs &h,
                                         uint32_t cs, uint32_t col, bool on) {
  constexpr uint32_t K = TILE / 4 / NT + 1; // nx/2 + 1 points, 2 lines per column in TILE
  const uint32_t C = 1u << cs, P = 2 * C, c = threadIdx.x & (C - 1);
  const uint32_t t0 = threadIdx.x >> cs, dt = NT >> cs;
  double2 r[K][3];
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t i = t0 + dt * k;
#pragma unroll
    for (int m = 0; m < 3; ++m)
      r[k][m] = make_double2(0., 0.);
    if (on && i < h.nx2) {
      const uint64_t at = static_cast<uint64_t>(i) * h.ncol + col;
      r[k][0] = H.x[at];
      r[k][1] = H.u[at];
      r[k][2] = H.v[at];
    }
  }
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t i = t0 + dt * k;
    if (i < h.nx2)
      join_lines(lds + c, i, h.nx, P, C, r[k][0], r[k][1], r[k][2]);
  }
}

template <uint32_t NT>
__device__ inline void store_half_columns(const double2 *lds, const HalfArrays &H,
                                          const HalfArgs &h, uint32_t cs, uint32_t col, bool on) {
  const uint32_t C = 1u << cs, P = 2 * C, c = threadIdx.x & (C - 1);
  if (!on)
    return;
  for (uint32_t i = threadIdx.x >> cs; i < h.nx2; i += NT >> cs) {
    const uint64_t at = static_cast<uint64_t>(i) * h.ncol + col;
    double2 X, U;
    split_pair(lds[i * P + c], lds[mirror_of(i, h.nx) * P + c], X, U);
    H.x[at] = X;
    H.u[at] = U;
    H.v[at] = lds[i * P + C + c];
  }
}

// x(-), Gram-Schmidt (brnd_es.cc:211-259) of the real even k-space vector,
// the even part of the result, x(+).  The vector is the same at k and -k, the
// results are not: a wave number beyond half its axis is i/L - n/L, which
// carries the rounding of n/L that its mirror's does not, and at half the axis it
// keeps its sign.  Each wave vector gives a result of its own and both enter the
// even part (with k's alone es 512x512x128 was 2.2e-15 to 3.0e-15 from a 64-bit
// reference, with both it is 1.0e-15, as the whole-array steps).  The wave numbers
// along x are formed once per workgroup, in LDS behind the engine's tables.
template <uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_es_gs_x(HalfArrays H, EsArgs a, HalfArgs h, FftLine L,
                                                uint32_t cs) {
  extern __shared__ double2 lds[];
  const uint32_t n = h.nx, C = 1u << cs, P = 2 * C;
  const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) << cs;
  if (col0 >= h.ncol)
    return; // uniform: the grid's last few workgroups
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint32_t c = threadIdx.x & (C - 1), t0 = threadIdx.x >> cs, dt = NT >> cs;
  const uint32_t col = col0 + c;
  const bool on = col < h.ncol;
  load_half_columns<TILE, NT>(lds, H, h, cs, col, on);
  double *kx = reinterpret_cast<double *>(lds) +
               2 * (L.len * P + (fft_lds_tw<TILE, MODE>() ? L.len : 0));
  for (uint32_t t = threadIdx.x; t < n; t += NT)
    kx[t] = wavenum(t, n, a.b.lx);
  __syncthreads();
  fft_lines<-1, TILE, NT, MODE>(lds, twl, L, cs + 1, P);
  const uint32_t j = col / h.nh, l = col - j * h.nh;
  const uint32_t js = mirror_of(j, h.ny), ls = mirror_of(l, h.nz);
  Vec3 k{0., wavenum(j, h.ny, a.b.ly), wavenum(l, h.nz, a.b.lz)};
  Vec3 ks{0., wavenum(js, h.ny, a.b.ly), wavenum(ls, h.nz, a.b.lz)};
#pragma unroll 1
  for (uint32_t t = t0; t < n; t += dt) {
    double2 &z = lds[t * P + c], &zv = lds[t * P + C + c];
    const Vec3 b{z.x, z.y, zv.x};
    k.x = kx[t];
    ks.x = kx[mirror_of(t, n)];
    const Vec3 f = es_gs(a, k, b), fs = es_gs(a, ks, b);
    z = make_double2(cgs::sqrtwo * (0.5 * (f.x + fs.x)), cgs::sqrtwo * (0.5 * (f.y + fs.y)));
    zv = make_double2(cgs::sqrtwo * (0.5 * (f.z + fs.z)), 0.);
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cs + 1, P);
  store_half_columns<NT>(lds, H, h, cs, col, on);
}

// Brnd_mhd's modes, their even part (the only part the extraction keeps) and
// x(+).  A mode and its mirror are evaluated each with its own wave vector (see
// k_es_gs_x; one spectrum for both, 121 instead of 125 us a realisation of
// 135x121x98, was 2.9e-15 instead of 6.5e-16 from a 64-bit reference).  Bound by
// FP64 instructions: mhd 135x121x98 149 -> 66 us with the spectra as powers of
// |k|^2 and no library pow.
template <uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_mhd_x(HalfArrays H, MhdArgs a, uint64_t seed,
                                              const double *__restrict__ bobs, HalfArgs h,
                                              FftLine L, uint32_t cs) {
  extern __shared__ double2 lds[];
  const uint32_t n = h.nx, C = 1u << cs, P = 2 * C;
  const uint32_t col0 = xcd_tile(blockIdx.x, gridDim.x) << cs;
  if (col0 >= h.ncol)
    return; // uniform: the grid's last few workgroups
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const Vec3 bh = versor3(Vec3{bobs[0], bobs[1], bobs[2]});
  const uint32_t c = threadIdx.x & (C - 1), t0 = threadIdx.x >> cs, dt = NT >> cs;
  const uint32_t col = col0 + c;
  const bool on = col < h.ncol;
  const uint32_t j = col / h.nh, l = col - j * h.nh;
  const uint32_t js = mirror_of(j, h.ny), ls = mirror_of(l, h.nz);
  Vec3 k{0., wavenum(j, h.ny, a.b.ly), wavenum(l, h.nz, a.b.lz)};
  Vec3 ks{0., wavenum(js, h.ny, a.b.ly), wavenum(ls, h.nz, a.b.lz)};
  double *kx = reinterpret_cast<double *>(lds) +
               2 * (L.len * P + (fft_lds_tw<TILE, MODE>() ? L.len : 0));
  for (uint32_t t = threadIdx.x; t < n; t += NT)
    kx[t] = wavenum(t, n, a.b.lx);
  __syncthreads();
#pragma unroll 1
  for (uint32_t t = t0; t < n; t += dt) {
    const uint32_t ts = mirror_of(t, n);
    const uint64_t idx = (static_cast<uint64_t>(t) * h.ny + j) * h.nz + l;
    const uint64_t sym = (static_cast<uint64_t>(ts) * h.ny + js) * h.nz + ls;
    Vec3 f{0., 0., 0.};
    if (on && idx != 0) {
      k.x = kx[t];
      ks.x = kx[ts];
      const double x = k.x * k.x + k.y * k.y + k.z * k.z;
      const double xs = ks.x * ks.x + ks.y * ks.y + ks.z * ks.z;
      MhdShape m = mhd_shape(a, bh, k);
      f = mhd_field(seed, m, mhd_power(a, x, a.bands.of(x), m.c), k, x, idx, t == 0 && j == 0);
      m = mhd_shape(a, bh, ks);
      const Vec3 s = mhd_field(seed, m, mhd_power(a, xs, a.bands.of(xs), m.c), ks, xs, sym,
                               t == 0 && j == 0);
      f = Vec3{f.x + s.x, f.y + s.y, f.z + s.z};
    }
    lds[t * P + c] = make_double2(0.5 * f.x, 0.5 * f.y);
    lds[t * P + C + c] = make_double2(0.5 * f.z, 0.);
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cs + 1, P);
  store_half_columns<NT>(lds, H, h, cs, col, on);
}

// ------------------------------------------------------ z(+), the outputs --
// CL stored lines; each vertex's value is its mirror's as well.
template <uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_half_out(HalfArrays H, double *__restrict__ bx,
                                                 double *__restrict__ by,
                                                 double *__restrict__ bz, double scale,
                                                 HalfArgs h, FftLine L, uint32_t cl) {
  extern __shared__ double2 lds[];
  constexpr uint32_t K = TILE / 4 / NT + 1; // nz/2 + 1 points, 2 lines per unit in TILE
  const uint32_t n = h.nz, CL = 1u << cl, P = 2 * CL + 1;
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint32_t L0 = blockIdx.x << cl;
  const uint32_t nl = h.lines - L0 < CL ? h.lines - L0 : CL;
  const uint64_t in0 = static_cast<uint64_t>(L0) * h.nh;
  for (uint32_t e0 = threadIdx.x; e0 < CL * h.nh; e0 += NT * K) {
    double2 r[K][3];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t e = e0 + NT * k;
#pragma unroll
      for (int m = 0; m < 3; ++m)
        r[k][m] = make_double2(0., 0.);
      if (e < nl * h.nh) {
        r[k][0] = H.x[in0 + e];
        r[k][1] = H.u[in0 + e];
        r[k][2] = H.v[in0 + e];
      }
    }
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t e = e0 + NT * k, q = fast_quot(h.dh, e);
      if (q < CL)
        join_lines(lds + q, e - q * h.nh, n, P, CL, r[k][0], r[k][1], r[k][2]);
    }
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cl + 1, P);
  for (uint32_t e = threadIdx.x; e < nl * n; e += NT) {
    const uint32_t q = fast_quot(h.dz, e), l = e - q * n;
    const uint32_t line = L0 + q, i = line / h.ny, j = line - i * h.ny;
    const double2 z = lds[l * P + q];
    const double x = z.x * scale, y = z.y * scale, v = lds[l * P + CL + q].x * scale;
    uint64_t at = static_cast<uint64_t>(line) * n + l;
    bx[at] = x;
    by[at] = y;
    bz[at] = v;
    if (i != 0 && 2 * i != h.nx) { // its mirror is not a stored line
      at = (static_cast<uint64_t>(h.nx - i) * h.ny + mirror_of(j, h.ny)) * n + mirror_of(l, n);
      bx[at] = x;
      by[at] = y;
      bz[at] = v;
    }
  }
}

// z(+) and the energy profile of TErnd_dft (ternd_dft.cc:109-128): CL z lines
// of the whole box.  SPLIT takes the profile's factors from tables in LDS (te
// 800x800x160 1072 -> 727 us, 579 with radix 8).
template <bool SPLIT, uint32_t TILE, uint32_t NT, int MODE>
__global__ __launch_bounds__(NT) void k_te_out(const double2 *__restrict__ tk,
                                               double *__restrict__ te, DftArgs a,
                                               const double *__restrict__ var, HalfArgs h,
                                               uint32_t lines, FftLine L, uint32_t cl) {
  extern __shared__ double2 lds[];
  constexpr uint32_t K = TILE / NT;
  const uint32_t n = h.nz, CL = 1u << cl, P = CL + 1;
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint32_t L0 = blockIdx.x << cl;
  const uint32_t nl = lines - L0 < CL ? lines - L0 : CL;
  const uint64_t at0 = static_cast<uint64_t>(L0) * n;
  double2 r[K];
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t e = threadIdx.x + NT * k;
    r[k] = e < nl * n ? tk[at0 + e] : make_double2(0., 0.);
  }
#pragma unroll
  for (uint32_t k = 0; k < K; ++k) {
    const uint32_t e = threadIdx.x + NT * k, q = fast_quot(h.dz, e);
    if (q < CL)
      lds[(e - q * n) * P + q] = r[k];
  }
  const double te_var_invsq = 1. / sqrt(var[0]);
  double *zt = reinterpret_cast<double *>(lds + L.len * P +
                                          (fft_lds_tw<TILE, MODE>() ? L.len : 0));
  if constexpr (SPLIT) {
    for (uint32_t e = threadIdx.x; e < n + nl; e += NT) {
      const uint32_t line = L0 + e - n, i = line / h.ny;
      zt[e] = e < n ? dft_z(a, e) : dft_line(a, i, line - i * h.ny, te_var_invsq);
    }
  }
  __syncthreads();
  fft_lines<1, TILE, NT, MODE>(lds, twl, L, cl, P);
#pragma unroll 1
  for (uint32_t e = threadIdx.x; e < nl * n; e += NT) {
    const uint32_t q = fast_quot(h.dz, e), l = e - q * n;
    if constexpr (SPLIT) {
      te[at0 + e] = lds[l * P + q].x * (zt[n + q] * zt[l]);
    } else {
      const uint32_t line = L0 + q, i = line / h.ny, j = line - i * h.ny;
      te[at0 + e] = lds[l * P + q].x * dft_ratio(a, i, j, l, te_var_invsq);
    }
  }
}

// -------------------------------------------------------------------- host --
// Calls f(TILE, NT, MODE) as integral constants.
template <typename F>
void with_tile(uint32_t tile, int mode, F f) {
  auto m = [&](auto T, auto NT) {
    if (mode == kFftPow2)
      f(T, NT, std::integral_constant<int, kFftPow2>{});
    else if (mode == kFftMixed)
      f(T, NT, std::integral_constant<int, kFftMixed>{});
    else
      f(T, NT, std::integral_constant<int, kFftBlue>{});
  };
  if (tile == 2048)
    m(std::integral_constant<uint32_t, 2048>{}, std::integral_constant<uint32_t, 256>{});
  else if (tile == 4096)
    m(std::integral_constant<uint32_t, 4096>{}, std::integral_constant<uint32_t, 512>{});
  else
    m(std::integral_constant<uint32_t, 8192>{}, std::integral_constant<uint32_t, 1024>{});
}

// A generator's box on the half-space passes.
struct HalfPlan {
  HalfArgs h; // ncol is set by each pass
  FftLine lx, ly, lz;
  // the tile and its columns (2^cs) of the passes along x with nl lines per
  // column: the smallest tile with four columns, whose rows are then 64 bytes
  uint32_t x_tile(int nl, uint32_t ncol, uint32_t *cs) const {
    for (uint32_t tile = 2048;; tile *= 2) {
      *cs = fft_cshift(tile / nl, lx.len, 4, ncol);
      if (*cs >= 2 || tile == kTileMax || (1ull << *cs) >= ncol)
        if (lx.len * nl <= tile)
          return tile;
    }
  }
  // ... and of the passes along z with nl lines in LDS per stored line
  uint32_t z_tile(int nl, uint32_t lines, uint32_t *cl) const {
    const uint32_t tile = 2 * nl * lz.len <= 2048 ? 2048 : 4096;
    *cl = fft_cshift(tile / nl, lz.len, 11, lines);
    return tile;
  }
};

// LDS bounds of the passes: two lines of x in the largest tile, four of z in
// 4096 values (hamx_rnd.hip takes the whole-array steps otherwise), and
// 32-bit vertex indices.
inline bool half_plan(hamx_ctx *ctx, const BoxArgs &b, HalfPlan *p, int *rc) {
  *rc = HAMX_OK;
  if (b.n > 0xffffffffull)
    return false;
  if ((*rc = fft_line(ctx, b.nx, &p->lx)) != HAMX_OK ||
      (*rc = fft_line(ctx, b.ny, &p->ly)) != HAMX_OK ||
      (*rc = fft_line(ctx, b.nz, &p->lz)) != HAMX_OK)
    return false;
  if (2 * p->lx.len > kTileMax || 4 * p->lz.len > 4096)
    return false;
  HalfArgs &h = p->h;
  h.nx = static_cast<uint32_t>(b.nx);
  h.ny = static_cast<uint32_t>(b.ny);
  h.nz = static_cast<uint32_t>(b.nz);
  h.nx2 = h.nx / 2 + 1;
  h.nh = h.nz / 2 + 1;
  h.lines = h.nx2 * h.ny;
  h.ncol = 0;
  h.dz = fast_div(h.nz);
  h.dh = fast_div(h.nh);
  return true;
}

inline HalfArrays half_arrays(const HalfPlan &p, void *w) {
  const uint64_t n = static_cast<uint64_t>(p.h.lines) * p.h.nh;
  double2 *d = static_cast<double2 *>(w);
  return HalfArrays{d, d + n, d + 2 * n};
}
inline size_t half_bytes(const HalfPlan &p) {
  return 3 * static_cast<size_t>(p.h.lines) * p.h.nh * sizeof(double2);
}

// y pass of the three half arrays.
inline int half_y(hamx_ctx *ctx, const HalfPlan &p, const HalfArrays &H, int sign) {
  FftAxis ax{};
  ax.s = ax.inner = p.h.nh;
  ax.outer = static_cast<uint64_t>(p.h.ny) * p.h.nh;
  ax.lines = static_cast<uint64_t>(p.h.nx2) * p.h.nh;
  double2 *const arr[3] = {H.x, H.u, H.v};
  return fft_strided(ctx, arr, 3, p.ly, ax, sign);
}

// z(+) of the half arrays and the outputs.
inline int half_out(hamx_ctx *ctx, const HalfPlan &p, const HalfArrays &H, double *bx, double *by,
                    double *bz, double scale) {
  uint32_t cl;
  const uint32_t tile = p.z_tile(2, p.h.lines, &cl);
  with_tile(tile, p.lz.mode, [&](auto T, auto NT, auto M) {
    hipLaunchKernelGGL((k_half_out<decltype(T)::value, decltype(NT)::value, decltype(M)::value>),
                       dim3((p.h.lines + (1u << cl) - 1) >> cl), dim3(decltype(NT)::value),
                       fft_lds_bytes(p.lz, (2u << cl) + 1, tile), ctx->stream, H, bx, by, bz,
                       scale, p.h, p.lz, cl);
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

// Draw and x(+), then y(+) with the variance of the first n doubles of the
// first array into red[0..1] (mean, variance).
template <typename Draw>
int half_draw(hamx_ctx *ctx, const HalfPlan &p, const Draw &dr, uint64_t seed, double2 *c0,
              double2 *c1, double *red) {
  HalfArgs h = p.h;
  h.ncol = h.ny * h.nz;
  uint32_t cs;
  const uint32_t tile = p.x_tile(Draw::NL, h.ncol, &cs);
  with_tile(tile, p.lx.mode, [&](auto T, auto NT, auto M) {
    hipLaunchKernelGGL((k_draw_axis<Draw, decltype(T)::value, decltype(NT)::value, decltype(M)::value>),
                       dim3((h.ncol + (1u << cs) - 1) >> cs), dim3(decltype(NT)::value),
                       fft_lds_bytes(p.lx, Draw::NL << cs, tile) + p.lx.n * sizeof(double),
                       ctx->stream, c0, c1, dr, seed,
                       h, p.lx, cs);
  });
  HAMX_HIP(ctx, hipGetLastError());
  FftAxis ax{};
  ax.s = ax.inner = h.nz;
  ax.outer = static_cast<uint64_t>(h.ny) * h.nz;
  ax.lines = static_cast<uint64_t>(h.nx) * h.nz;
  const uint64_t zlines = static_cast<uint64_t>(h.nx) * h.ny;
  double2 *const arr[3] = {c0, c1, nullptr};
  uint32_t np = 0;
  double *part;
  HAMX_TRY(fft_strided_var(ctx, arr, Draw::NL, p.ly, ax, zlines / 2, &part, &np));
  const double2 *rest = zlines % 2 ? c0 + zlines / 2 * h.nz : nullptr;
  with_tile(2048, p.lz.mode, [&](auto, auto, auto M) {
    hipLaunchKernelGGL((k_var_half<decltype(M)::value>), dim3(1), dim3(1024),
                       fft_lds_bytes(p.lz, 1, 2048), ctx->stream, part, np, rest, p.lz,
                       static_cast<double>(dr.a.b.n), red);
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

// z(+), rescale, even part, z(-) of Brnd_es.
template <bool SPLIT>
int half_mid(hamx_ctx *ctx, const HalfPlan &p, const double2 *c0, const double2 *c1,
             const HalfArrays &H, const EsArgs &a, const double *var) {
  uint32_t cl;
  const uint32_t tile = p.z_tile(4, p.h.lines, &cl);
  const uint32_t tables = SPLIT ? p.lz.n * sizeof(EsZ) + (2u << cl) * sizeof(EsLine) : 0;
  with_tile(tile, p.lz.mode, [&](auto T, auto NT, auto M) {
    hipLaunchKernelGGL((k_es_mid<SPLIT, decltype(T)::value, decltype(NT)::value,
                                 decltype(M)::value>),
                       dim3((p.h.lines + (1u << cl) - 1) >> cl), dim3(decltype(NT)::value),
                       fft_lds_bytes(p.lz, (4u << cl) + 1, tile) + tables, ctx->stream, c0, c1,
                       H, a, var,
                       p.h, p.lz, cl);
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

// The passes along x of the half arrays.
inline int half_gs_x(hamx_ctx *ctx, const HalfPlan &p, const HalfArrays &H, const EsArgs &a) {
  HalfArgs h = p.h;
  h.ncol = h.ny * h.nh;
  uint32_t cs;
  const uint32_t tile = p.x_tile(2, h.ncol, &cs);
  with_tile(tile, p.lx.mode, [&](auto T, auto NT, auto M) {
    hipLaunchKernelGGL((k_es_gs_x<decltype(T)::value, decltype(NT)::value, decltype(M)::value>),
                       dim3(xcd_grid((h.ncol + (1u << cs) - 1) >> cs)), dim3(decltype(NT)::value),
                       fft_lds_bytes(p.lx, 2u << cs, tile) + p.lx.n * sizeof(double),
                       ctx->stream, H, a, h, p.lx, cs);
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

inline int half_mhd_x(hamx_ctx *ctx, const HalfPlan &p, const HalfArrays &H, const MhdArgs &a,
                      uint64_t seed, const double *bobs) {
  HalfArgs h = p.h;
  h.ncol = h.ny * h.nh;
  uint32_t cs;
  const uint32_t tile = p.x_tile(2, h.ncol, &cs);
  with_tile(tile, p.lx.mode, [&](auto T, auto NT, auto M) {
    hipLaunchKernelGGL((k_mhd_x<decltype(T)::value, decltype(NT)::value, decltype(M)::value>),
                       dim3(xcd_grid((h.ncol + (1u << cs) - 1) >> cs)), dim3(decltype(NT)::value),
                       fft_lds_bytes(p.lx, 2u << cs, tile) + p.lx.n * sizeof(double),
                       ctx->stream, H, a, seed, bobs, h, p.lx, cs);
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

// z(+) and rescale of TErnd_dft.
inline int half_te_out(hamx_ctx *ctx, const HalfPlan &p, const double2 *tk, double *te,
                       const DftArgs &a, bool split, const double *var) {
  const uint32_t lines = p.h.nx * p.h.ny;
  uint32_t cl;
  const uint32_t tile = p.z_tile(1, lines, &cl);
  const uint32_t tables = split ? (p.lz.n + (1u << cl)) * sizeof(double) : 0;
  with_tile(tile, p.lz.mode, [&](auto T, auto NT, auto M) {
    auto launch = [&](auto S) {
      hipLaunchKernelGGL((k_te_out<decltype(S)::value, decltype(T)::value, decltype(NT)::value,
                                   decltype(M)::value>),
                         dim3((lines + (1u << cl) - 1) >> cl), dim3(decltype(NT)::value),
                         fft_lds_bytes(p.lz, (1u << cl) + 1, tile) + tables, ctx->stream, tk, te,
                         a, var, p.h, lines, p.lz, cl);
    };
    if (split)
      launch(std::true_type{});
    else
      launch(std::false_type{});
  });
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

} // namespace hamx
