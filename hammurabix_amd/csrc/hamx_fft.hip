// In-place 3D complex128 FFT for gfx950: one kernel launch per axis, each
// workgroup transforming a tile of C lines held in LDS (the engine of
// hamx_fft.h).  Unnormalised, exponent sign * 2 pi i jk / n: sign = +1 is the
// reference's FFTW_BACKWARD plan, -1 its FFTW_FORWARD plan
// (grid_brnd.cc:42-54, grid_ternd.cc:35-37).  FFTW plans any length; so does
// this file (2^a 3^b 5^c 7^d up to 8192, any other length up to 4096).
//
// Along the contiguous z axis each line is a contiguous run of memory; along
// y and x the tile's C lines are C adjacent columns, so every tile row is
// C * 16 contiguous bytes.  Twiddles and chirps come from per-length tables
// computed on the host in long double.
#include <hip/hip_runtime.h>

#include <cmath>
#include <complex>
#include <cstring>
#include <map>
#include <tuple>
#include <vector>

#include "hamx_fft.h"
#include "hamx_internal.h"

namespace hamx {

struct FftArrays {
  double2 *p[3];
};

// Partial sums of the random fields' variance (hamx_rnd_half.h): the first
// `nfull` z lines of the first array count, line i ny + j being point j of
// the columns (i, .); `part` holds four doubles per workgroup.
struct FftVar {
  double *part;
  uint64_t nfull;
};

// Sums over the NT threads of a workgroup, the result in every thread.
template <uint32_t NT>
__device__ inline void block_sums(double &a, double &b, double &c) {
  __shared__ double sm[3][NT / 64];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    a += __shfl_xor(a, o, 64);
    b += __shfl_xor(b, o, 64);
    c += __shfl_xor(c, o, 64);
  }
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    sm[0][w] = a;
    sm[1][w] = b;
    sm[2][w] = c;
  }
  __syncthreads();
  a = b = c = 0.;
  for (uint32_t i = 0; i < NT / 64; ++i) {
    a += sm[0][i];
    b += sm[1][i];
    c += sm[2][i];
  }
}

// A tile of C lines, points ax.s apart (CONTIG false: C adjacent columns) or
// contiguous (CONTIG true: one run of C n elements).  blockIdx.y picks the
// array.  A thread issues all of its loads (at most TILE / NT = 8) before it
// waits for the first.  VAR (strided axis) also writes the variance's partial
// sums over the first array: the k = 0 columns' mean, count and squared
// deviations, and the other columns' sum of squares.
template <int SIGN, uint32_t TILE, uint32_t NT, int MODE, bool CONTIG, bool VAR>
__global__ __launch_bounds__(NT) void k_fft_axis(FftArrays arr, FftAxis ax, FftLine L,
                                                 FastDiv dn, FftVar var) {
  extern __shared__ double2 lds[];
  constexpr uint32_t K = TILE / NT;
  double2 *__restrict__ data = arr.p[blockIdx.y];
  const uint32_t n = L.n, cs = ax.cshift, C = 1u << cs, P = ax.P;
  const uint32_t tile = CONTIG ? blockIdx.x : xcd_tile(blockIdx.x, gridDim.x);
  const uint64_t L0 = static_cast<uint64_t>(tile) << cs;
  if (L0 >= ax.lines)
    return; // uniform: the grid's last few workgroups
  const double2 *twl = fft_tables<TILE, NT, MODE>(lds, L, P);
  const uint64_t left = ax.lines - L0; // lines of this tile that exist (>= 1)
  const uint32_t total = C * n;
  if constexpr (CONTIG) {
    const uint32_t valid = static_cast<uint32_t>(left < C ? left : C) * n;
    double2 *__restrict__ run = data + L0 * n;
    double2 v[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t e = threadIdx.x + NT * k;
      v[k] = e < valid ? run[e] : make_double2(0., 0.);
    }
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t e = threadIdx.x + NT * k;
      if (e < total) {
        const uint32_t c = fast_quot(dn, e);
        lds[(e - c * n) * P + c] = v[k];
      }
    }
    __syncthreads();
    fft_lines<SIGN, TILE, NT, MODE>(lds, twl, L, cs, P);
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t e = threadIdx.x + NT * k;
      if (e < valid) {
        const uint32_t c = fast_quot(dn, e);
        run[e] = lds[(e - c * n) * P + c];
      }
    }
  } else {
    // NT is a multiple of C, so a thread stays on one column
    const uint32_t c = threadIdx.x & (C - 1), t0 = threadIdx.x >> cs, dt = NT >> cs;
    const bool on = c < left;
    double2 *__restrict__ col = data + (on ? line_base(ax, L0 + c) : 0);
    double2 v[K];
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t t = t0 + dt * k;
      v[k] = on && t < n ? col[t * ax.s] : make_double2(0., 0.);
    }
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t t = t0 + dt * k;
      if (t < n)
        lds[t * P + c] = v[k];
    }
    __syncthreads();
    fft_lines<SIGN, TILE, NT, MODE>(lds, twl, L, cs, P);
#pragma unroll
    for (uint32_t k = 0; k < K; ++k) {
      const uint32_t t = t0 + dt * k;
      if (on && t < n)
        col[t * ax.s] = lds[t * P + c];
    }
    if constexpr (VAR) {
      if (blockIdx.y != 0)
        return;
      const uint64_t i = (L0 + c) / ax.inner;
      const bool dc = (L0 + c) - i * ax.inner == 0;
      const uint32_t lines =
          !on || i * n >= var.nfull ? 0
          : var.nfull - i * n < n   ? static_cast<uint32_t>(var.nfull - i * n)
                                    : n;
      double sum = 0., cnt = 0., e = 0.;
      for (uint32_t t = t0; t < lines; t += dt) {
        const double2 v = lds[t * P + c];
        if (dc) {
          sum += v.x + v.y;
          cnt += 2.;
        } else {
          e += v.x * v.x + v.y * v.y;
        }
      }
      block_sums<NT>(sum, cnt, e);
      const double mean = cnt > 0. ? sum / cnt : 0.;
      double m2 = 0., z0 = 0., z1 = 0.;
      if (cnt > 0.) { // uniform
        for (uint32_t t = t0; dc && t < lines; t += dt) {
          const double2 v = lds[t * P + c];
          m2 += (v.x - mean) * (v.x - mean) + (v.y - mean) * (v.y - mean);
        }
        block_sums<NT>(m2, z0, z1);
      }
      if (threadIdx.x == 0) {
        double *p = var.part + 4 * static_cast<uint64_t>(tile);
        p[0] = mean;
        p[1] = cnt;
        p[2] = m2;
        p[3] = e;
      }
    }
  }
}

// ------------------------------------------------------------------ host --
namespace {

using cld = std::complex<long double>;
const long double kTwoPiL = 6.283185307179586476925286766559005768394L;

// Stockham plan of n: radix 4 and 8, then 3, 5, 7.
bool make_plan(uint32_t n, FftPlan &pl) {
  std::memset(&pl, 0, sizeof(pl));
  pl.n = n;
  uint32_t m = n, p = 1;
  auto push = [&](uint32_t r) {
    if (pl.npass >= kMaxPass)
      return false;
    FftPass &ps = pl.pass[pl.npass++];
    ps.radix = static_cast<uint16_t>(r);
    ps.p = static_cast<uint16_t>(p);
    ps.q = static_cast<uint16_t>(n / r);
    ps.tstep = static_cast<uint16_t>(n / (r * p));
    ps.inv_p = 1.0f / static_cast<float>(p);
    m /= r;
    p *= r;
    return true;
  };
  // the power of two in the fewest passes of radix 8 and 4 (2 alone as 2)
  int e = 0;
  while (m % (2u << e) == 0)
    ++e;
  if (e == 1 && !push(2))
    return false;
  for (int fours = (3 - e % 3) % 3; e > 1; --fours) {
    const bool four = fours > 0;
    if (!push(four ? 4u : 8u))
      return false;
    e -= four ? 2 : 3;
  }
  for (uint32_t r : {3u, 5u, 7u})
    while (m % r == 0)
      if (!push(r))
        return false;
  return m == 1;
}

// Device tables cached per context: kind 0 = twiddles exp(2 pi i m / n),
// kinds 1 and 2 = Bluestein chirp and kernel transform of exponent +1.
std::map<std::tuple<hamx_ctx *, uint64_t, int>, double2 *> g_tables;

int upload(hamx_ctx *ctx, const std::vector<double2> &h, std::tuple<hamx_ctx *, uint64_t, int> key,
           const double2 **out) {
  double2 *d = nullptr;
  HAMX_HIP(ctx, hipMalloc(&d, h.size() * sizeof(double2)));
  HAMX_HIP(ctx, hipMemcpy(d, h.data(), h.size() * sizeof(double2), hipMemcpyHostToDevice));
  g_tables[key] = d;
  *out = d;
  return HAMX_OK;
}

int twiddle_table(hamx_ctx *ctx, uint64_t n, const double2 **out) {
  auto key = std::make_tuple(ctx, n, 0);
  auto it = g_tables.find(key);
  if (it != g_tables.end()) {
    *out = it->second;
    return HAMX_OK;
  }
  std::vector<double2> h(n);
  for (uint64_t m = 0; m < n; ++m) {
    const long double a = kTwoPiL * static_cast<long double>(m) / static_cast<long double>(n);
    h[m] = make_double2(static_cast<double>(cosl(a)), static_cast<double>(sinl(a)));
  }
  return upload(ctx, h, key, out);
}

// In-place radix-2 transform of a power-of-two length, exponent sign (host,
// long double; for the Bluestein kernel table only).
void host_fft_pow2(std::vector<cld> &a, int sign) {
  const size_t n = a.size();
  for (size_t i = 1, j = 0; i < n; ++i) {
    size_t bit = n >> 1;
    for (; j & bit; bit >>= 1)
      j ^= bit;
    j ^= bit;
    if (i < j)
      std::swap(a[i], a[j]);
  }
  for (size_t len = 2; len <= n; len <<= 1) {
    for (size_t k = 0; k < len / 2; ++k) {
      const long double ang = sign * kTwoPiL * static_cast<long double>(k) /
                              static_cast<long double>(len);
      const cld w(cosl(ang), sinl(ang));
      for (size_t s = 0; s < n; s += len) {
        const cld u = a[s + k], v = a[s + k + len / 2] * w;
        a[s + k] = u + v;
        a[s + k + len / 2] = u - v;
      }
    }
  }
}

int bluestein_tables(hamx_ctx *ctx, uint64_t n, uint64_t M, const double2 **chirp,
                     const double2 **bhat) {
  auto kchirp = std::make_tuple(ctx, n, 1), kbhat = std::make_tuple(ctx, n, 2);
  auto ic = g_tables.find(kchirp), ib = g_tables.find(kbhat);
  if (ic != g_tables.end() && ib != g_tables.end()) {
    *chirp = ic->second;
    *bhat = ib->second;
    return HAMX_OK;
  }
  // c_j = exp(i pi (j^2 mod 2n) / n): the reduction keeps the angle exact
  std::vector<cld> c(n);
  for (uint64_t j = 0; j < n; ++j) {
    const uint64_t r = (j * j) % (2 * n);
    const long double a = (kTwoPiL / 2) * static_cast<long double>(r) / static_cast<long double>(n);
    c[j] = cld(cosl(a), sinl(a));
  }
  std::vector<cld> b(M, cld(0, 0));
  b[0] = std::conj(c[0]);
  for (uint64_t j = 1; j < n; ++j)
    b[j] = b[M - j] = std::conj(c[j]);
  host_fft_pow2(b, -1);
  std::vector<double2> hc(n), hb(M);
  for (uint64_t j = 0; j < n; ++j)
    hc[j] = make_double2(static_cast<double>(c[j].real()), static_cast<double>(c[j].imag()));
  for (uint64_t j = 0; j < M; ++j)
    hb[j] = make_double2(static_cast<double>(b[j].real()), static_cast<double>(b[j].imag()));
  HAMX_TRY(upload(ctx, hc, kchirp, chirp));
  return upload(ctx, hb, kbhat, bhat);
}

uint64_t next_pow2(uint64_t v) {
  uint64_t p = 1;
  while (p < v)
    p <<= 1;
  return p;
}

} // namespace

void release_twiddles(hamx_ctx *ctx) {
  for (auto it = g_tables.begin(); it != g_tables.end();) {
    if (std::get<0>(it->first) == ctx) {
      (void)hipFree(it->second);
      it = g_tables.erase(it);
    } else {
      ++it;
    }
  }
}

bool fft_length_ok(uint64_t n) {
  FftPlan pl;
  if (n >= 1 && n <= kTileMax && make_plan(static_cast<uint32_t>(n), pl))
    return true;
  return n >= 1 && n <= kTileMax / 2;
}

int fft_line(hamx_ctx *ctx, uint64_t n, FftLine *out) {
  FftLine &L = *out;
  std::memset(&L, 0, sizeof(L));
  L.n = L.len = static_cast<uint32_t>(n);
  if (make_plan(L.n, L.plan)) {
    L.mode = is_pow2(n) ? kFftPow2 : kFftMixed;
  } else {
    L.mode = kFftBlue;
    L.len = static_cast<uint32_t>(next_pow2(2 * n - 1));
    make_plan(L.len, L.plan);
    HAMX_TRY(bluestein_tables(ctx, n, L.len, &L.chirp, &L.bhat));
  }
  return twiddle_table(ctx, L.len, &L.tw);
}

uint32_t fft_cshift(uint32_t tile, uint32_t len, uint32_t most, uint64_t lines) {
  uint32_t cs = 0;
  while (cs < most && (len << (cs + 1)) <= tile && (1ull << cs) < lines)
    ++cs;
  return cs;
}

namespace {

template <int SIGN, uint32_t TILE, uint32_t NT, int MODE, bool CONTIG, bool VAR>
int launch_axis(hamx_ctx *ctx, const FftArrays &arr, unsigned arrays, const FftLine &L,
                const FftAxis &ax, const FftVar &var) {
  const uint64_t tiles = (ax.lines + (1ull << ax.cshift) - 1) >> ax.cshift;
  hipLaunchKernelGGL((k_fft_axis<SIGN, TILE, NT, MODE, CONTIG, VAR>),
                     dim3(CONTIG ? static_cast<unsigned>(tiles) : xcd_grid(tiles), arrays), dim3(NT),
                     fft_lds_bytes(L, ax.P, TILE), ctx->stream, arr, ax, L, fast_div(L.n), var);
  HAMX_HIP(ctx, hipGetLastError());
  return HAMX_OK;
}

template <int SIGN, uint32_t TILE, uint32_t NT, bool CONTIG, bool VAR>
int launch_mode(hamx_ctx *ctx, const FftArrays &arr, unsigned arrays, const FftLine &L,
                const FftAxis &ax, const FftVar &var) {
  switch (L.mode) {
  case kFftPow2:
    return launch_axis<SIGN, TILE, NT, kFftPow2, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
  case kFftMixed:
    return launch_axis<SIGN, TILE, NT, kFftMixed, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
  default:
    return launch_axis<SIGN, TILE, NT, kFftBlue, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
  }
}

// The tile: 2048 values (32 KB of LDS) for lines of up to 2048 points along
// the contiguous axis; along the strided axes the smallest one up to 4096
// values that holds eight columns (128-byte rows), else four, else what fits.
uint32_t axis_tile(const FftLine &L, bool contig, FftAxis &ax) {
  const uint32_t want = contig ? L.len : (8 * L.len <= 4096 ? 8 : 4) * L.len;
  uint32_t tile = want <= 2048 ? 2048 : 4096;
  if (L.len > tile || (!contig && 2 * L.len > tile))
    tile = kTileMax;
  ax.cshift = fft_cshift(tile, L.len, contig ? 11 : 4, ax.lines);
  const uint32_t C = 1u << ax.cshift;
  ax.P = contig && C >= 4 ? C + 1 : C;
  return tile;
}

template <int SIGN, bool CONTIG, bool VAR>
int launch_tile(hamx_ctx *ctx, const FftArrays &arr, unsigned arrays, const FftLine &L,
                FftAxis ax, const FftVar &var) {
  const uint32_t tile = axis_tile(L, CONTIG, ax);
  if (tile == 2048)
    return launch_mode<SIGN, 2048, 256, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
  if (tile == 4096)
    return launch_mode<SIGN, 4096, 512, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
  return launch_mode<SIGN, kTileMax, 1024, CONTIG, VAR>(ctx, arr, arrays, L, ax, var);
}

} // namespace

int fft_strided(hamx_ctx *ctx, double2 *const data[3], unsigned arrays, const FftLine &L,
                FftAxis ax, int sign) {
  const FftArrays arr{{data[0], data[1], data[2]}};
  return sign > 0 ? launch_tile<1, false, false>(ctx, arr, arrays, L, ax, FftVar{})
                  : launch_tile<-1, false, false>(ctx, arr, arrays, L, ax, FftVar{});
}

int fft_strided_var(hamx_ctx *ctx, double2 *const data[3], unsigned arrays, const FftLine &L,
                    FftAxis ax, uint64_t nfull, double **part, uint32_t *np) {
  const FftArrays arr{{data[0], data[1], data[2]}};
  (void)axis_tile(L, false, ax);
  *np = static_cast<uint32_t>((ax.lines + (1ull << ax.cshift) - 1) >> ax.cshift);
  void *w;
  HAMX_TRY(ws_get(ctx, kSlotRndPart, 4 * static_cast<size_t>(*np) * sizeof(double), &w));
  *part = static_cast<double *>(w);
  return launch_tile<1, false, true>(ctx, arr, arrays, L, ax, FftVar{*part, nfull});
}

int fft3d_dev(hamx_ctx *ctx, double2 *data, uint64_t nx, uint64_t ny,
              uint64_t nz, int sign) {
  return fft3d_dev2(ctx, data, nullptr, nx, ny, nz, sign);
}

int fft3d_dev2(hamx_ctx *ctx, double2 *data, double2 *data2, uint64_t nx, uint64_t ny,
               uint64_t nz, int sign) {
  const FftArrays arr{{data, data2, nullptr}};
  const unsigned arrays = data2 ? 2u : 1u;
  const uint64_t dims[3] = {nx, ny, nz};
  for (int a = 0; a < 3; ++a)
    if (!fft_length_ok(dims[a]))
      return set_err(ctx, HAMX_ERR_UNSUPPORTED,
                     "FFT axis length %llu: lengths of the form 2^a 3^b 5^c 7^d up to %u "
                     "and any other length up to %u are supported",
                     static_cast<unsigned long long>(dims[a]), kTileMax, kTileMax / 2);
  const uint64_t total = nx * ny * nz;
  // axis order z, y, x (any order gives the same transform)
  for (int a = 2; a >= 0; --a) {
    const uint64_t n = dims[a];
    if (n < 2)
      continue;
    FftLine L;
    HAMX_TRY(fft_line(ctx, n, &L));
    FftAxis ax;
    std::memset(&ax, 0, sizeof(ax));
    ax.lines = total / n;
    if (a == 2) {
      HAMX_TRY(sign > 0 ? (launch_tile<1, true, false>(ctx, arr, arrays, L, ax, FftVar{}))
                        : (launch_tile<-1, true, false>(ctx, arr, arrays, L, ax, FftVar{})));
      continue;
    }
    ax.s = ax.inner = a == 1 ? nz : ny * nz;
    ax.outer = n * ax.s;
    HAMX_TRY(fft_strided(ctx, arr.p, arrays, L, ax, sign));
  }
  return HAMX_OK;
}

} // namespace hamx

using namespace hamx;

extern "C" int hamx_fft3d(hamx_ctx *ctx, double *data, uint64_t nx, uint64_t ny,
                          uint64_t nz, int sign, uint32_t flags) {
  if (!ctx)
    return HAMX_ERR_ARG;
  if (!data || (sign != 1 && sign != -1))
    return set_err(ctx, HAMX_ERR_ARG, "hamx_fft3d: null data or sign not +-1");
  HAMX_HIP(ctx, hipSetDevice(ctx->device));
  const uint64_t total = nx * ny * nz;
  const size_t bytes = total * sizeof(double2);
  double2 *d = reinterpret_cast<double2 *>(data);
  const bool in_dev = (flags & HAMX_IN_DEVICE) != 0;
  if (!in_dev) {
    void *w;
    HAMX_TRY(ws_get(ctx, kSlotFft, bytes, &w));
    HAMX_HIP(ctx, hipMemcpyAsync(w, data, bytes, hipMemcpyHostToDevice, ctx->stream));
    d = static_cast<double2 *>(w);
  }
  HAMX_TRY(fft3d_dev(ctx, d, nx, ny, nz, sign));
  if (!in_dev)
    HAMX_HIP(ctx, hipMemcpyAsync(data, d, bytes, hipMemcpyDeviceToHost, ctx->stream));
  HAMX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return HAMX_OK;
}
