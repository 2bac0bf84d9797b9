// Runtime-size mixed-radix FFTs for gfx950.
//
// The fused step kernels are compiled per transform size (powers of two and
// the two small mixed-radix sizes 48 and 50). Every other grid size the
// reference accepts (_spectral.py:614-721 takes any N: odd N, 100, 513, ...)
// runs through the passes below: a workgroup stages `lpb` lines side by side
// in LDS and runs the self-sorting Stockham passes of a factorisation
// n = R_1 ... R_m (Govindaraju et al., "High performance discrete Fourier
// transforms on graphics processors", SC 2008; gfft.hpp). The twiddles index
// one table of the n-th roots of unity (formed in double precision, rounded
// once), in LDS when it fits. Radices up to 16 (and 17, 19) are register
// butterflies; any other radix (a prime factor above the largest pass) is a
// direct-sum pass, so every n factors.
//
// What bounds it: LDS traffic and instruction issue, not memory (four fields
// of eight 513^2 grids along y: 67 MB in and out, 45 MB of it inside the
// cutoff). Real lines run two per complex transform where they are neighbouring
// rows of one field; divisions by runtime sizes are float multiplications, and
// 64-bit ones are made once per line; the lines of a workgroup share their
// twiddle reads and lie side by side at an odd pitch.
// Measured (eight 513^2 fields, one transform along one axis): forward lines
// 14 us, inverse lines 13 us, r2c 14 us, c2r 12 us (16 and 15 us with a row's
// start divided out at every point), against 33, 33, 42 and 43 us with one real
// line per transform, R^2 complex products per radix-R butterfly and integer
// divisions; a prime pass of 199 points (N = 597, one step of 100 trajectories)
// 60 us per step against 185 us with direct sums.
#include <cstdio>

#include "gfft.hpp"

namespace exmi {

struct GfftArgs {
  GfftDev d;
  int lpb;
  GfftLines g;
  long long nrun;  // lines (C2C), or complex lines of one or two real lines
  const void* in;
  void* out;
  float scale;
  const cf* tw;
};

template <int MODE, int RMAX, bool TWL>
__global__ void __launch_bounds__(GFFT_WG) gfft_kernel(GfftArgs a) {
  extern __shared__ cf gfft_smem[];
  __shared__ long long b0[GFFT_MAX_LINES], b1[GFFT_MAX_LINES];
  __shared__ int two[GFFT_MAX_LINES];
  constexpr bool INV = MODE == GFFT_INV || MODE == GFFT_C2R;
  constexpr bool REAL = MODE == GFFT_R2C || MODE == GFFT_C2R;
  const int n = a.d.n, nz = n / 2 + 1, tid = threadIdx.x;
  const long long run0 = (long long)(REAL ? blockIdx.x : xcd_block()) * a.lpb;
  const int L = (int)(a.nrun - run0 < a.lpb ? a.nrun - run0 : a.lpb);
  const int pitch = REAL ? gfft_pitch(a.lpb) : gfft_pitch_by_point(n, a.lpb);
  cf* A = gfft_smem;
  cf* B = gfft_smem + n * pitch;
  // TWL: the twiddle table is staged in LDS (it fits beside the two line buffers)
  const cf* T = TWL ? gfft_smem + 2 * n * pitch : a.tw;
  if constexpr (TWL)
    for (int i = tid; i < n; i += GFFT_WG) gfft_smem[2 * n * pitch + i] = a.tw[i];
  // where each line starts: C2C b0; real lines: its first row in the real
  // array b0 and in the complex one b1, and whether the row behind it is the
  // line's second (one of the same field, so right behind it in both arrays)
  if (tid < L) {
    const long long run = run0 + tid;
    if constexpr (REAL) {
      const long long per = (a.g.rows + 1) / 2, f = run / per, q = run - f * per;
      const long long row = f * a.g.rows + 2 * q;
      b0[tid] = a.g.rpg > 0 ? (row / a.g.rpg) * a.g.gstride + (row % a.g.rpg) * n : row * n;
      b1[tid] = row * nz;
      two[tid] = 2 * q + 1 < a.g.rows;
    } else {
      const int mk = gfft_midkeep(a.g.midn, a.g.cut);
      const long long r = run / a.g.kkeep, o = r / mk;
      b0[tid] = o * a.g.outer_stride + (long long)gfft_kept((int)(r - o * mk), mk, a.g.midn) * a.g.nz + run % a.g.kkeep;
    }
  }
  __syncthreads();
  const float rL = 1.f / (float)L, rn = a.d.rn, rnz = 1.f / (float)nz;
  // load: consecutive threads read consecutive addresses (along the line for
  // contiguous lines, across neighbouring lines for a strided axis)
  if constexpr (MODE == GFFT_R2C) {
    const float* in = static_cast<const float*>(a.in);
    for (int idx = tid; idx < L * n; idx += GFFT_WG) {
      const int ll = fdiv(idx, rn), pt = idx - ll * n;
      const float* x = in + b0[ll] + pt;
      A[pt * pitch + ll] = cf{x[0], two[ll] ? x[n] : 0.f};
    }
  } else if constexpr (MODE == GFFT_C2R) {
    const cf* in = static_cast<const cf*>(a.in);
    for (int idx = tid; idx < L * nz; idx += GFFT_WG) {
      const int ll = fdiv(idx, rnz), k = idx - ll * nz;
      const cf* x = in + b1[ll] + k;
      cf p = x[0], q = two[ll] ? x[nz] : cf{0.f, 0.f};
      const bool self = k == 0 || 2 * k == n;
      if (self) p.im = q.im = 0.f;
      A[k * pitch + ll] = cf{p.re - q.im, p.im + q.re};
      if (!self) A[(n - k) * pitch + ll] = cf{p.re + q.im, q.re - p.im};
    }
  } else {
    const cf* in = static_cast<const cf*>(a.in);
    for (int idx = tid; idx < L * n; idx += GFFT_WG) {
      const int pt = fdiv(idx, rL), ll = idx - pt * L;
      const bool zero = INV && a.g.pcut >= 0 && pt > a.g.pcut && n - pt > a.g.pcut;
      A[pt * pitch + ll] = zero ? cf{0.f, 0.f} : in[b0[ll] + pt * a.g.pstride];
    }
  }
  __syncthreads();
  const cf* Z = gfft_run<INV, RMAX>(A, B, T, a.d, L, pitch, tid, GFFT_WG);
  // store
  if constexpr (MODE == GFFT_R2C) {
    cf* out = static_cast<cf*>(a.out);
    for (int idx = tid; idx < L * nz; idx += GFFT_WG) {
      const int ll = fdiv(idx, rnz), k = idx - ll * nz;
      const cf zk = Z[k * pitch + ll];
      cf* x = out + b1[ll] + k;
      if (!two[ll]) {
        x[0] = zk;
      } else {
        cf p, q;
        unpack_pair(zk, Z[(k == 0 ? 0 : n - k) * pitch + ll], p, q);
        x[0] = p;
        x[nz] = q;
      }
    }
  } else if constexpr (MODE == GFFT_C2R) {
    float* out = static_cast<float*>(a.out);
    for (int idx = tid; idx < L * n; idx += GFFT_WG) {
      const int ll = fdiv(idx, rn), pt = idx - ll * n;
      const cf v = Z[pt * pitch + ll];
      float* x = out + b0[ll] + pt;
      x[0] = a.scale * v.re;
      if (two[ll]) x[n] = a.scale * v.im;
    }
  } else {
    cf* out = static_cast<cf*>(a.out);
    for (int idx = tid; idx < L * n; idx += GFFT_WG) {
      const int pt = fdiv(idx, rL), ll = idx - pt * L;
      if (!INV && a.g.pcut >= 0 && pt > a.g.pcut && n - pt > a.g.pcut) continue;
      out[b0[ll] + pt * a.g.pstride] = a.scale * Z[pt * pitch + ll];
    }
  }
}

GfftDev gfft_dev(const GfftCfg& c, bool reversed) {
  GfftDev d;
  d.n = c.n;
  d.npass = c.npass;
  d.rn = 1.f / (float)c.n;
  int Ns = 1;
  for (int i = 0; i < c.npass; ++i) {
    GfftPass& p = d.p[i];
    p.R = c.radix[reversed ? c.npass - 1 - i : i];
    p.Ns = Ns;
    p.m = c.n / p.R;
    p.tws = c.n / (Ns * p.R);
    p.rNs = 1.f / (float)Ns;
    Ns *= p.R;
  }
  return d;
}

bool gfft_big(const GfftCfg& c) {
  bool big = false;  // a pass of radix 9..17 or 19 to run as register butterflies
  for (int i = 0; i < c.npass; ++i) big = big || (c.radix[i] > 8 && (c.radix[i] <= 17 || c.radix[i] == 19));
  return big && c.reg19;
}

bool gfft_make_cfg(int n, int max_radix, int points_per_wg, GfftCfg* cfg) {
  if (n < 2 || n > GFFT_MAX_N || max_radix < 2) return false;
  // The best factorisation of every divisor of n (at most 48 of them up to
  // 4096), from those of the smaller ones: fewest passes, then the smallest sum
  // of radices. A standalone transform plans on each call, so the loops run
  // over divisors only and nothing is allocated: 0.7 us at n = 3000, where
  // trying every number up to n took 28 us, twice the transform's own time.
  int div[64], nd = 0;
  for (int f = 1; f * f <= n; ++f)
    if (n % f == 0) div[nd++] = f;
  for (int i = nd - 1; i >= 0; --i)
    if (div[i] * div[i] != n) div[nd++] = n / div[i];
  short at[GFFT_MAX_N + 1];  // index of a divisor
  int rad[64], nr = 0;       // the divisors that can be a pass: up to max_radix, or prime
  int passes[64], sum[64], last[64];
  passes[0] = sum[0] = last[0] = 0;
  at[1] = 0;
  for (int i = 1; i < nd; ++i) {
    const int d = div[i];
    at[d] = (short)i;
    bool prime = true;
    for (int j = 1; j < i && prime; ++j) prime = d % div[j] != 0;
    if (d <= max_radix || prime) rad[nr++] = d;
    passes[i] = sum[i] = 1 << 20;
    for (int k = 0; k < nr; ++k) {
      const int r = rad[k];
      if (d % r) continue;
      const int q = at[d / r], np = passes[q] + 1, ns = sum[q] + r;
      if (np < passes[i] || (np == passes[i] && ns < sum[i])) {
        passes[i] = np;
        sum[i] = ns;
        last[i] = r;
      }
    }
  }
  if (passes[nd - 1] > GFFT_MAX_PASS) return false;
  GfftCfg c;
  c.n = n;
  // the radices without a register butterfly first (see gfft_pass_direct)
  for (int big = 1; big >= 0; --big)
    for (int d = n; d > 1; d /= last[at[d]])
      if ((last[at[d]] > 19) == (big == 1)) c.radix[c.npass++] = last[at[d]];
  const int lpb = points_per_wg / n;
  c.lpb = lpb < 1 ? 1 : lpb > GFFT_MAX_LINES ? GFFT_MAX_LINES : lpb;
  // two line buffers stay within 64 KiB of LDS (less the line starts)
  while (c.lpb > 1 && sizeof(cf) * 2 * n * gfft_pitch(c.lpb) > GFFT_LDS_MAX - 2048) --c.lpb;
  *cfg = c;
  return true;
}

static const int k_gfft_cands[] = {8 * 100000 + 512,   8 * 100000 + 1024,
                                   8 * 100000 + 2048,  8 * 100000 + 4096,
                                   100000000 + 10 * 100000 + 1024, 100000000 + 10 * 100000 + 2048,
                                   100000000 + 16 * 100000 + 512,  100000000 + 16 * 100000 + 1024,
                                   100000000 + 16 * 100000 + 2048, 100000000 + 16 * 100000 + 4096,
                                   100000000 + 8 * 100000 + 1024,  100000000 + 8 * 100000 + 2048,
                                   100000000 + 8 * 100000 + 256,   100000000 + 8 * 100000 + 768};
int gfft_num_candidates() { return (int)(sizeof k_gfft_cands / sizeof k_gfft_cands[0]); }
int gfft_candidate(int i) { return k_gfft_cands[i]; }
int gfft_default_code() { return 100000000 + 8 * 100000 + 2048; }
bool gfft_cfg_from_code(int n, int code, GfftCfg* cfg) {
  const int flag = code / 100000000, max_radix = (code / 100000) % 1000;
  if (code <= 100000 || flag > 1 || !gfft_make_cfg(n, max_radix, code % 100000, cfg)) return false;
  cfg->reg19 = flag;
  return true;
}

hipError_t launch_gfft(const GfftCfg& c, int mode, const void* in, void* out, const GfftLines& g, float scale,
                       const cf* tw, hipStream_t st) {
  const bool real = mode == GFFT_R2C || mode == GFFT_C2R;
  if ((real ? g.nlines : g.nouter) <= 0) return hipSuccess;
  if (c.n < 2 || c.n > GFFT_MAX_N || c.lpb < 1 || c.lpb > GFFT_MAX_LINES) return hipErrorInvalidValue;
  GfftArgs a;
  a.d = gfft_dev(c);
  a.lpb = c.lpb;
  a.g = g;
  a.in = in;
  a.out = out;
  a.scale = scale;
  a.tw = tw;
  if (real) {
    if (g.rows < 1 || g.nlines % g.rows) return hipErrorInvalidValue;
    a.nrun = g.nlines / g.rows * ((g.rows + 1) / 2);
  } else {
    if (g.kkeep < 1 || g.kkeep > g.nz || g.midn < 1) return hipErrorInvalidValue;
    a.nrun = g.nouter * gfft_midkeep(g.midn, g.cut) * g.kkeep;
  }
  const long long grid = (a.nrun + c.lpb - 1) / c.lpb;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const size_t buf = sizeof(cf) * 2 * (size_t)c.n * (real ? gfft_pitch(c.lpb) : gfft_pitch_by_point(c.n, c.lpb));
  const size_t fixed = 20 * GFFT_MAX_LINES;
  size_t lds = buf + sizeof(cf) * (size_t)c.n;
  const bool twl = lds + fixed <= GFFT_LDS_MAX;
  if (!twl) lds = buf;
  const bool big = gfft_big(c);
#define EXMI_GFFT_LAUNCH(M)                                                                     \
  hipLaunchKernelGGL((big ? (twl ? gfft_kernel<M, 19, true> : gfft_kernel<M, 19, false>)        \
                          : (twl ? gfft_kernel<M, 8, true> : gfft_kernel<M, 8, false>)),        \
                     dim3((unsigned)grid), dim3(GFFT_WG), lds, st, a);
  switch (mode) {
    case GFFT_FWD: EXMI_GFFT_LAUNCH(GFFT_FWD) break;
    case GFFT_INV: EXMI_GFFT_LAUNCH(GFFT_INV) break;
    case GFFT_R2C: EXMI_GFFT_LAUNCH(GFFT_R2C) break;
    case GFFT_C2R: EXMI_GFFT_LAUNCH(GFFT_C2R) break;
    default: return hipErrorInvalidValue;
  }
#undef EXMI_GFFT_LAUNCH
  return hipGetLastError();
}

}  // namespace exmi
