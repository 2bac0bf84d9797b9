// Runtime-size mixed-radix FFTs (gfft.hip) for grid sizes outside the fused
// kernels' compile-time set: any line length 2..4096, shared with the fused
// passes of those sizes (gspec.hip) and the C-ABI layer.
#pragma once
#include "exmi_internal.hpp"
#include "fft1d.hpp"

namespace exmi {

constexpr int GFFT_MAX_N = 4096;
constexpr int GFFT_MAX_PASS = 16;
constexpr int GFFT_WG = 256;
constexpr int GFFT_MAX_LINES = 64;  // lines per workgroup
constexpr size_t GFFT_LDS_MAX = 65536;

// How a line length is transformed: the radices of the Stockham passes in
// order (their product is n) and how many lines one 256-thread workgroup
// holds in LDS. Chosen per size by the plan's autotuner (max_radix and the
// points per workgroup are the tuned knobs).
struct GfftCfg {
  int n = 0;
  int npass = 0;
  int radix[GFFT_MAX_PASS] = {};
  int lpb = 1;  // lines per workgroup
  int reg19 = 0;  // 1: radices 9..17 and 19 as register butterflies (a kernel of lower occupancy)
};

// Transforms of lines.
//  C2C (forward or inverse), along one axis of `nouter` blocks: line (o, m, z)
//      starts at o * outer_stride + m * nz + z (z < nz, m < midn) and its
//      points are pstride apart, in `in` and in `out` alike (which may be the
//      same); the result is multiplied by `scale`. What a dealias cutoff
//      makes zero or unread may be left out: only the lines with z < kkeep
//      run, and with cut >= 0 only those whose signed index m is within
//      +-cut (where midn > 1), and the points whose signed index is beyond
//      pcut are read as zero (inverse) or not stored (forward); -1: all.
//  R2C: real lines of n contiguous floats -> n/2+1 complex (contiguous).
//  C2R: n/2+1 complex (Hermitian half, Im of the DC and, for even n, the
//      Nyquist bin ignored) -> n real, multiplied by `scale`.
//  Real lines r of R2C / C2R run two per complex transform where they are
//  neighbouring rows of one field (`rows` > 1 rows per field, nlines a
//  multiple of it). With rpg > 0 real line r starts at
//  (r / rpg) * gstride + (r % rpg) * n floats, else at r * n.
enum GfftMode { GFFT_FWD = 0, GFFT_INV = 1, GFFT_R2C = 2, GFFT_C2R = 3 };

struct GfftLines {
  long long nouter = 0, outer_stride = 0, pstride = 1;
  int midn = 1, nz = 1, kkeep = 1, cut = -1, pcut = -1;
  long long nlines = 0, rows = 1, rpg = 0, gstride = 0;
};
// Lines of the middle axis that run: all, or the signed indices within +-cut.
__host__ __device__ __forceinline__ int gfft_midkeep(int midn, int cut) {
  return cut < 0 || midn == 1 || cut >= midn / 2 ? midn : 2 * cut + 1;
}
// The index of the i-th of `keep` kept entries of an axis of n.
__host__ __device__ __forceinline__ int gfft_kept(int i, int keep, int n) {
  return i < (keep + 1) / 2 ? i : i + n - keep;
}

// The fewest passes of at most max_radix points (ties: the smallest sum of
// radices) where n allows; a prime factor above max_radix is a pass of its
// own. lpb from the target number of points per workgroup. Returns false
// when n is outside 2..GFFT_MAX_N.
bool gfft_make_cfg(int n, int max_radix, int points_per_wg, GfftCfg* cfg);
// Encoded knobs (reg19 * 100000000 + max_radix * 100000 + points_per_wg) of
// the candidates the autotuner times, and the default used without tuning.
int gfft_num_candidates();
int gfft_candidate(int i);
int gfft_default_code();
bool gfft_cfg_from_code(int n, int code, GfftCfg* cfg);

hipError_t launch_gfft(const GfftCfg& c, int mode, const void* in, void* out, const GfftLines& g, float scale,
                       const cf* tw, hipStream_t st);

// ---------------------------------------------------------- device building
// The passes as the kernels take them: divisions by runtime sizes go through
// float reciprocals.
struct GfftPass {
  int R, Ns, m, tws;  // radix, product of the earlier radices, n / R, n / (Ns R)
  float rNs;
};
struct GfftDev {
  int n, npass;
  float rn;
  GfftPass p[GFFT_MAX_PASS];
};
GfftDev gfft_dev(const GfftCfg& c, bool reversed = false);
// LDS entries between the points of a line: the lines of a workgroup lie
// side by side, with an odd pitch so that neither neighbouring lines nor the
// passes' strided points share banks.
__host__ __device__ __forceinline__ int gfft_pitch(int lines) { return lines | 1; }
// The same where the lines are filled point by point, all lines of a point by
// neighbouring threads: an odd n has odd radices only, whose strides spread an
// even pitch over the banks as well, and the entry saved admits another
// workgroup to the CU (four lines of n = 513: 37 KiB, four instead of three).
__host__ __device__ __forceinline__ int gfft_pitch_by_point(int n, int lines) { return n & 1 ? lines : lines | 1; }
// Workgroups are dealt to the 8 XCDs in turn, each with an L2 of its own;
// logical block numbers that run through one XCD's workgroups first. A
// strided axis is read and written in segments of a few lines (24 bytes at
// three lines of n = 513), so the neighbours of a cache line belong to
// neighbouring workgroups, and this keeps them in one L2 (eight 513^2
// spectra: inverse lines 18.6 -> 13.3 us, the four fields' lines 33 -> 28 us).
__device__ __forceinline__ unsigned xcd_block() {
  const unsigned grid = gridDim.x, x = blockIdx.x & 7, per = grid >> 3, rem = grid & 7;
  return x * per + (x < rem ? x : rem) + (blockIdx.x >> 3);
}
// Whether a configuration runs a pass in the kernels of RMAX = 19.
bool gfft_big(const GfftCfg& c);

// x / d for 0 <= x < 2^21 and 1 <= d <= 2^21 with r = 1.f / d: x + 1/2 is
// exact, and (x + 1/2) / d keeps 1/(2d) from every integer, more than the
// product's rounding.
__device__ __forceinline__ int fdiv(int x, float r) { return (int)(((float)x + 0.5f) * r); }

// cos and sin of 2 pi k / R at compile time (double Taylor series after
// folding the angle into [-pi/4, pi/4], rounded once to float).
constexpr double gfft_taylor(double x, int first) {
  double term = first ? x : 1.0, sum = term;
  for (int i = first + 1; i < 30; i += 2) {
    term *= -x * x / (double)(i * (i + 1));
    sum += term;
  }
  return sum;
}
constexpr double gfft_cos(int k, int R) {
  const double pi = 3.14159265358979323846;
  k = ((k % R) + R) % R;
  const int q = (8 * k + R) / (2 * R);  // the multiple of pi / 2 nearest 2 pi k / R
  const double x = pi * (4.0 * k - (double)q * R) / (2.0 * R);
  return q % 4 == 0 ? gfft_taylor(x, 0) : q % 4 == 1 ? -gfft_taylor(x, 1)
         : q % 4 == 2 ? -gfft_taylor(x, 0) : gfft_taylor(x, 1);
}
constexpr double gfft_sin(int k, int R) { return gfft_cos(4 * k - R, 4 * R); }
template <int R>
struct Roots {
  float c[R] = {}, s[R] = {};
  constexpr Roots() {
    for (int k = 0; k < R; ++k) {
      c[k] = (float)gfft_cos(k, R);
      s[k] = (float)gfft_sin(k, R);
    }
  }
};

// Odd radices: with t_k = x_k + x_{R-k}, d_k = x_k - x_{R-k},
// X_q, X_{R-q} = x_0 + sum_k cos(2 pi q k / R) t_k -+ i sum_k sin(2 pi q k / R) d_k
// (forward; signs swapped for the inverse), (R-1)^2 real multiply-adds.
template <int R, bool INV>
struct DftOdd {
  __device__ __forceinline__ static void run(cf* v) {
    constexpr Roots<R> w{};
    constexpr int H = (R - 1) / 2;
    cf t[H], d[H];
    cf x0 = v[0], sum = v[0];
#pragma unroll
    for (int k = 0; k < H; ++k) {
      t[k] = v[k + 1] + v[R - 1 - k];
      d[k] = v[k + 1] - v[R - 1 - k];
      sum = sum + t[k];
    }
    v[0] = sum;
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      cf a = x0, b = cf{0.f, 0.f};
#pragma unroll
      for (int k = 1; k <= H; ++k) {
        const float c = w.c[(q * k) % R], s = w.s[(q * k) % R];
        a = cf{fmaf(c, t[k - 1].re, a.re), fmaf(c, t[k - 1].im, a.im)};
        b = cf{fmaf(s, d[k - 1].re, b.re), fmaf(s, d[k - 1].im, b.im)};
      }
      b = rot90<INV>(b);
      v[q] = a + b;
      v[R - q] = a - b;
    }
  }
};
template <bool INV> struct Dft<7, INV> : DftOdd<7, INV> {};
template <bool INV> struct Dft<11, INV> : DftOdd<11, INV> {};
template <bool INV> struct Dft<13, INV> : DftOdd<13, INV> {};
template <bool INV> struct Dft<17, INV> : DftOdd<17, INV> {};
template <bool INV> struct Dft<19, INV> : DftOdd<19, INV> {};

// Composite radices R1 R2: R1-point transforms down the columns, the
// twiddles W_R^(n2 k1), R2-point transforms along the rows.
template <int R1, int R2, bool INV>
struct DftComp {
  __device__ __forceinline__ static void run(cf* v) {
    constexpr int R = R1 * R2;
    constexpr Roots<R> w{};
    cf a[R2][R1];
#pragma unroll
    for (int n2 = 0; n2 < R2; ++n2) {
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) a[n2][n1] = v[R2 * n1 + n2];
      Dft<R1, INV>::run(a[n2]);
#pragma unroll
      for (int k1 = 1; k1 < R1; ++k1)
        if (n2 > 0) a[n2][k1] = twid<INV>(a[n2][k1], cf{w.c[n2 * k1], -w.s[n2 * k1]});
    }
#pragma unroll
    for (int k1 = 0; k1 < R1; ++k1) {
      cf r[R2];
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) r[n2] = a[n2][k1];
      Dft<R2, INV>::run(r);
#pragma unroll
      for (int k2 = 0; k2 < R2; ++k2) v[k1 + R1 * k2] = r[k2];
    }
  }
};
template <bool INV> struct Dft<6, INV> : DftComp<3, 2, INV> {};
template <bool INV> struct Dft<9, INV> : DftComp<3, 3, INV> {};
template <bool INV> struct Dft<10, INV> : DftComp<5, 2, INV> {};
template <bool INV> struct Dft<12, INV> : DftComp<3, 4, INV> {};
template <bool INV> struct Dft<14, INV> : DftComp<7, 2, INV> {};
template <bool INV> struct Dft<15, INV> : DftComp<5, 3, INV> {};

// One Stockham pass of radix R over L lines side by side: butterfly j of a
// line reads x[j + s n/R] (s < R), multiplies input s by
// exp(-2 pi i s (j mod Ns) / (Ns R)), forms the R-point DFT in registers and
// writes output q to ((j / Ns) Ns R + j mod Ns + q Ns). Neighbouring threads
// take neighbouring lines of one butterfly: their accesses are consecutive
// and they share their twiddles.
template <int R, bool INV>
__device__ __forceinline__ void gfft_pass_r(const cf* A, cf* B, const cf* T, const GfftPass& p, int L, float rL,
                                            int pitch, int tid, int nthr) {
  const int work = L * p.m;
  for (int idx = tid; idx < work; idx += nthr) {
    const int j = fdiv(idx, rL), ll = idx - j * L;
    const cf* src = A + j * pitch + ll;
    const int ss = p.m * pitch;
    cf x[R];
#pragma unroll
    for (int s = 0; s < R; ++s) x[s] = src[s * ss];
    int o = j * R;
    if (p.Ns > 1) {
      const int jm = j - fdiv(j, p.rNs) * p.Ns, e1 = jm * p.tws;  // s * e1 < n for s < R
      o = (j - jm) * R + jm;
      const cf* t = T;
#pragma unroll
      for (int s = 1; s < R; ++s) {
        t += e1;
        x[s] = twid<INV>(x[s], *t);
      }
    }
    Dft<R, INV>::run(x);
    cf* dst = B + o * pitch + ll;
    const int ds = p.Ns * pitch;
#pragma unroll
    for (int q = 0; q < R; ++q) dst[q * ds] = x[q];
  }
}

// Any radix: each output one R-term sum whose twiddle exponents
// s ((j mod Ns) n/(Ns R) + q n/R) mod n index the table.
template <bool INV>
__device__ __forceinline__ void gfft_pass_direct(const cf* A, cf* B, const cf* T, const GfftPass& p, int n, int L,
                                                 float rL, int pitch, int tid, int nthr) {
  const float rm = 1.f / (float)p.m;
  if (p.Ns == 1 && (p.R & 1)) {
    // the first pass of an odd radix (the order the large primes take): the
    // outputs q and R - q from the sums of DftOdd, a quarter of the direct
    // sums' multiply-adds; neighbouring threads share q and so the roots
    const int H = (p.R - 1) / 2, ss = p.m * pitch;
    for (int idx = tid; idx < L * p.m * (H + 1); idx += nthr) {
      const int r = fdiv(idx, rL), ll = idx - r * L;
      const int q = fdiv(r, rm), j = r - q * p.m, es = q * p.m;
      const cf* lo = A + j * pitch + ll;
      const cf* hi = lo + p.R * ss;
      cf a = *lo, b = cf{0.f, 0.f};
      int e = 0;
#pragma unroll 4
      for (int s = 1; s <= H; ++s) {
        e += es;
        if (e >= n) e -= n;
        lo += ss;
        hi -= ss;
        const cf w = T[e], x = *lo, y = *hi;
        a = cf{fmaf(w.re, x.re + y.re, a.re), fmaf(w.re, x.im + y.im, a.im)};
        b = cf{fmaf(-w.im, x.re - y.re, b.re), fmaf(-w.im, x.im - y.im, b.im)};
      }
      b = rot90<INV>(b);
      cf* dst = B + j * p.R * pitch + ll;
      dst[q * pitch] = a + b;  // q = 0: every sine is 0
      if (q > 0) dst[(p.R - q) * pitch] = a - b;
    }
    return;
  }
  for (int idx = tid; idx < L * n; idx += nthr) {
    const int rem = fdiv(idx, rL), ll = idx - rem * L;
    const int q = fdiv(rem, rm), j = rem - q * p.m;
    const int jm = j - fdiv(j, p.rNs) * p.Ns;
    int es = jm * p.tws + q * p.m;
    if (es >= n) es -= n;
    const cf* src = A + j * pitch + ll;
    const int ss = p.m * pitch;
    cf acc = src[0];
    int e = es;
    for (int s = 1; s < p.R; ++s) {
      acc = cfma<INV>(acc, src[s * ss], T[e]);
      e += es;
      if (e >= n) e -= n;
    }
    B[((j - jm) * p.R + jm + q * p.Ns) * pitch + ll] = acc;
  }
}

// All passes over the L lines in A (B: as much again); returns the buffer
// the result is in (the other one is free), after a barrier.
// RMAX: the largest radix run as register butterflies (8 keeps the kernel's
// registers, and so its occupancy, low; 19 adds 9..17 and 19).
template <bool INV, int RMAX>
__device__ __forceinline__ cf* gfft_run(cf* A, cf* B, const cf* T, const GfftDev& d, int L, int pitch, int tid,
                                        int nthr) {
  const float rL = 1.f / (float)L;
  for (int i = 0; i < d.npass; ++i) {
    const GfftPass p = d.p[i];
    switch (p.R) {
#define EXMI_GFFT_R(RR)                                                          \
  case RR:                                                                       \
    if constexpr (RR <= RMAX) {                                                  \
      gfft_pass_r<RR, INV>(A, B, T, p, L, rL, pitch, tid, nthr);                 \
    } else {                                                                     \
      gfft_pass_direct<INV>(A, B, T, p, d.n, L, rL, pitch, tid, nthr);           \
    }                                                                            \
    break;
      EXMI_GFFT_R(2) EXMI_GFFT_R(3) EXMI_GFFT_R(4) EXMI_GFFT_R(5) EXMI_GFFT_R(6) EXMI_GFFT_R(7)
      EXMI_GFFT_R(8) EXMI_GFFT_R(9) EXMI_GFFT_R(10) EXMI_GFFT_R(11) EXMI_GFFT_R(12) EXMI_GFFT_R(13)
      EXMI_GFFT_R(14) EXMI_GFFT_R(15) EXMI_GFFT_R(16) EXMI_GFFT_R(17) EXMI_GFFT_R(19)
#undef EXMI_GFFT_R
      default: gfft_pass_direct<INV>(A, B, T, p, d.n, L, rL, pitch, tid, nthr); break;
    }
    __syncthreads();
    cf* t = A;
    A = B;
    B = t;
  }
  return A;
}

// Two real lines a, b of one complex line (a + i b): their half spectra from
// the complex spectrum's entries k and n - k (zk, zn).
__device__ __forceinline__ void unpack_pair(cf zk, cf zn, cf& a, cf& b) {
  a = cf{0.5f * (zk.re + zn.re), 0.5f * (zk.im - zn.im)};
  b = cf{0.5f * (zk.im + zn.im), 0.5f * (zn.re - zk.re)};
}

}  // namespace exmi
