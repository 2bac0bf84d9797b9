// Fused passes of the runtime-size plans (grid sizes outside the compiled
// set) around the line transforms of gfft.hpp: the spectral fields with the
// first inverse axis, the rows of the last axis with the pointwise products,
// and in 1-D whole ETDRK rollouts in one launch.
// One nonlinear evaluation of eight 513^2 Kolmogorov instances: 27 us of
// fields, 41 us of rows and products, 24 us of forward lines with the stage,
// against 358 us as separate fields, transforms of whole fields (119 + 88 us
// for the four fields), products, transforms and stage. What bounds them is
// the latency of the short passes between barriers at three to five
// workgroups per CU; passes in place in registers (half the LDS, twice the
// barriers) took the rows at 513 from 48 to 42 us when the odd sizes' lines
// still had a pad entry per point, and cost 8% of a step at 48^3.
#include "gspec.hpp"
#include "nl3d.hpp"

namespace exmi {

// ------------------------------------------------ fields + first inverse axis
struct GFieldsArgs {
  NL3DArgs a;
  GfftDev d;
  int lpb, kkeep, midn, midkeep;
  long long nrun, pstride;  // lines that run; points of a line are pstride apart
  float scale;
  const cf* S;
  cf* F;
  const cf* tw;
};

// One workgroup: lpb neighbouring lines (field g = inst * nf + f, m, kz) of
// the outermost axis. The field is formed from the state's spectrum as it is
// read, so neither a fields pass nor its spectra exist in memory, and what
// the dealias cutoff makes zero is neither read nor transformed.
template <int RMAX, bool TWL>
__global__ void __launch_bounds__(GFFT_WG) gfields_kernel(GFieldsArgs g) {
  extern __shared__ cf gspec_smem[];
  __shared__ long long b0[GFFT_MAX_LINES];
  __shared__ int bf[GFFT_MAX_LINES], bm[GFFT_MAX_LINES], bz[GFFT_MAX_LINES];
  __shared__ long long bi[GFFT_MAX_LINES];
  const int n = g.d.n, tid = threadIdx.x;
  const long long run0 = (long long)xcd_block() * g.lpb;
  const int L = (int)(g.nrun - run0 < g.lpb ? g.nrun - run0 : g.lpb);
  const int pitch = gfft_pitch_by_point(n, g.lpb);
  cf* A = gspec_smem;
  cf* B = gspec_smem + n * pitch;
  const cf* T = TWL ? gspec_smem + 2 * n * pitch : g.tw;
  if constexpr (TWL)
    for (int i = tid; i < n; i += GFFT_WG) gspec_smem[2 * n * pitch + i] = g.tw[i];
  if (tid < L) {
    const long long run = run0 + tid;
    const long long r = run / g.kkeep, fl = r / g.midkeep;
    const int z = (int)(run - r * g.kkeep), m = gfft_kept((int)(r - fl * g.midkeep), g.midkeep, g.midn);
    bi[tid] = fl / g.a.nf;
    bf[tid] = (int)(fl % g.a.nf);
    bm[tid] = m;
    bz[tid] = z;
    b0[tid] = (long long)m * g.a.NZ + z;
  }
  __syncthreads();
  const float rL = 1.f / (float)L;
  for (int idx = tid; idx < L * n; idx += GFFT_WG) {
    const int pt = fdiv(idx, rL), ll = idx - pt * L;
    cf v = cf{0.f, 0.f};
    if (pt <= g.a.kmax || n - pt <= g.a.kmax) {
      // 3-D: the line runs along x at (ky, kz) = (bm, bz); 2-D: along the
      // first axis (the middle one of the embedding) at kz = bz
      const Mode3D m = g.midn > 1 ? mode3d_at(g.a, pt, bm[ll], bz[ll]) : mode3d_at(g.a, 0, pt, bz[ll]);
      v = field_at(g.a, g.S, bi[ll], bf[ll], b0[ll] + pt * g.pstride, m);
    }
    A[pt * pitch + ll] = v;
  }
  __syncthreads();
  const cf* Z = gfft_run<true, RMAX>(A, B, T, g.d, L, pitch, tid, GFFT_WG);
  for (int idx = tid; idx < L * n; idx += GFFT_WG) {
    const int pt = fdiv(idx, rL), ll = idx - pt * L;
    g.F[(bi[ll] * g.a.nf + bf[ll]) * g.a.Nr + b0[ll] + pt * g.pstride] = g.scale * Z[pt * pitch + ll];
  }
}

hipError_t launch_gfields(const GfftCfg& c, const NL3DArgs& a, const cf* S, cf* F, float scale, int kkeep,
                          const cf* tw, hipStream_t st) {
  if (a.dims < 2 || c.n != a.N || kkeep < 1 || kkeep > a.NZ || a.kmax < 0) return hipErrorInvalidValue;
  GFieldsArgs g;
  g.a = a;
  g.d = gfft_dev(c);
  g.lpb = c.lpb;
  g.kkeep = kkeep;
  g.midn = a.dims == 3 ? a.ny : 1;
  g.midkeep = gfft_midkeep(g.midn, a.kmax);
  g.pstride = a.dims == 3 ? (long long)a.ny * a.NZ : a.NZ;
  g.nrun = a.ninst * a.nf * g.midkeep * kkeep;
  g.scale = scale;
  g.S = S;
  g.F = F;
  g.tw = tw;
  const long long grid = (g.nrun + c.lpb - 1) / c.lpb;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const size_t buf = sizeof(cf) * 2 * (size_t)c.n * gfft_pitch_by_point(c.n, c.lpb), fixed = 28 * GFFT_MAX_LINES;
  size_t lds = buf + sizeof(cf) * (size_t)c.n;
  const bool twl = lds + fixed <= GFFT_LDS_MAX;
  if (!twl) lds = buf;
  auto* k = gfft_big(c) ? (twl ? gfields_kernel<19, true> : gfields_kernel<19, false>)
                        : (twl ? gfields_kernel<8, true> : gfields_kernel<8, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(GFFT_WG), lds, st, g);
  return hipGetLastError();
}

// ------------------------------------------------------- rows + products
struct GProdArgs {
  NL3DArgs a;
  GfftDev d;
  int units, nft, npt, kkeep;  // pairs of rows per workgroup; fields and products per trajectory
  long long nunits, rows;
  float scale;
  const cf* F;
  cf* P;
  const cf* tw;
};

// One unit: two neighbouring rows (2q, 2q + 1) of one trajectory, each
// field's two rows packed into one complex line (they are of one field, so
// of one magnitude), their c2r, the products at every point of both rows,
// and the products' r2c, two rows to a line again. The fields' and products'
// physical values stay in LDS.
template <int RMAX, bool TWL>
__global__ void __launch_bounds__(GFFT_WG) gprod_kernel(GProdArgs g) {
  extern __shared__ cf gspec_smem[];
  const int n = g.d.n, nz = g.a.NZ, tid = threadIdx.x;
  const long long u0 = (long long)blockIdx.x * g.units;
  const int U = (int)(g.nunits - u0 < g.units ? g.nunits - u0 : g.units);
  const int LF = U * g.nft, LP = U * g.npt;
  const int pf = gfft_pitch_by_point(n, g.units * g.nft), pp = gfft_pitch_by_point(n, g.units * g.npt);
  const int half = n * (pf > pp ? pf : pp);
  cf* A = gspec_smem;
  cf* B = gspec_smem + half;
  const cf* T = TWL ? gspec_smem + 2 * half : g.tw;
  if constexpr (TWL)
    for (int i = tid; i < n; i += GFFT_WG) gspec_smem[2 * half + i] = g.tw[i];
  const float rnz = 1.f / (float)nz, rU = 1.f / (float)U, rnf = 1.f / (float)g.nft, rnp = 1.f / (float)g.npt;
  const float rkk = 1.f / (float)g.kkeep;
  // where line l of unit u starts: row 0, and whether it has a row 1. The
  // first unit's trajectory and row are divided out once; a unit further on
  // is rarely past the trajectory's end.
  const long long per = (g.rows + 1) / 2, tb = u0 / per, tq = u0 - tb * per;  // per: units per trajectory
  auto where = [&](int u, int l, int count, long long& at, bool& two) {
    long long b = tb, q = tq + u;
    while (q >= per) {
      q -= per;
      ++b;
    }
    at = (b * count + l) * g.a.Nr + 2 * q * nz;
    two = 2 * q + 1 < g.rows;
  };
  for (int idx = tid; idx < LF * nz; idx += GFFT_WG) {
    const int ll = fdiv(idx, rnz), k = idx - ll * nz;
    const int u = fdiv(ll, rnf);
    long long at;
    bool two;
    where(u, ll - u * g.nft, g.nft, at, two);
    cf p = cf{0.f, 0.f}, q = p;
    if (k < g.kkeep) {
      p = g.F[at + k];
      if (two) q = g.F[at + nz + k];
    }
    const bool self = k == 0 || 2 * k == n;
    if (self) p.im = q.im = 0.f;
    A[k * pf + ll] = cf{p.re - q.im, p.im + q.re};
    if (!self) A[(n - k) * pf + ll] = cf{p.re + q.im, q.re - p.im};
  }
  __syncthreads();
  cf* Z = gfft_run<true, RMAX>(A, B, T, g.d, LF, pf, tid, GFFT_WG);
  cf* O = Z == A ? B : A;
  for (int idx = tid; idx < U * n; idx += GFFT_WG) {
    const int pt = fdiv(idx, rU), u = idx - pt * U;
    const cf* z = Z + pt * pf + u * g.nft;
    cf* o = O + pt * pp + u * g.npt;
    nl_products<v2>(
        g.a,
        [&](int c, int f) {
          const cf v = z[c * g.a.nf + f];
          return v2{g.scale * v.re, g.scale * v.im};
        },
        [&](int c, int j, v2 v) { o[c * g.a.np + j] = cf{v.a, v.b}; });
  }
  __syncthreads();
  const cf* Y = gfft_run<false, RMAX>(O, Z, T, g.d, LP, pp, tid, GFFT_WG);
  for (int idx = tid; idx < LP * g.kkeep; idx += GFFT_WG) {
    const int ll = fdiv(idx, rkk), k = idx - ll * g.kkeep;
    const int u = fdiv(ll, rnp);
    long long at;
    bool two;
    where(u, ll - u * g.npt, g.npt, at, two);
    cf p, q;
    unpack_pair(Y[k * pp + ll], Y[(k == 0 ? 0 : n - k) * pp + ll], p, q);
    g.P[at + k] = p;
    if (two) g.P[at + nz + k] = q;
  }
}

// LDS of one workgroup of `units` units, without and with the twiddle table.
static size_t gprod_lds(int n, int nft, int npt, int units, bool tw) {
  const int pf = gfft_pitch_by_point(n, units * nft), pp = gfft_pitch_by_point(n, units * npt);
  return sizeof(cf) * ((size_t)2 * n * (pf > pp ? pf : pp) + (tw ? n : 0));
}

bool gprod_fits(const GfftCfg& c, const NL3DArgs& a) {
  return a.dims >= 2 && gprod_lds(c.n, a.channels * a.nf, a.channels * a.np, 1, false) <= GFFT_LDS_MAX;
}

hipError_t launch_gprod(const GfftCfg& c, const NL3DArgs& a, const cf* F, cf* P, float scale, int kkeep,
                        const cf* tw, hipStream_t st) {
  if (!gprod_fits(c, a) || c.n != a.N || kkeep < 1 || kkeep > a.NZ) return hipErrorInvalidValue;
  GProdArgs g;
  g.a = a;
  g.d = gfft_dev(c);
  g.nft = a.channels * a.nf;
  g.npt = a.channels * a.np;
  const int most = g.nft > g.npt ? g.nft : g.npt;
  g.rows = a.dims == 3 ? (long long)a.nx * a.ny : a.ny;
  g.nunits = a.ninst / a.channels * ((g.rows + 1) / 2);
  g.units = c.lpb / most;  // the tuned lines per workgroup
  // Short lines leave most of a workgroup's lanes without a butterfly: up to
  // 1400 points to a workgroup while that leaves three workgroups to a CU (3-D
  // Burgers, two of 12 fields, two units instead of one: 20 steps at 48^3 2266
  // -> 2090 us, 16 at 45^3 1751 -> 1585; four vorticity fields of 16 x 135^2,
  // 1088 units, would lose 1015 -> 1047). Swept from 0 to 3500 points over 21
  // shapes, 16 steps (none / 1152 / 1400 / 1800 points): 3-D Burgers 2 x 48^3
  // 1548 / 1430 / 1434 / 1465 us, 2 x 54^3 1830 / 1872 / 1731 / 1697,
  // Navier-Stokes 4 x 50^3 1708 / 1634 / 1621 / 1671; the others of 1152 points
  // and more within 1%.
  long long fill = 1400 / ((long long)most * c.n);
  if (fill > g.nunits / 768) fill = g.nunits / 768;
  if (fill > GFFT_MAX_LINES / most) fill = GFFT_MAX_LINES / most;
  if (g.units < fill) g.units = (int)fill;
  if (g.units < 1) g.units = 1;
  while (g.units > 1 && gprod_lds(c.n, g.nft, g.npt, g.units, false) > GFFT_LDS_MAX) --g.units;
  g.kkeep = kkeep;
  g.scale = scale;
  g.F = F;
  g.P = P;
  g.tw = tw;
  const long long grid = (g.nunits + g.units - 1) / g.units;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const bool twl = gprod_lds(c.n, g.nft, g.npt, g.units, true) <= GFFT_LDS_MAX;
  const size_t lds = gprod_lds(c.n, g.nft, g.npt, g.units, twl);
  auto* k = gfft_big(c) ? (twl ? gprod_kernel<19, true> : gprod_kernel<19, false>)
                        : (twl ? gprod_kernel<8, true> : gprod_kernel<8, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(GFFT_WG), lds, st, g);
  return hipGetLastError();
}

// -------------------------------------- last forward axis + combine + stage
struct GStageArgs {
  NL3DArgs a;
  GfftDev d;
  int units, npt, kkeep, midn, cut;  // lines (trajectory, m, kz) per workgroup; products per trajectory
  long long nunits, pstride;
  const cf* P;
  cf* N0out;
  const cf* tw;
};

// The combine and stage M at every point of the workgroup's U lines.
template <int M>
__device__ __forceinline__ void gstage_points(const GStageArgs& g, const Stage3DArgs& st, const cf* Z, const long long* b0, const int* bm,
                                              const int* bz, const int* bk, int U, int pitch) {
  const int C = g.a.channels, np = g.a.np, n = g.d.n;
  const float rU = 1.f / (float)U, rC = 1.f / (float)C;
  for (int idx = threadIdx.x; idx < U * C * n; idx += GFFT_WG) {
    const int q = fdiv(idx, rU), u = idx - q * U, pt = fdiv(q, rC), c = q - pt * C;
    const Mode3D md = g.midn > 1 ? mode3d_at(g.a, pt, bm[u], bz[u]) : mode3d_at(g.a, 0, pt, bz[u]);
    const cf* z = Z + pt * pitch + u;
    const int keep = bk[u];
    const cf nh = combine_core(g.a, md, c, [=](int cc, int j) { return keep ? z[(cc * np + j) * U] : cf{0.f, 0.f}; });
    const long long k = pt * g.pstride + (long long)bm[u] * g.a.NZ + bz[u];
    const long long at = (b0[u] * C + c) * g.a.Nr + k;
    cf n0 = nh;
    if (g.N0out) g.N0out[at] = nh;
    else if (stage_reads_n0(M)) n0 = st.N0[at];
    stage_core<M>(st.e_im, st.nr, stage_table(st, b0[u], c), k, at, st.U0, st.S, st.S1, st.A, n0, nh);
  }
}

// The products' lines of the outermost axis, transformed and then combined
// into N_hat and the stage at every point while they are in LDS: neither the
// product spectra's last pass nor a combine pass goes through memory: 25 us
// for eight 513^2 instances, 17 + 13 us as two passes. Lines beyond the
// dealias cutoff hold no products; their N_hat is zero. The stage's arguments
// are a kernel parameter of their own: inside the other struct its ten-way
// switch made the compiler copy all arguments to scratch (44 us).
template <int RMAX, bool TWL>
__global__ void __launch_bounds__(GFFT_WG) gstage_kernel(GStageArgs g, Stage3DArgs st) {
  extern __shared__ cf gspec_smem[];
  __shared__ long long b0[GFFT_MAX_LINES];  // trajectory
  __shared__ int bm[GFFT_MAX_LINES], bz[GFFT_MAX_LINES], bk[GFFT_MAX_LINES];
  const int n = g.d.n, tid = threadIdx.x;
  const long long u0 = (long long)xcd_block() * g.units;
  const int U = (int)(g.nunits - u0 < g.units ? g.nunits - u0 : g.units);
  const int L = U * g.npt, pitch = gfft_pitch_by_point(n, g.units * g.npt);
  cf* A = gspec_smem;
  cf* B = gspec_smem + n * pitch;
  const cf* T = TWL ? gspec_smem + 2 * n * pitch : g.tw;
  if constexpr (TWL)
    for (int i = tid; i < n; i += GFFT_WG) gspec_smem[2 * n * pitch + i] = g.tw[i];
  if (tid < U) {
    const long long unit = u0 + tid, r = unit / g.a.NZ, b = r / g.midn;
    const int z = (int)(unit - r * g.a.NZ), m = (int)(r - b * g.midn);
    b0[tid] = b;
    bm[tid] = m;
    bz[tid] = z;
    bk[tid] = z < g.kkeep && (g.midn == 1 || m <= g.cut || g.midn - m <= g.cut);
  }
  __syncthreads();
  bool any = false;
  for (int u = 0; u < U; ++u) any = any || bk[u];
  const float rL = 1.f / (float)L, rU = 1.f / (float)U;
  const cf* Z = A;
  if (any) {
    for (int idx = tid; idx < L * n; idx += GFFT_WG) {
      const int pt = fdiv(idx, rL), l = idx - pt * L;  // line l = j * U + u: neighbouring threads, neighbouring kz
      const int j = fdiv(l, rU), u = l - j * U;
      A[pt * pitch + l] = bk[u] ? g.P[(b0[u] * g.npt + j) * g.a.Nr + pt * g.pstride + (long long)bm[u] * g.a.NZ + bz[u]]
                                : cf{0.f, 0.f};
    }
    __syncthreads();
    Z = gfft_run<false, RMAX>(A, B, T, g.d, L, pitch, tid, GFFT_WG);
  }
  switch (st.mode) {
#define EXMI_GSTAGE(M) \
  case M: gstage_points<M>(g, st, Z, b0, bm, bz, bk, U, pitch); break;
    EXMI_GSTAGE(ST1) EXMI_GSTAGE(ST2A) EXMI_GSTAGE(ST2B) EXMI_GSTAGE(ST3A) EXMI_GSTAGE(ST3B) EXMI_GSTAGE(ST3C)
    EXMI_GSTAGE(ST4A) EXMI_GSTAGE(ST4B) EXMI_GSTAGE(ST4C) EXMI_GSTAGE(ST4D)
#undef EXMI_GSTAGE
  }
}

static size_t gstage_lds(int n, int npt, int units, bool tw) {
  return sizeof(cf) * ((size_t)2 * n * gfft_pitch_by_point(n, units * npt) + (tw ? n : 0));
}
constexpr size_t GSTAGE_FIXED = 20 * GFFT_MAX_LINES;

bool gstage_fits(const GfftCfg& c, const NL3DArgs& a) {
  return a.dims >= 2 && gstage_lds(c.n, a.channels * a.np, 1, false) + GSTAGE_FIXED <= GFFT_LDS_MAX;
}

hipError_t launch_gstage(const GfftCfg& c, const NL3DArgs& a, const Stage3DArgs& sa, const cf* P, cf* N0out,
                         int kkeep, int cut, const cf* tw, hipStream_t st) {
  if (!gstage_fits(c, a) || c.n != a.N || kkeep < 1 || kkeep > a.NZ) return hipErrorInvalidValue;
  GStageArgs g;
  g.a = a;
  g.d = gfft_dev(c);
  g.npt = a.channels * a.np;
  g.units = c.lpb / g.npt;
  if (g.units < 1) g.units = 1;
  while (g.units > 1 && gstage_lds(c.n, g.npt, g.units, false) + GSTAGE_FIXED > GFFT_LDS_MAX) --g.units;
  g.kkeep = kkeep;
  g.cut = cut;
  g.midn = a.dims == 3 ? a.ny : 1;
  g.pstride = a.dims == 3 ? (long long)a.ny * a.NZ : a.NZ;
  g.nunits = a.ninst / a.channels * g.midn * a.NZ;
  g.P = P;
  g.N0out = N0out;
  g.tw = tw;
  const long long grid = (g.nunits + g.units - 1) / g.units;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  const bool twl = gstage_lds(c.n, g.npt, g.units, true) + GSTAGE_FIXED <= GFFT_LDS_MAX;
  const size_t lds = gstage_lds(c.n, g.npt, g.units, twl);
  auto* k = gfft_big(c) ? (twl ? gstage_kernel<19, true> : gstage_kernel<19, false>)
                        : (twl ? gstage_kernel<8, true> : gstage_kernel<8, false>);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(GFFT_WG), lds, st, g, sa);
  return hipGetLastError();
}

// ------------------------------------------------------ 1-D whole rollouts
constexpr int G1D_WG_MAX = 512;

static int g1d_lines(int channels, int nf, int np) {
  const int f = channels * (nf > 0 ? nf : 1), p = channels * (np > 0 ? np : 1);
  return f > p ? f : p;
}
// State-sized spectra a step of this order holds: U, S, N0; the accumulated
// state of orders 3 and 4; S1 of order 4.
static int g1d_spectra(int order) { return order <= 2 ? 3 : order == 3 ? 4 : 5; }
static size_t g1d_lds(int N, int channels, int lines, int order) {
  return sizeof(cf) * ((size_t)2 * N * gfft_pitch(lines) + N + (size_t)g1d_spectra(order) * channels * (N / 2 + 1));
}
bool g1d_fits(int N, int channels, int nf, int np, int order, int lin_channels, int ncoef) {
  return g1d_lds(N, channels, g1d_lines(channels, nf, np), order) +
             sizeof(float) * (size_t)lin_channels * ncoef * (N / 2 + 1) <=
         GFFT_LDS_MAX;
}

// One workgroup owns one trajectory (all its channels) for all steps: the
// spectra of the state and the stages, the line buffers and the twiddles stay
// in LDS, only the emitted states cross memory. At these sizes a step is a
// chain of short dependent passes, so its time is the latency of that chain:
// the multi-pass form launches 9 to 20 kernels of 3 to 8 us for it.
// Measured: two-field Burgers, N = 100, 100 trajectories, 11.4 us per step
// against 52 us.
template <int RMAX>
__global__ void __launch_bounds__(G1D_WG_MAX) g1d_kernel(G1dArgs g) {
  extern __shared__ cf gspec_smem[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const NL3DArgs& a = g.nl;
  const int n = a.N, nz = a.NZ, C = a.channels;
  const int nft = C * a.nf, npt = C * a.np, S1N = C * nz;
  const int most = nft > npt ? nft : npt;
  const int pitch = gfft_pitch(most > C ? most : C);
  cf* A = gspec_smem;
  cf* B = A + n * pitch;
  cf* T = B + n * pitch;
  cf* U = T + n;
  cf* S = U + S1N;
  cf* N0 = S + S1N;
  cf* AC = N0 + S1N;                    // orders 3, 4
  cf* SA = AC + (g.order >= 3 ? S1N : 0);  // order 4
  float* TB = reinterpret_cast<float*>(SA + (g.order >= 4 ? S1N : 0));
  for (int i = tid; i < n; i += nthr) T[i] = g.tw[i];
  const long long b = blockIdx.x;
  const long long tb0 = (g.lin_batch > 1 ? b : 0) * g.lin_channels * (long long)g.ncoef * nz;
  const long long tbs = g.lin_channels > 1 ? (long long)g.ncoef * nz : 0;  // per channel
  for (int i = tid; i < g.lin_channels * g.ncoef * nz; i += nthr) TB[i] = g.tables[tb0 + i];
  const float* tables = TB;
  const float rC = 1.f / (float)C, rnz = 1.f / (float)nz, rn = 1.f / (float)n;
  const float scale = rn;
  const int stages = g.order;
  // physical states of the C channels -> lines of A, transformed into U
  auto forward = [&](cf* from, cf* other) {
    const cf* Z = gfft_run<false, RMAX>(from, other, T, g.d, C, pitch, tid, nthr);
    for (int idx = tid; idx < S1N; idx += nthr) {
      const int k = fdiv(idx, rC), c = idx - k * C;
      U[c * nz + k] = Z[k * pitch + c];
    }
    __syncthreads();
  };
  const float* u0 = g.u0 + b * g.u0_bs;
  for (int idx = tid; idx < C * n; idx += nthr) {
    const int c = fdiv(idx, rn), pt = idx - c * n;
    A[pt * pitch + c] = cf{u0[idx], 0.f};
  }
  __syncthreads();
  forward(A, B);
  int slot = 0, next = next_written(0, g.every, g.nsteps);
  for (int t = 0; t < g.nsteps; ++t) {
    if (g.order == 0) {
      for (int idx = tid; idx < S1N; idx += nthr) {
        const int c = fdiv(idx, rnz), k = idx - c * nz;
        const float* tb = tables + c * tbs;
        const cf x = U[idx];
        const float er = tb[k];
        S[idx] = er * x;
        if (g.e_im >= 0) {
          const float ei = tb[g.e_im * nz + k];
          S[idx] = cf{fmaf(er, x.re, -ei * x.im), fmaf(er, x.im, ei * x.re)};
        }
      }
      __syncthreads();
    }
    for (int i = 0; i < stages; ++i) {
      const cf* X = i == 0 ? U : S;
      for (int idx = tid; idx < nft * nz; idx += nthr) {
        const int ll = fdiv(idx, rnz), k = idx - ll * nz;
        const int c = ll / a.nf, f = ll - c * a.nf;
        cf v = field_at(a, X, c, f, k, mode3d_at(a, 0, 0, k));
        const bool self = k == 0 || 2 * k == n;
        if (self) v.im = 0.f;
        A[k * pitch + ll] = v;
        if (!self) A[(n - k) * pitch + ll] = conj(v);
      }
      __syncthreads();
      cf* Z = gfft_run<true, RMAX>(A, B, T, g.d, nft, pitch, tid, nthr);
      cf* O = Z == A ? B : A;
      for (int pt = tid; pt < n; pt += nthr) {
        const cf* z = Z + pt * pitch;
        cf* o = O + pt * pitch;
        nl_products<float>(
            a, [&](int c, int f) { return scale * z[c * a.nf + f].re; },
            [&](int c, int j, float v) { o[c * a.np + j] = cf{v, 0.f}; });
      }
      __syncthreads();
      const cf* Y = gfft_run<false, RMAX>(O, Z, T, g.d, npt, pitch, tid, nthr);
      const int mode = (g.order == 1 ? ST1 : g.order == 2 ? ST2A : g.order == 3 ? ST3A : ST4A) + i;
      for (int idx = tid; idx < S1N; idx += nthr) {
        const int c = fdiv(idx, rnz), k = idx - c * nz;
        const cf r = combine_core(a, mode3d_at(a, 0, 0, k), c,
                                  [&](int cc, int j) { return Y[k * pitch + cc * a.np + j]; });
        cf n0 = r;
        if (i == 0) N0[idx] = r;
        else n0 = N0[idx];
        with_stage_mode(mode, [&](auto m) {
          stage_core<decltype(m)::value>(g.e_im, nz, tables + c * tbs, k, idx, U, S, SA, AC, n0, r);
        });
      }
      __syncthreads();
    }
    const bool emit = t + 1 == next;
    if (emit || g.roundtrip) {
      for (int idx = tid; idx < S1N; idx += nthr) {
        const int c = fdiv(idx, rnz), k = idx - c * nz;
        cf v = S[idx];
        const bool self = k == 0 || 2 * k == n;
        if (self) v.im = 0.f;
        A[k * pitch + c] = v;
        if (!self) A[(n - k) * pitch + c] = conj(v);
      }
      __syncthreads();
      cf* Z = gfft_run<true, RMAX>(A, B, T, g.d, C, pitch, tid, nthr);
      cf* O = Z == A ? B : A;
      float* out = written_at(g.out, g.out_ts, slot, g.last, t + 1 == g.nsteps) + b * g.out_bs;
      for (int idx = tid; idx < C * n; idx += nthr) {
        const int c = fdiv(idx, rn), pt = idx - c * n;
        const float v = scale * Z[pt * pitch + c].re;
        if (emit) out[idx] = v;
        if (g.roundtrip) O[pt * pitch + c] = cf{v, 0.f};
      }
      __syncthreads();
      if (emit) {
        ++slot;
        next = next_written(next, g.every, g.nsteps);
      }
      if (g.roundtrip) {
        if (t < g.nsteps - 1) forward(O, Z);
        continue;
      }
    }
    cf* s = U;
    U = S;
    S = s;
  }
}

// The same for one channel, one field and one product (convection in flux
// form, the gradient norm, the polynomials), where the spectrum is carried or
// one step is taken: the transforms' outer passes do the pointwise work.
// The first inverse pass reads the field from the spectrum; the last inverse
// pass holds the points j + q n/R of its R outputs, which are the inputs of a
// forward pass of the same radix, so with the forward's radices in reverse
// order the product and the first forward pass follow in registers; the last
// forward pass's outputs go straight into the stage. A nonlinear evaluation
// of two-pass lengths is three dependent phases with an LDS exchange between
// them, of three-pass lengths five. The emission of a state is a second line
// beside the first evaluation of the next step.
// Measured (Burgers, 100 trajectories): N = 100 7.1 us per step, N = 360
// 9.3 us, N = 500 10.3 us; the launches of the separate passes take 52 us at
// N = 100. One wavefront's instruction issue bounds it: 12 phases of some 150
// instructions each at N = 100.
constexpr int G1S_MAX_PASS = 4;

// The radices the fused single-field kernel is built for: those the fewest
// passes of at most 8 points use, and the primes above.
__host__ __device__ constexpr bool g1s_radix(int R) {
  return (R >= 2 && R <= 10) || R == 11 || R == 13 || R == 17 || R == 19;
}
template <class F>
__device__ __forceinline__ void with_g1s_radix(int R, F&& f) {
  switch (R) {
#define EXMI_G1S_R(RR) \
  case RR: f(std::integral_constant<int, RR>{}); break;
    EXMI_G1S_R(2) EXMI_G1S_R(3) EXMI_G1S_R(4) EXMI_G1S_R(5) EXMI_G1S_R(6) EXMI_G1S_R(7) EXMI_G1S_R(8)
    EXMI_G1S_R(9) EXMI_G1S_R(10) EXMI_G1S_R(11) EXMI_G1S_R(13) EXMI_G1S_R(17) EXMI_G1S_R(19)
#undef EXMI_G1S_R
  }
}

// Buffers as offsets into the workgroup's LDS array (entries): two line
// buffers of 2 n, the twiddles, and the spectra.
__global__ void __launch_bounds__(G1D_WG_MAX) g1s_kernel(G1dArgs g) {
  extern __shared__ cf sm[];
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int n = g.nl.N, nz = g.nl.NZ, np = g.d.npass, kmax = g.nl.kmax, order = g.order, nsteps = g.nsteps;
  const int every = g.every, e_im = g.e_im;
  const bool grad = g.nl.kind == NL_GRADNORM, poly = g.nl.kind == NL_POLY;
  const float kscale = g.nl.kscale, scale = 1.f / (float)n;
  const GfftPass i0 = g.d.p[0], i1 = g.d.p[1], i2 = g.d.p[2], i3 = g.d.p[3];
  const GfftPass f0 = g.df.p[0], f1 = g.df.p[1], f2 = g.df.p[2], f3 = g.df.p[3];
  const int iT = 4 * n;
  int a = 0, b = 2 * n;  // the line buffers
  int iU = 5 * n, iS = iU + nz;
  const int iN0 = iS + nz, iAC = iN0 + nz, iSA = iAC + (order >= 3 ? nz : 0);
  const int iTB = iSA + (order >= 4 ? nz : 0);
  const long long traj = blockIdx.x;
  {
    const float* tables = g.tables + (g.lin_batch > 1 ? traj : 0) * (long long)g.ncoef * nz;
    float* tb = reinterpret_cast<float*>(sm + iTB);
    for (int i = tid; i < g.ncoef * nz; i += nthr) tb[i] = tables[i];
    const float* u0 = g.u0 + traj * g.u0_bs;
    for (int i = tid; i < n; i += nthr) {
      sm[iT + i] = g.tw[i];
      sm[a + i] = cf{u0[i], 0.f};
    }
  }
  float* at = g.out + traj * g.out_bs;  // where the next written state goes
  float* const last = g.last ? g.last + traj * g.out_bs : nullptr;
  const long long out_ts = g.out_ts;
  int next = next_written(0, every, nsteps);
  __syncthreads();
  // one inner pass of L lines side by side, LDS to LDS
  auto pass = [&](auto inv, const GfftPass p, int L) __attribute__((always_inline)) {
    with_g1s_radix(p.R, [&](auto r) {
      gfft_pass_r<decltype(r)::value, decltype(inv)::value>(sm + a, sm + b, sm + iT, p, L, 1.f / (float)L, L, tid, nthr);
    });
    __syncthreads();
    const int t = a;
    a = b;
    b = t;
  };
  const std::false_type fwd{};
  const std::true_type inv{};
  // pass i of four (uniform; in scalar registers, no indexed table in memory)
  static_assert(G1S_MAX_PASS == 4, "passes held by name");
  auto pick = [](int i, GfftPass p0, GfftPass p1, GfftPass p2, GfftPass p3) __attribute__((always_inline)) {
    GfftPass r;
    r.R = i == 0 ? p0.R : i == 1 ? p1.R : i == 2 ? p2.R : p3.R;
    r.Ns = i == 0 ? p0.Ns : i == 1 ? p1.Ns : i == 2 ? p2.Ns : p3.Ns;
    r.m = i == 0 ? p0.m : i == 1 ? p1.m : i == 2 ? p2.m : p3.m;
    r.tws = i == 0 ? p0.tws : i == 1 ? p1.tws : i == 2 ? p2.tws : p3.tws;
    r.rNs = i == 0 ? p0.rNs : i == 1 ? p1.rNs : i == 2 ? p2.rNs : p3.rNs;
    return r;
  };
#pragma unroll 1
  for (int i = 0; i < np; ++i) pass(fwd, pick(i, f0, f1, f2, f3), 1);
  for (int k = tid; k < nz; k += nthr) sm[iU + k] = sm[a + k];
  __syncthreads();
  for (int t = 0; t <= nsteps; ++t) {
    // t == nsteps: only the last state's emission
    const bool emit = t == next, step = t < nsteps;
    const int stages = step ? order : 1;
    float* const dst = step || !last ? at : last;
    if (emit) {
      at += out_ts;
      next = next_written(next, every, nsteps);
    }
    for (int i = 0; i < stages; ++i) {
      const int iX = i == 0 ? iU : iS;
      const int L = (i == 0 && emit && step) ? 2 : 1;
      const int line_e = (i == 0 && emit) ? L - 1 : L;  // the line that is the emitted state
      // the field, first inverse pass
      with_g1s_radix(i0.R, [&](auto rr) {
        constexpr int R = decltype(rr)::value;
        const int m = i0.m, x0 = iX;
        for (int idx = tid; idx < L * m; idx += nthr) {
          const int j = L == 1 ? idx : idx >> 1, ll = idx - j * L;
          cf x[R];
          int pt = j;
#pragma unroll
          for (int s = 0; s < R; ++s) {
            const bool upper = pt >= nz;
            const int k = upper ? n - pt : pt;
            cf v = sm[x0 + k];
            if (ll != line_e) {
              // the dealiased field (field_at of these kinds)
              if (grad) v = imul(kscale * (float)k, v);
              if (k > kmax) v = cf{0.f, 0.f};
            }
            if (k == 0 || 2 * k == n) v.im = 0.f;
            x[s] = upper ? conj(v) : v;
            pt += m;
          }
          Dft<R, true>::run(x);
          const int o = b + j * (R * L) + ll;
#pragma unroll
          for (int q = 0; q < R; ++q) sm[o + q * L] = x[q];
        }
      });
      __syncthreads();
      {
        const int t1 = a;
        a = b;
        b = t1;
      }
#pragma unroll 1
      for (int e = 1; e < np - 1; ++e) pass(inv, pick(e, i0, i1, i2, i3), L);
      // last inverse pass, the product, first forward pass
      const GfftPass plast = pick(np - 1, i0, i1, i2, i3);
      with_g1s_radix(plast.R, [&](auto rr) {
        constexpr int R = decltype(rr)::value;
        const int m = plast.m;  // = Ns: output q of butterfly j is point j + q m
        const int in = a, o = b;
        for (int idx = tid; idx < L * m; idx += nthr) {
          const int j = L == 1 ? idx : idx >> 1, ll = idx - j * L;
          cf x[R];
          const int at = in + j * L + ll, ms = m * L;
          int tj = iT;
#pragma unroll
          for (int s = 0; s < R; ++s) {
            x[s] = sm[at + s * ms];
            if (s > 0) x[s] = twid<true>(x[s], sm[tj]);
            tj += j;
          }
          Dft<R, true>::run(x);
          if (ll == line_e) {
            float* d = dst + j;
#pragma unroll
            for (int q = 0; q < R; ++q) d[q * m] = scale * x[q].re;
          } else {
#pragma unroll
            for (int q = 0; q < R; ++q) {
              // nl_products of these kinds
              const float u = scale * x[q].re;
              float v = u * u;
              if (poly) {
                float pw = 1.f;
                v = 0.f;
#pragma unroll 1
                for (int e = 0; e < g.nl.npoly; ++e) {
                  v += g.nl.poly[e] * pw;
                  pw *= u;
                }
              }
              x[q] = cf{v, 0.f};
            }
            Dft<R, false>::run(x);
            const int to = o + j * R;
#pragma unroll
            for (int q = 0; q < R; ++q) sm[to + q] = x[q];
          }
        }
      });
      if (!step) break;
      __syncthreads();
      {
        const int t2 = a;
        a = b;
        b = t2;
      }
#pragma unroll 1
      for (int e = 1; e < np; ++e) pass(fwd, pick(e, f0, f1, f2, f3), 1);
      const int mode = (order == 1 ? ST1 : order == 2 ? ST2A : order == 3 ? ST3A : ST4A) + i;
#pragma unroll 1
      for (int k = tid; k < nz; k += nthr) {
        const cf v = sm[a + k];
        const cf nh = combine_core(g.nl, mode3d_at(g.nl, 0, 0, k), 0, [&](int, int) { return v; });
        cf n0 = nh;
        if (i == 0) sm[iN0 + k] = nh;
        else n0 = sm[iN0 + k];
        const float* tb = reinterpret_cast<const float*>(sm + iTB);
        with_stage_mode(mode, [&](auto m) {
          stage_core<decltype(m)::value>(e_im, nz, tb, k, k, sm + iU, sm + iS, sm + iSA, sm + iAC, n0, nh);
        });
      }
      __syncthreads();
    }
    const int s = iU;
    iU = iS;
    iS = s;
  }
}

hipError_t launch_g1d(const GfftCfg& c, G1dArgs a, hipStream_t st) {
  const NL3DArgs& nl = a.nl;
  const int most = g1d_lines(nl.channels, nl.nf, nl.np);
  if (nl.dims != 1 || c.n != nl.N || a.nsteps < 1 || a.order < 0 || a.order > 4) return hipErrorInvalidValue;
  const size_t tab = sizeof(float) * (size_t)a.lin_channels * a.ncoef * nl.NZ;
  const size_t lds = g1d_lds(nl.N, nl.channels, most, a.order) + tab;
  if (lds > GFFT_LDS_MAX) return hipErrorInvalidValue;
  a.d = gfft_dev(c);
  a.df = gfft_dev(c, true);
  const long long traj = nl.ninst / nl.channels;
  // one field, one product, register radices, two passes or more
  bool single = (nl.kind == NL_POLY || nl.kind == NL_GRADNORM || nl.kind == NL_CONV_CONS) && nl.channels == 1 && nl.nf == 1 && nl.np == 1 && a.order >= 1 && c.npass >= 2 &&
                (!a.roundtrip || a.nsteps == 1);
  single = single && c.npass <= G1S_MAX_PASS;
  for (int i = 0; i < c.npass; ++i) single = single && g1s_radix(c.radix[i]);
  if (single) {
    // two lines side by side; a thread per butterfly of the first pass
    const int work = 2 * nl.N / c.radix[0];
    const int wg = work <= 64 ? 64 : work <= 128 ? 128 : work <= 256 ? 256 : G1D_WG_MAX;
    const size_t l = sizeof(cf) * ((size_t)5 * nl.N + (size_t)g1d_spectra(a.order) * nl.NZ) + tab;
    if (l <= GFFT_LDS_MAX) {
      hipLaunchKernelGGL(g1s_kernel, dim3((unsigned)traj), dim3(wg), l, st, a);
      return hipGetLastError();
    }
  }
  int widest = 2;
  for (int i = 0; i < c.npass; ++i) widest = c.radix[i] > widest && c.radix[i] <= 19 ? c.radix[i] : widest;
  // a thread per butterfly of the widest pass and line, one wavefront at least
  const int work = nl.N * most / widest;
  const int wg = work <= 64 ? 64 : work <= 128 ? 128 : work <= 256 ? 256 : G1D_WG_MAX;
  if (gfft_big(c))
    hipLaunchKernelGGL(g1d_kernel<19>, dim3((unsigned)traj), dim3(wg), lds, st, a);
  else
    hipLaunchKernelGGL(g1d_kernel<8>, dim3((unsigned)traj), dim3(wg), lds, st, a);
  return hipGetLastError();
}

}  // namespace exmi
