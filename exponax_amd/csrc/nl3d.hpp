// Pointwise pieces of the multi-pass plans, shared by the 3-D kernels
// (spectral3d.hip) and the runtime-size ones (gspec.hip): the wavenumbers of
// an entry, the spectral fields, the pointwise products, the combination of
// the product spectra into N_hat, and the ETDRK stage combinations.
#pragma once
#include <type_traits>

#include "exmi_internal.hpp"
#include "fft1d.hpp"
#include "spectral3d.hpp"

namespace exmi {

struct Mode3D {
  float kx, ky, kz;  // kappa = (2 pi / L) k along the three axes (0 on absent ones)
  bool keep;         // |k| <= kmax on every axis
  bool zero;         // the mean mode
  bool inj;          // the Kolmogorov forcing mode
};

// Signed wavenumber of index i on a full (fftfreq) axis of n points: i for
// i <= (n - 1) / 2, else i - n (even n: the Nyquist index n/2 is -n/2).
__device__ __forceinline__ int signed_k(int i, int n) { return i <= (n - 1) / 2 ? i : i - n; }

__device__ __forceinline__ Mode3D mode3d_at(const NL3DArgs& a, int ix, int iy, int iz) {
  const int kx = signed_k(ix, a.nx), ky = signed_k(iy, a.ny);
  Mode3D m;
  m.kx = a.kscale * (float)kx;
  m.ky = a.kscale * (float)ky;
  m.kz = a.kscale * (float)iz;
  m.keep = (kx < 0 ? -kx : kx) <= a.kmax && (ky < 0 ? -ky : ky) <= a.kmax && iz <= a.kmax;
  m.zero = kx == 0 && ky == 0 && iz == 0;
  m.inj = a.inj_axis == 2 ? (kx == 0 && ky == 0 && iz == a.inj_mode) : (kx == 0 && ky == a.inj_mode && iz == 0);
  return m;
}

__device__ __forceinline__ Mode3D mode3d(const NL3DArgs& a, long long k) {
  const int iz = (int)(k % a.NZ);
  const long long r = k / a.NZ;
  return mode3d_at(a, (int)(r / a.ny), (int)(r % a.ny), iz);
}

// kappa of spatial derivative d (axis 3 - D + d)
__device__ __forceinline__ float kap_d(const NL3DArgs& a, const Mode3D& m, int d) {
  const int axis = 3 - a.dims + d;
  return axis == 0 ? m.kx : axis == 1 ? m.ky : m.kz;
}

__device__ __forceinline__ cf imul(float kap, cf w) { return cf{-kap * w.im, kap * w.re}; }

// Field f of instance inst at entry k (mode m) of the spectra S.
__device__ __forceinline__ cf field_at(const NL3DArgs& a, const cf* __restrict__ S, long long inst, int f,
                                       long long k, const Mode3D& m) {
  if (!m.keep) return cf{0.f, 0.f};
  if (a.kind == NL_PROJ3D && f == 1) {
    // the curl component omega_c = (i kappa x u_hat)_c of the dealiased
    // spectra (_projected_convection.py:8-16, 120-123); field 0 is u_c
    const long long b = (inst - inst % a.channels) * a.Nr + k;
    const int c = (int)(inst % a.channels);
    const cf w0 = S[b], w1 = S[b + a.Nr], w2 = S[b + 2 * a.Nr];
    return c == 0 ? imul(m.ky, w2) - imul(m.kz, w1) : c == 1 ? imul(m.kz, w0) - imul(m.kx, w2)
                                                           : imul(m.kx, w1) - imul(m.ky, w0);
  }
  const cf w = S[inst * a.Nr + k];
  if (a.kind == NL_GRADNORM) return imul(kap_d(a, m, f), w);
  if (a.kind == NL_CONV_NONCONS || a.kind == NL_GENERAL) return f == 0 ? w : imul(kap_d(a, m, f - 1), w);
  if (a.kind == NL_VORT) {
    // 2-D (_vorticity_convection.py:78-99): psi = Laplace^-1 omega (1 at
    // the mean mode), u = d_y psi, v = -d_x psi, omega_x, omega_y; x is
    // axis 1, y the last axis
    const float kx = m.ky, ky = m.kz;
    const float lap = -(kx * kx + ky * ky);
    const cf psi = (lap == 0.f ? 1.f : 1.f / lap) * w;
    return f == 0 ? imul(ky, psi) : f == 1 ? imul(kx, w) : f == 2 ? imul(-kx, psi) : imul(ky, w);
  }
  return w;
}

// N_hat of channel ch at mode m from the product spectra, ph(c, j) product j
// of channel c there.
template <class PH>
__device__ __forceinline__ cf combine_core(const NL3DArgs& a, const Mode3D& m, int ch, PH&& ph) {
  cf r = cf{0.f, 0.f};
  switch (a.kind) {
    case NL_POLY:
      r = a.poly_lap ? (a.scale * -(m.kx * m.kx + m.ky * m.ky + m.kz * m.kz)) * ph(ch, 0) : ph(ch, 0);
      break;
    case NL_GRADNORM: r = (a.zero_mode_fix && m.zero) ? cf{0.f, 0.f} : (-0.5f * a.scale) * ph(ch, 0); break;
    case NL_CONV_CONS: {
      cf acc = cf{0.f, 0.f};
      for (int j = 0; j < a.dims; ++j) acc = acc + imul(kap_d(a, m, j), ph(ch, j));
      r = (-0.5f * a.scale) * acc;
      break;
    }
    case NL_CONV_NONCONS:
    case NL_VORT: r = -a.scale * ph(ch, 0); break;
    case NL_GENERAL: {
      const float cg = (a.zero_mode_fix && m.zero) ? 0.f : 0.5f * a.g2;
      const cf p0 = ph(ch, 0);
      r = a.g0 * p0 + imul(0.5f * a.g1 * (m.kx + m.ky + m.kz), p0) + cg * ph(ch, 1);
      break;
    }
    case NL_PROJ3D: {
      // Leray projection (_leray.py:86-103): c + i kappa_c p with
      // p = -div / Laplace = (i kappa . c) / |kappa|^2 (p = 0 at the mean mode)
      const cf p0 = ph(0, 0), p1 = ph(1, 0), p2 = ph(2, 0);
      const cf div = imul(m.kx, p0) + imul(m.ky, p1) + imul(m.kz, p2);
      const float k2 = m.kx * m.kx + m.ky * m.ky + m.kz * m.kz;
      const cf pr = k2 != 0.f ? (1.f / k2) * div : cf{0.f, 0.f};
      r = (ch == 0 ? p0 : ch == 1 ? p1 : p2) + imul(ch == 0 ? m.kx : ch == 1 ? m.ky : m.kz, pr);
      break;
    }
    default: r = ph(ch, 0);
  }
  cf out = m.keep ? r : cf{0.f, 0.f};
  if ((a.kind == NL_PROJ3D || a.kind == NL_VORT) && m.inj && ch == 0) out = out + cf{a.inj_value, 0.f};
  return out;
}

// N_hat at entry idx (instance idx / Nr) from the product spectra PH.
__device__ __forceinline__ cf combine_at(const NL3DArgs& a, const cf* __restrict__ PH, long long idx) {
  const long long inst = idx / a.Nr, k = idx % a.Nr;
  const int ch = (int)(inst % a.channels);
  const cf* ph = PH + (inst - ch) * a.np * a.Nr + k;
  return combine_core(a, mode3d(a, k), ch, [&](int c, int j) { return ph[((long long)c * a.np + j) * a.Nr]; });
}

// One value, or two grid points' values side by side.
struct v2 {
  float a, b;
};
__device__ __forceinline__ v2 operator+(v2 x, v2 y) { return v2{x.a + y.a, x.b + y.b}; }
__device__ __forceinline__ v2 operator-(v2 x, v2 y) { return v2{x.a - y.a, x.b - y.b}; }
__device__ __forceinline__ v2 operator*(v2 x, v2 y) { return v2{x.a * y.a, x.b * y.b}; }
__device__ __forceinline__ v2 operator*(float s, v2 y) { return v2{s * y.a, s * y.b}; }
template <class V>
__device__ __forceinline__ V splat(float s);
template <>
__device__ __forceinline__ float splat<float>(float s) {
  return s;
}
template <>
__device__ __forceinline__ v2 splat<v2>(float s) {
  return v2{s, s};
}

// The pointwise products of one trajectory at one grid point: fld(c, f) field
// f of channel c, out(c, j, value) product j of channel c.
template <class V, class Fld, class Out>
__device__ __forceinline__ void nl_products(const NL3DArgs& a, Fld&& fld, Out&& out) {
  const int C = a.channels;
  switch (a.kind) {
    case NL_POLY:
      for (int c = 0; c < C; ++c) {
        const V u = fld(c, 0);
        V pw = splat<V>(1.f), acc = splat<V>(0.f);
        for (int i = 0; i < a.npoly; ++i) {
          acc = acc + a.poly[i] * pw;
          pw = pw * u;
        }
        out(c, 0, acc);
      }
      break;
    case NL_GRADNORM:
      for (int c = 0; c < C; ++c) {
        V acc = splat<V>(0.f);
        for (int d = 0; d < a.dims; ++d) {
          const V g = fld(c, d);
          acc = acc + g * g;
        }
        out(c, 0, acc);
      }
      break;
    case NL_CONV_CONS:
      for (int c = 0; c < C; ++c) {
        const V u = fld(c, 0);
        for (int j = 0; j < a.dims; ++j) out(c, j, u * fld(j, 0));
      }
      break;
    case NL_CONV_NONCONS:
      for (int c = 0; c < C; ++c) {
        V acc = splat<V>(0.f);
        for (int j = 0; j < a.dims; ++j) acc = acc + fld(j, 0) * fld(c, 1 + j);
        out(c, 0, acc);
      }
      break;
    case NL_GENERAL:
      for (int c = 0; c < C; ++c) {
        const V u = fld(c, 0);
        V gs = splat<V>(0.f), g2 = splat<V>(0.f);
        for (int d = 0; d < a.dims; ++d) {
          const V g = fld(c, 1 + d);
          gs = gs + g;
          g2 = g2 + g * g;
        }
        out(c, 0, a.prod_nc ? u * gs : u * u);
        out(c, 1, g2);
      }
      break;
    case NL_VORT:
      for (int c = 0; c < C; ++c) out(c, 0, fld(c, 0) * fld(c, 1) + fld(c, 2) * fld(c, 3));
      break;
    case NL_GRAY_SCOTT: {
      const V u0 = fld(0, 0), u1 = fld(1, 0);
      const V uvv = u0 * u1 * u1;
      out(0, 0, a.feed * (splat<V>(1.f) - u0) - uvv);
      out(1, 0, -(a.feed + a.kill) * u1 + uvv);
      break;
    }
    case NL_BZ: {
      const V u0 = fld(0, 0), u1 = fld(1, 0), u2 = fld(2, 0);
      out(0, 0, u0 + u1 - u0 * u1 - u0 * u0);
      out(1, 0, u2 - u1 - u0 * u1);
      out(2, 0, u0 - u2);
      break;
    }
    case NL_PROJ3D:
      for (int c = 0; c < 3; ++c) {  // (u x omega)_c
        const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
        out(c, 0, fld(c1, 0) * fld(c2, 1) - fld(c2, 0) * fld(c1, 1));
      }
      break;
    default:
      for (int c = 0; c < C; ++c) out(c, 0, splat<V>(0.f));
  }
}

// Stages that read the first nonlinear term N0, and those that read the
// latest one NC.
__device__ __forceinline__ bool stage_reads_n0(int m) {
  return m == ST1 || m == ST2A || m == ST2B || m == ST3A || m == ST3B || m == ST4A || m == ST4C;
}
__device__ __forceinline__ bool stage_reads_nc(int m) { return !(m == ST1 || m == ST2A || m == ST3A || m == ST4A); }

// The coefficient table of instance (trajectory traj, channel ch).
__device__ __forceinline__ const float* stage_table(const Stage3DArgs& a, long long traj, long long ch) {
  return a.tables +
         ((a.lin_batch > 1 ? traj : 0) * a.lin_channels + (a.lin_channels > 1 ? ch : 0)) * (long long)a.ncoef * a.nr;
}

// The stage combination of stage MODE at entry idx (mode k of its instance,
// tb the instance's coefficient table) with the nonlinear terms n0 (N0) and
// nc (NC) given; U0, S, S1, A as in Stage3DArgs. Returns the new S[idx].
template <int MODE>
__device__ __forceinline__ cf stage_core(int e_im, long long nr, const float* tb, long long k, long long idx,
                                         const cf* U0, cf* S, cf* S1, cf* A, cf n0, cf nc) {
  auto c = [&](int i) { return tb[(long long)i * nr + k]; };
  // coefficient i (0: E, 1: E_half for orders 3-4) times x, complex when L is
  auto cmul = [&](int i, cf x) -> cf {
    const float er = c(i);
    if (e_im < 0) return er * x;
    const float ei = c(e_im + i);
    return cf{fmaf(er, x.re, -ei * x.im), fmaf(er, x.im, ei * x.re)};
  };
  auto emul = [&](cf x) -> cf { return cmul(0, x); };
  cf r;
  if constexpr (MODE == ST1 || MODE == ST2A) {
    r = emul(U0[idx]) + c(1) * n0;
  } else if constexpr (MODE == ST2B) {
    r = S[idx] + c(2) * (nc - n0);
  } else if constexpr (MODE == ST3A) {
    const cf u0 = U0[idx];
    A[idx] = emul(u0) + c(4) * n0;
    r = cmul(1, u0) + c(2) * n0;
  } else if constexpr (MODE == ST3B) {
    const cf u0 = U0[idx];
    A[idx] = A[idx] + c(5) * nc;
    r = emul(u0) + c(3) * (2.f * nc - n0);
  } else if constexpr (MODE == ST3C) {
    r = A[idx] + c(6) * nc;
  } else if constexpr (MODE == ST4A) {
    const cf u0 = U0[idx];
    A[idx] = emul(u0) + c(3) * n0;
    r = cmul(1, u0) + c(2) * n0;
    S1[idx] = r;
  } else if constexpr (MODE == ST4B) {
    const cf u0 = U0[idx];
    A[idx] = A[idx] + (2.f * c(4)) * nc;
    r = cmul(1, u0) + c(2) * nc;
  } else if constexpr (MODE == ST4C) {
    A[idx] = A[idx] + (2.f * c(4)) * nc;
    r = cmul(1, S1[idx]) + c(2) * (2.f * nc - n0);
  } else {
    static_assert(MODE == ST4D, "stage mode");
    r = A[idx] + c(5) * nc;
  }
  S[idx] = r;
  return r;
}

// Calls f(std::integral_constant<int, mode>) for the runtime stage mode.
template <class F>
__device__ __forceinline__ void with_stage_mode(int mode, F&& f) {
  switch (mode) {
    case ST1: f(std::integral_constant<int, ST1>{}); break;
    case ST2A: f(std::integral_constant<int, ST2A>{}); break;
    case ST2B: f(std::integral_constant<int, ST2B>{}); break;
    case ST3A: f(std::integral_constant<int, ST3A>{}); break;
    case ST3B: f(std::integral_constant<int, ST3B>{}); break;
    case ST3C: f(std::integral_constant<int, ST3C>{}); break;
    case ST4A: f(std::integral_constant<int, ST4A>{}); break;
    case ST4B: f(std::integral_constant<int, ST4B>{}); break;
    case ST4C: f(std::integral_constant<int, ST4C>{}); break;
    case ST4D: f(std::integral_constant<int, ST4D>{}); break;
  }
}

// The stage combination at entry idx with the nonlinear terms n0 (N0) and
// nc (NC) given.
__device__ __forceinline__ void stage_at(const Stage3DArgs& a, long long idx, cf n0, cf nc) {
  const long long inst = idx / a.nr, k = idx % a.nr;
  const float* tb = stage_table(a, inst / a.channels, inst % a.channels);
  with_stage_mode(a.mode, [&](auto m) {
    stage_core<decltype(m)::value>(a.e_im, a.nr, tb, k, idx, a.U0, a.S, a.S1, a.A, n0, nc);
  });
}

}  // namespace exmi
