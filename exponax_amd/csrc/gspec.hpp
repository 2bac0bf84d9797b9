// Launch interface of the fused passes of the runtime-size plans (gspec.hip).
#pragma once
#include "gfft.hpp"
#include "spectral3d.hpp"

namespace exmi {

// The fields of every instance with their first inverse pass (the lines of
// the outermost axis, 2-D and 3-D): S -> F, planes kz < kkeep and, in 3-D,
// rows |ky| <= a.kmax only.
hipError_t launch_gfields(const GfftCfg& c, const NL3DArgs& a, const cf* S, cf* F, float scale, int kkeep,
                          const cf* tw, hipStream_t st);

// The rows along the last axis (2-D and 3-D): every field's c2r (times
// scale), the pointwise products, and the products' r2c: F -> P, of which
// kz < kkeep is read and stored. gprod_fits: whether one pair of rows of all
// fields of a trajectory fits LDS.
bool gprod_fits(const GfftCfg& c, const NL3DArgs& a);
hipError_t launch_gprod(const GfftCfg& c, const NL3DArgs& a, const cf* F, cf* P, float scale, int kkeep,
                        const cf* tw, hipStream_t st);

// The last forward axis of the products P (2-D and 3-D) with the combine and
// the stage st (N0out: also store N_hat, the first stage's): lines kz < kkeep
// and, in 3-D, |ky| <= cut hold products.
bool gstage_fits(const GfftCfg& c, const NL3DArgs& a);
hipError_t launch_gstage(const GfftCfg& c, const NL3DArgs& a, const Stage3DArgs& st, const cf* P, cf* N0out,
                         int kkeep, int cut, const cf* tw, hipStream_t stream);

// 1-D: `nsteps` whole ETDRK steps (orders 0-4) of every trajectory in one launch.
struct G1dArgs {
  NL3DArgs nl;
  GfftDev d, df;  // the inverse's passes (and the forward's); df the same in reverse order
  int order, ncoef, lin_batch, lin_channels, e_im;
  int nsteps;
  int every;    // written: the states after every, 2 every, ... steps and the last one
  float* last;  // where the last one goes, or null: in its turn
  int roundtrip;  // 1: every step transforms the emitted state forward again, 0: the spectrum is carried
  const float* tables;
  const cf* tw;
  const float* u0;
  long long u0_bs;
  float* out;  // the written states of trajectory b at out + b * out_bs (last + b * out_bs), one out_ts apart
  long long out_bs, out_ts;
};
bool g1d_fits(int N, int channels, int nf, int np, int order, int lin_channels, int ncoef);
hipError_t launch_g1d(const GfftCfg& c, G1dArgs a, hipStream_t st);

}  // namespace exmi
