// Kernels and C ABI of the learned corrector (see corrector.hpp): forward
// (inference, or training with stored intermediates), input-gradient pass,
// weight-gradient passes and the deterministic reduction of their per-wave
// partial sums.
#include <hip/hip_runtime.h>

#include "../../include/exmi.h"
#include "corrector.hpp"

namespace exmi {
int set_error(int code, const char* msg);
}

namespace exmi {
namespace cnn {

// The hidden layers' A fragments from the parameters: consecutive threads read
// consecutive weights, the bfloat16 values go to their fragment slots.
template <bool T>
__device__ __forceinline__ void pack_frags(__bf16* dst, const float* __restrict__ p, int tid, int nthr) {
  for (int i = tid; i < 3 * CH * CH * KW; i += nthr) {
    const int L = i / (CH * CH * KW), r = i - L * (CH * CH * KW);
    const int co = r / (CH * KW), q = r - co * (CH * KW), ci = q / KW, k = q - ci * KW;
    dst[frag_slot<T>(L, co, ci, k)] = static_cast<__bf16>(p[OW2 + L * (OW3 - OW2) + r]);
  }
}

// The forward fragments once, for rollouts that call the network every step.
__global__ void pack_kernel(const float* __restrict__ p, bf16x8* __restrict__ frag) {
  pack_frags<false>(reinterpret_cast<__bf16*>(frag), p, blockIdx.x * blockDim.x + threadIdx.x,
                    gridDim.x * blockDim.x);
}

struct Args {
  const float* params;
  const bf16x8* frag;  // packed forward fragments (pack_kernel), or null: each workgroup packs its own
  const float* x;      // forward input, sample i at x + i * xs
  float* y;            // forward output, sample i at y + i * ys
  long long xs, ys;    // sample strides in floats (N when contiguous)
  const float* dy;     // backward: cotangent of y (count, N)
  float* dx;           // backward: cotangent of x, or null
  Workspace ws;        // training intermediates, or all null
  long long count;
};

template <int N>
struct Lds {
  Edge e;
  bf16x8 frag[NFRAG];
  __attribute__((aligned(16))) __bf16 act[WAVES][2][N * LDA];
  float vec[WAVES][N];
};

// The forward pass's workgroup: where one layer's output tiles are all
// formed before any is written (N / 32 tiles, all taken together), a wave
// keeps one activation buffer and overwrites it in place (its reads of a
// layer's input precede its writes of the output in program order, and a
// wave's LDS operations complete in order); the LDS saved holds eight waves
// per workgroup, two workgroups per CU: four waves per SIMD to overlap
// one wave's GELU with another's matrix-core work. With no more samples than
// the chip has SIMDs, workgroups of four waves instead, one wave per SIMD.
// One wavefront takes about 15 us per sample, so a batch below the chip's
// size is spread over as many wavefronts as it has samples: 512 samples of 64
// points 24 us, against 51 us at four samples per wave on 16 CUs; 8192 samples 38.5 us with two samples per wave in 512
// workgroups against 40.0 us with four in 256.
template <int N>
struct FwdCfg {
  static constexpr int NB = N / 32 == tiles_together<N>() ? 1 : 2;  // activation buffers per wave
  static constexpr int NW = NB == 1 ? 8 : WAVES;                    // waves per workgroup
};

template <int N, int NW>
struct LdsFwd {
  Edge e;
  bf16x8 frag[NFRAG];
  __attribute__((aligned(16))) __bf16 act[NW][FwdCfg<N>::NB][N * LDA];
  float vec[NW][N];
};

template <int N, bool TRAIN, int NW>
__global__ void __launch_bounds__(64 * NW) forward_kernel(Args a) {
  constexpr int NB = FwdCfg<N>::NB;
  __shared__ LdsFwd<N, NW> sh;
  load_edge(sh.e, a.params);
  if (a.frag) {
    for (int i = threadIdx.x; i < NFRAG; i += 64 * NW) sh.frag[i] = a.frag[i];
  } else {
    pack_frags<false>(reinterpret_cast<__bf16*>(sh.frag), a.params, threadIdx.x, 64 * NW);
  }
  __syncthreads();
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const bf16x8* W = sh.frag;
  float* xs = sh.vec[w];
  // every wave runs the same bounded loop over its samples
  for (long long smp = (long long)blockIdx.x * NW + w; smp < a.count; smp += (long long)gridDim.x * NW) {
    for (int p = lane; p < N; p += 64) xs[p] = a.x[smp * a.xs + p];
    wave_sync();
    forward_sample<N, TRAIN>(sh.e, W, xs, sh.act[w][0], sh.act[w][NB - 1], a.y + smp * a.ys, a.ws, smp, a.count,
                             lane);
  }
}

// Input-gradient pass: deltas of layers 4..1 (stored for the weight pass)
// and dx = dy + the transposed first layer.
template <int N>
__global__ void __launch_bounds__(64 * WAVES) backward_data_kernel(Args a) {
  __shared__ Lds<N> sh;
  load_edge(sh.e, a.params);
  pack_frags<true>(reinterpret_cast<__bf16*>(sh.frag), a.params, threadIdx.x, 64 * WAVES);
  __syncthreads();
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int c = lane & 31, h = lane >> 5;
  const bf16x8* W = sh.frag;
  const Edge& e = sh.e;
  float* dys = sh.vec[w];
  const Workspace ws = a.ws;
  const long long cnt = a.count;
  for (long long smp = (long long)blockIdx.x * WAVES + w; smp < cnt; smp += (long long)gridDim.x * WAVES) {
    for (int p = lane; p < N; p += 64) dys[p] = a.dy[smp * N + p];
    wave_sync();
    __bf16* in = sh.act[w][0];
    __bf16* out = sh.act[w][1];
    // layer 5 transposed (VALU): da4[p][ci] = sum_k W5[ci][k] dy[p - k + 2]
    for (int p = lane; p < N; p += 64) {
      float dv[KW];
#pragma unroll
      for (int k = 0; k < KW; ++k) dv[k] = dys[(p - k + 2) & (N - 1)];
      __bf16 outv[CH];
#pragma unroll
      for (int ci = 0; ci < CH; ++ci) {
        float da = 0.f;
#pragma unroll
        for (int k = 0; k < KW; ++k) da = fmaf(e.w5[ci * KW + k], dv[k], da);
        const long long o = ((3 * cnt + smp) * CH + ci) * N + p;
        const __bf16 d = static_cast<__bf16>(da * gelu_grad(ws.Z[o]));
        outv[ci] = d;
        ws.D[o] = d;
      }
#pragma unroll
      for (int g = 0; g < CH / 8; ++g) {
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = outv[8 * g + i];
        *reinterpret_cast<bf16x8*>(in + p * LDA + 8 * g) = v;
      }
    }
    wave_sync();
    // layers 4, 3, 2 transposed on the matrix cores -> deltas of layers 3, 2, 1
    constexpr int NTL = tiles_together<N>();
#pragma unroll
    for (int L = 2; L >= 0; --L) {
#pragma unroll
      for (int t0 = 0; t0 < N / 32; t0 += NTL) {
        f32x16 acc[NTL];
        conv_tiles<N, true, NTL>(acc, [&](int s) { return W[(L * KSTEPS + s) * 64 + lane]; }, in, t0, lane);
#pragma unroll
        for (int q = 0; q < NTL; ++q) {
          const int pos = (t0 + q) * 32 + c;
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            bf16x4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int ci = 8 * j + 4 * h + r;
              const long long o = (((long long)L * cnt + smp) * CH + ci) * N + pos;
              const __bf16 d = static_cast<__bf16>(acc[q][4 * j + r] * gelu_grad(ws.Z[o]));
              v[r] = d;
              ws.D[o] = d;
            }
            *reinterpret_cast<bf16x4*>(out + pos * LDA + 8 * j + 4 * h) = v;
          }
        }
      }
      wave_sync();
      __bf16* tmp = in;
      in = out;
      out = tmp;
    }
    // layer 1 transposed (VALU): dx = dy + sum_{co,k} W1[co][k] d1[p - k + 2][co]
    if (a.dx) {
      for (int p = lane; p < N; p += 64) {
        float g = dys[p];
#pragma unroll
        for (int k = 0; k < KW; ++k) {
          const __bf16* row = in + ((p - k + 2) & (N - 1)) * LDA;
#pragma unroll
          for (int q = 0; q < CH / 8; ++q) {
            const bf16x8 v = *reinterpret_cast<const bf16x8*>(row + 8 * q);
#pragma unroll
            for (int i = 0; i < 8; ++i) g = fmaf(e.w1[(8 * q + i) * KW + k], static_cast<float>(v[i]), g);
          }
        }
        a.dx[smp * N + p] = g;
      }
    }
    wave_sync();
  }
}

// Weight gradients of the 32 -> 32 layers on the matrix cores:
// dW[co][ci][k] = sum_{samples, p} d[co][p] a[ci][(p + k - 2) mod N],
// M = co, N = ci (one tile per k), K = positions. Bias gradients on the
// VALU. One workgroup takes one layer; its waves' sums are added in LDS, in
// wave order, so memory holds one set of partial sums per workgroup.
template <int N>
__device__ __forceinline__ void wgrad_hidden(const Args& a, int L, float* red, float* part) {
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int c = lane & 31, h = lane >> 5;
  const Workspace ws = a.ws;
  const long long cnt = a.count;
  f32x16 acc[KW];
#pragma unroll
  for (int k = 0; k < KW; ++k) acc[k] = f32x16{};
  float bsum = 0.f;
  for (long long smp = (long long)blockIdx.x * WAVES + w; smp < cnt; smp += (long long)gridDim.x * WAVES) {
    const __bf16* D = ws.D + (((long long)(L + 1) * cnt + smp) * CH + c) * N;  // delta of layer L + 2
    const __bf16* A = ws.A + (((long long)L * cnt + smp) * CH + c) * N;        // its input a_{L+1}
#pragma unroll
    for (int q = 0; q < N / 16; ++q) {
      const int p0 = 16 * q + 8 * h;
      const bf16x8 av = *reinterpret_cast<const bf16x8*>(D + p0);
      // positions p0 - 8 .. p0 + 15 of the input: every tap's eight are among them
      const bf16x8 lo = *reinterpret_cast<const bf16x8*>(A + ((p0 - 8) & (N - 1)));
      const bf16x8 mid = *reinterpret_cast<const bf16x8*>(A + p0);
      const bf16x8 hi = *reinterpret_cast<const bf16x8*>(A + ((p0 + 8) & (N - 1)));
#pragma unroll
      for (int i = 0; i < 8; ++i) bsum += static_cast<float>(av[i]);
#pragma unroll
      for (int k = 0; k < KW; ++k) {
        bf16x8 bv;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int o = i + k - 2;
          bv[i] = o < 0 ? lo[o + 8] : o < 8 ? mid[o] : hi[o - 8];
        }
        acc[k] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av, bv, acc[k], 0, 0, 0);
      }
    }
  }
  // bias: lanes c and c + 32 hold the two halves of the positions of channel c
  bsum += __shfl_xor(bsum, 32);
  for (int t = 0; t < WAVES; ++t) {
    if (w == t) {
#pragma unroll
      for (int k = 0; k < KW; ++k)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int co = 8 * (i >> 2) + 4 * h + (i & 3), at = (co * CH + c) * KW + k;
          red[at] = t == 0 ? acc[k][i] : red[at] + acc[k][i];
        }
      if (h == 0) red[CH * CH * KW + c] = t == 0 ? bsum : red[CH * CH * KW + c] + bsum;
    }
    __syncthreads();
  }
  // weights and biases of a layer are neighbours in the parameter vector
  float* out = part + OW2 + L * (OW3 - OW2);
  for (int i = threadIdx.x; i < OW3 - OW2; i += 64 * WAVES) out[i] = red[i];
}

// Weight gradients of the 1 -> 32 and 32 -> 1 layers (VALU):
// dW1[co][k] = sum d1[co][p] a0[p + k - 2], db1[co] = sum d1[co][p],
// dW5[ci][k] = sum dy[p] a4[ci][p + k - 2] = sum a4[ci][q] dy[q - k + 2],
// db5 = sum dy[p]. Output j = lane + 64 m (0..159 dW1, 160..191 db1, 192..351
// dW5, 352 db5) is one row of bfloat16 against a shifted vector in LDS; one
// workgroup takes one m.
constexpr int EDGE_M = 6;
template <int N>
__device__ __forceinline__ void wgrad_edge(const Args& a, int m, float* red, float* part) {
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64;
  const Workspace ws = a.ws;
  const long long cnt = a.count;
  float* v0 = red + w * 3 * N;  // a0, dy, ones
  const int j = lane + 64 * m;
  int vec = 2, sh = 0;
  long long row = -1;  // row offset of sample 0 from its array (D of layer 1, or A of layer 4)
  bool fromA = false;
  if (j < 160) {
    row = (long long)(j / KW) * N;
    vec = 0;
    sh = j % KW - 2;
  } else if (j < 192) {
    row = (long long)(j - 160) * N;
  } else if (j < 352) {
    row = (3 * cnt * CH + (j - 192) / KW) * N;
    fromA = true;
    vec = 1;
    sh = 2 - (j - 192) % KW;
  }
  float acc = 0.f;
  for (long long smp = (long long)blockIdx.x * WAVES + w; smp < cnt; smp += (long long)gridDim.x * WAVES) {
    wave_sync();
    for (int p = lane; p < N; p += 64) {
      v0[p] = static_cast<float>(ws.A0[smp * N + p]);
      v0[N + p] = a.dy[smp * N + p];
      v0[2 * N + p] = 1.f;
    }
    wave_sync();
    float s = 0.f;
    if (row >= 0) {
      const __bf16* r = (fromA ? ws.A : ws.D) + row + smp * CH * N;
#pragma unroll
      for (int q = 0; q < N / 8; ++q) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(r + 8 * q);
#pragma unroll
        for (int i = 0; i < 8; ++i)
          s = fmaf(static_cast<float>(x[i]), v0[vec * N + ((8 * q + i + sh) & (N - 1))], s);
      }
    } else if (j == 352) {
      for (int p = 0; p < N; ++p) s += v0[N + p];
    }
    acc += s;
  }
  __syncthreads();
  red[w * 64 + lane] = acc;
  __syncthreads();
  if (w == 0 && j <= 352) {
    float s = red[lane];
#pragma unroll
    for (int t = 1; t < WAVES; ++t) s += red[t * 64 + lane];
    part[j < 160 ? OW1 + j : j < 192 ? OB1 + j - 160 : j < 352 ? OW5 + j - 192 : OB5] = s;
  }
}

// grid (groups, 3 hidden layers + EDGE_M slices of the edge layers): the
// layers and slices are independent, so each has its own workgroups. What
// bounds it at 512 samples is the 8 MB of partial sums and the latency of one
// sample's chain: 13.6 us and 4.3 us of reduction, against 25 + 24 us for the
// hidden and edge passes in turn and 16 us of reducing one set per wavefront.
template <int N>
__global__ void __launch_bounds__(64 * WAVES) wgrad_kernel(Args a) {
  __shared__ float red[CH * CH * KW + CH];
  static_assert(CH * CH * KW + CH >= WAVES * 3 * N && CH * CH * KW + CH == OW3 - OW2, "reduction buffer");
  float* part = a.ws.P + (long long)blockIdx.x * NPARAM;
  if (blockIdx.y < 3) wgrad_hidden<N>(a, blockIdx.y, red, part);
  else wgrad_edge<N>(a, blockIdx.y - 3, red, part);
}

// The workgroups' partial sums, added in a fixed order: each of the four
// waves of a workgroup adds every fourth set for 64 parameters, then the four
// sums are added in wave order. Deterministic for a given number of groups.
__global__ void __launch_bounds__(64 * WAVES) reduce_kernel(const float* __restrict__ partial, int groups,
                                                            float* __restrict__ out) {
  __shared__ float red[WAVES][64];
  const int w = threadIdx.x / 64, lane = threadIdx.x % 64, j = blockIdx.x * 64 + lane;
  float s = 0.f;
  if (j < NPARAM) {
#pragma unroll 8
    for (int g = w; g < groups; g += WAVES) s += partial[(long long)g * NPARAM + j];
  }
  red[w][lane] = s;
  __syncthreads();
  if (w == 0 && j < NPARAM) out[j] = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
}

// Workgroups of `waves` wavefronts: one sample per wavefront until
// `resident` workgroups fill the chip, then a loop over the rest.
int grid_for(long long count, int waves, int resident) {
  const long long g = (count + waves - 1) / waves;
  return g < 1 ? 1 : g > resident ? resident : (int)g;
}

template <int N, bool TRAIN>
hipError_t launch_forward_t(const Args& a, hipStream_t st) {
  constexpr int NW = FwdCfg<N>::NW;
  if (NW > WAVES && a.count <= 1024)
    hipLaunchKernelGGL((forward_kernel<N, TRAIN, WAVES>), dim3(grid_for(a.count, WAVES, 512)), dim3(64 * WAVES), 0, st,
                       a);
  else
    hipLaunchKernelGGL((forward_kernel<N, TRAIN, NW>), dim3(grid_for(a.count, NW, 512)), dim3(64 * NW), 0, st, a);
  return hipGetLastError();
}

template <int N>
hipError_t launch_forward(const Args& a, bool train, hipStream_t st) {
  return train ? launch_forward_t<N, true>(a, st) : launch_forward_t<N, false>(a, st);
}

template <int N>
hipError_t launch_backward(const Args& a, hipStream_t st) {
  hipLaunchKernelGGL((backward_data_kernel<N>), dim3(grid_for(a.count, WAVES, 512)), dim3(64 * WAVES), 0, st, a);
  hipLaunchKernelGGL((wgrad_kernel<N>), dim3(wgrad_groups(a.count), 3 + EDGE_M), dim3(64 * WAVES), 0, st, a);
  return hipGetLastError();
}

bool size_ok(int N) { return N == 32 || N == 64 || N == 128; }

}  // namespace cnn

// Internal entry points for the corrected rollout in abi.hip.
size_t cnn_frag_bytes() { return sizeof(cnn::bf16x8) * cnn::NFRAG; }

hipError_t cnn_pack(const float* params, void* frag, hipStream_t st) {
  hipLaunchKernelGGL(cnn::pack_kernel, dim3(16), dim3(256), 0, st, params, static_cast<cnn::bf16x8*>(frag));
  return hipGetLastError();
}

hipError_t cnn_forward_strided(const float* params, const void* frag, int N, long long count, const float* x,
                               long long xs, float* y, long long ys, hipStream_t st) {
  cnn::Args a{};
  a.params = params;
  a.frag = static_cast<const cnn::bf16x8*>(frag);
  a.x = x;
  a.y = y;
  a.xs = xs;
  a.ys = ys;
  a.count = count;
  return N == 32 ? cnn::launch_forward<32>(a, false, st)
                 : (N == 64 ? cnn::launch_forward<64>(a, false, st) : cnn::launch_forward<128>(a, false, st));
}

}  // namespace exmi

using namespace exmi::cnn;

extern "C" {

int64_t exmi_cnn_workspace_bytes(int32_t num_points, int32_t count) {
  return workspace_bytes(num_points, count);
}

int exmi_cnn_forward(const float* params, int32_t N, int32_t count, const float* x, float* y, void* workspace,
                     void* stream) {
  if (!params || !x || !y) return exmi::set_error(EXMI_ERR_INVALID, "exmi_cnn_forward: null argument");
  if (!size_ok(N)) return exmi::set_error(EXMI_ERR_UNSUPPORTED, "exmi_cnn_forward: num_points must be 32, 64 or 128");
  if (count <= 0) return EXMI_OK;
  hipStream_t st = (hipStream_t)stream;
  Args a{};
  a.params = params;
  a.x = x;
  a.y = y;
  a.xs = a.ys = N;
  a.count = count;
  const bool train = workspace != nullptr;
  if (train) a.ws = workspace_at(workspace, N, count);
  hipError_t e = N == 32 ? launch_forward<32>(a, train, st)
                         : (N == 64 ? launch_forward<64>(a, train, st) : launch_forward<128>(a, train, st));
  return e == hipSuccess ? EXMI_OK : exmi::set_error(EXMI_ERR_HIP, hipGetErrorString(e));
}

int exmi_cnn_backward(const float* params, int32_t N, int32_t count, const float* dy, float* dx, float* dparams,
                      void* workspace, void* stream) {
  if (!params || !dy || !dparams || !workspace)
    return exmi::set_error(EXMI_ERR_INVALID, "exmi_cnn_backward: null argument");
  if (!size_ok(N)) return exmi::set_error(EXMI_ERR_UNSUPPORTED, "exmi_cnn_backward: num_points must be 32, 64 or 128");
  if (count <= 0) return EXMI_OK;
  hipStream_t st = (hipStream_t)stream;
  Args a{};
  a.params = params;
  a.dy = dy;
  a.dx = dx;
  a.ws = workspace_at(workspace, N, count);
  a.count = count;
  hipError_t e = N == 32 ? launch_backward<32>(a, st)
                         : (N == 64 ? launch_backward<64>(a, st) : launch_backward<128>(a, st));
  if (e == hipSuccess) {
    hipLaunchKernelGGL(reduce_kernel, dim3((NPARAM + 63) / 64), dim3(64 * WAVES), 0, st, a.ws.P, wgrad_groups(count),
                       dparams);
    e = hipGetLastError();
  }
  return e == hipSuccess ? EXMI_OK : exmi::set_error(EXMI_ERR_HIP, hipGetErrorString(e));
}

}  // extern "C"
