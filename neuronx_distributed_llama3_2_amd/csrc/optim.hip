// Optimizer / gradient kernels over FLAT contiguous buffers (the native replacement of
// torch_xla's ZeroRedundancyOptimizer internals and of the reference's per-parameter Python
// loops: src/neuronx_distributed/utils/adamw_fp32_optim_params.py:91-155,
// src/neuronx_distributed/parallel_layers/grads.py:33-240).
//
// Parameters, fp32 master weights, Adam moments and gradients each live in ONE flat buffer
// (or one ZeRO-1 shard of it), so a whole optimizer step is a handful of launches regardless of
// the number of tensors:
//   * sumsq:  sum(x^2) (or max|x|) of a flat bf16/fp32 range -> fp32 partials -> one scalar
//             (the grad-norm; no per-tensor torch.norm launches);
//   * adamw:  fused decoupled-weight-decay Adam with bias correction, grad scaling (clip
//             coefficient read from device memory, so no host sync for clipping), fp32 master
//             update and bf16 copy-out of the model weights in the same pass.
#include "common.h"

#include <algorithm>

namespace nxd {
namespace optim {

template <bool BF16>
__device__ __forceinline__ void ld4(const void* p, int64_t i, float* f) {
  if constexpr (BF16) {
    const u32x2_t v = *reinterpret_cast<const u32x2_t*>((const uint16_t*)p + i);
    f[0] = __uint_as_float(v[0] << 16);
    f[1] = __uint_as_float(v[0] & 0xffff0000u);
    f[2] = __uint_as_float(v[1] << 16);
    f[3] = __uint_as_float(v[1] & 0xffff0000u);
  } else {
    const f32x4_t v = *reinterpret_cast<const f32x4_t*>((const float*)p + i);
    f[0] = v[0]; f[1] = v[1]; f[2] = v[2]; f[3] = v[3];
  }
}

template <bool BF16>
__device__ __forceinline__ float ld1(const void* p, int64_t i) {
  if constexpr (BF16) return bf2f(((const uint16_t*)p)[i]);
  else return ((const float*)p)[i];
}

// mode 0: sum of squares, mode 1: max |x|
template <bool BF16, int MODE>
__global__ void __launch_bounds__(256) partial_kernel(const void* __restrict__ x, int64_t n, float* __restrict__ part) {
  __shared__ float red[16];
  float acc = 0.f;
  const int64_t n4 = n / 4;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (int64_t)gridDim.x * 256) {
    float f[4];
    ld4<BF16>(x, i * 4, f);
#pragma unroll
    for (int j = 0; j < 4; ++j) acc = MODE == 0 ? acc + f[j] * f[j] : fmaxf(acc, fabsf(f[j]));
  }
  if (blockIdx.x == 0)
    for (int64_t i = n4 * 4 + threadIdx.x; i < n; i += 256) {
      const float f = ld1<BF16>(x, i);
      acc = MODE == 0 ? acc + f * f : fmaxf(acc, fabsf(f));
    }
  const float t = MODE == 0 ? block_sum(acc, red) : block_max(acc, red);
  if (threadIdx.x == 0) part[blockIdx.x] = t;
}

template <int MODE>
__global__ void __launch_bounds__(256) final_kernel(const float* __restrict__ part, int np, float* __restrict__ out, int accumulate) {
  __shared__ float red[16];
  float acc = 0.f;
  for (int i = threadIdx.x; i < np; i += 256) acc = MODE == 0 ? acc + part[i] : fmaxf(acc, part[i]);
  const float t = MODE == 0 ? block_sum(acc, red) : block_max(acc, red);
  if (threadIdx.x == 0) out[0] = accumulate ? (MODE == 0 ? out[0] + t : fmaxf(out[0], t)) : t;
}

struct AdamHyper {
  float lr, beta1, beta2, eps, wd, bc1, bc2;  // bc = 1 - beta^t
  uint32_t sr_seed;                           // != 0: stochastic rounding of the bf16 copy-out
};

// Stochastic rounding fp32 -> bf16 (reference: NEURON_RT_STOCHASTIC_ROUNDING_EN for the bf16
// weights): add 16 uniform random bits below the bf16 mantissa, then truncate, so an update smaller
// than half a bf16 ulp still moves the weight with the right probability.  Counter-based hash of
// (seed, element index): no RNG state, identical on every replica of a parameter.
__device__ __forceinline__ uint32_t sr_hash(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}
__device__ __forceinline__ uint16_t f2bf_sr(float f, uint32_t seed, int64_t idx) {
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return f2bf(f);   // inf / nan: round as usual
  const uint32_t r = sr_hash((uint32_t)idx * 0x9E3779B1u ^ (uint32_t)(idx >> 32) ^ seed) & 0xffffu;
  return (uint16_t)((u + r) >> 16);
}

// hyper (nullable): device [lr, 1 - beta1^t, 1 - beta2^t] overriding h.lr / h.bc1 / h.bc2, so a
// captured optimizer step (hipGraph) replays with the current step's values.
//
// Seven streams of memory, 30 bytes a parameter (32-bit gradients, bf16 weights written), nothing else counts.  A workgroup
// takes U x 4 KB of each stream, all its loads in flight before the first is used, stores non-temporally, and ends.  491 M
// parameters with U = 4: two launches of 1.69 ms -> 1.44 (4.35 -> 5.1 TB/s; a large copy reaches 4.9); 2,048 workgroups that go
// on from block to block take 1.50.  Which U: see adamw_flat_launch.
template <bool GBF16, bool HAS_OUT, int U>
__global__ void __launch_bounds__(256) adamw_kernel(float* __restrict__ p, const void* __restrict__ g, float* __restrict__ m,
                                                    float* __restrict__ v, uint16_t* __restrict__ p16, int64_t n, AdamHyper h,
                                                    const float* __restrict__ gscale_ptr, float gscale_host,
                                                    const float* __restrict__ hyper) {
  if (hyper) {
    h.lr = hyper[0];
    h.bc1 = hyper[1];
    h.bc2 = hyper[2];
  }
  const float gs = gscale_ptr ? gscale_ptr[0] * gscale_host : gscale_host;
  const float step = h.lr / h.bc1;
  const float rbc2 = rsqrtf(h.bc2);
  const float decay = 1.f - h.lr * h.wd;
  auto update = [&](float gr, float& pv, float& mv, float& vv) {
    gr *= gs;
    mv = h.beta1 * mv + (1.f - h.beta1) * gr;
    vv = h.beta2 * vv + (1.f - h.beta2) * gr * gr;
    const float denom = sqrtf(vv) * rbc2 + h.eps;
    pv = pv * decay - step * mv / denom;
  };
  const int64_t n4 = n / 4;
  for (int64_t i0 = (int64_t)blockIdx.x * 256 * U; i0 < n4; i0 += (int64_t)gridDim.x * 256 * U) {
    float gf[U][4];
    f32x4_t pv[U], mv[U], vv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t e = 4 * min(i0 + 256 * u + threadIdx.x, n4 - 1);   // (past the end: read, not written)
      ld4<GBF16>(g, e, gf[u]);
      mv[u] = *reinterpret_cast<const f32x4_t*>(m + e);
      vv[u] = *reinterpret_cast<const f32x4_t*>(v + e);
      pv[u] = *reinterpret_cast<const f32x4_t*>(p + e);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (i0 + 256 * u + threadIdx.x >= n4) break;
      const int64_t e = 4 * (i0 + 256 * u + threadIdx.x);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float pj = pv[u][j], mj = mv[u][j], vj = vv[u][j];
        update(gf[u][j], pj, mj, vj);
        pv[u][j] = pj; mv[u][j] = mj; vv[u][j] = vj;
      }
      __builtin_nontemporal_store(pv[u], reinterpret_cast<f32x4_t*>(p + e));
      __builtin_nontemporal_store(mv[u], reinterpret_cast<f32x4_t*>(m + e));
      __builtin_nontemporal_store(vv[u], reinterpret_cast<f32x4_t*>(v + e));
      if constexpr (HAS_OUT) {
        u32x2_t o;
        if (h.sr_seed) {
          o[0] = (uint32_t)f2bf_sr(pv[u][0], h.sr_seed, e) | ((uint32_t)f2bf_sr(pv[u][1], h.sr_seed, e + 1) << 16);
          o[1] = (uint32_t)f2bf_sr(pv[u][2], h.sr_seed, e + 2) | ((uint32_t)f2bf_sr(pv[u][3], h.sr_seed, e + 3) << 16);
        } else {
          o[0] = pack2bf(pv[u][0], pv[u][1]);
          o[1] = pack2bf(pv[u][2], pv[u][3]);
        }
        __builtin_nontemporal_store(o, reinterpret_cast<u32x2_t*>(p16 + e));
      }
    }
  }
  if (blockIdx.x == 0)
    for (int64_t i = n4 * 4 + threadIdx.x; i < n; i += 256) {
      update(ld1<GBF16>(g, i), p[i], m[i], v[i]);
      if constexpr (HAS_OUT) p16[i] = h.sr_seed ? f2bf_sr(p[i], h.sr_seed, i) : f2bf(p[i]);
    }
}

// clip coefficient on device: coef = min(1, max_norm / (sqrt(sumsq) + 1e-6)) (or from max-norm)
__global__ void clip_coef_kernel(const float* __restrict__ stat, float* __restrict__ coef, float max_norm, int is_sumsq) {
  const float norm = is_sumsq ? sqrtf(stat[0]) : stat[0];
  const float c = max_norm / (norm + 1e-6f);
  coef[0] = c < 1.f ? c : 1.f;
  coef[1] = norm;
}

__global__ void __launch_bounds__(256) scale_kernel(float* __restrict__ x, int64_t n, const float* __restrict__ s) {
  const float sc = s[0];
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) x[i] *= sc;
}

}  // namespace optim

static inline int grid_for(int64_t n4) {
  int64_t g = (n4 + 255) / 256;
  return (int)(g < 2048 ? (g > 0 ? g : 1) : 2048);
}

// out[0] = sum(x^2) (mode 0) or max|x| (mode 1); part must hold >= 2048 floats.
int flat_reduce_launch(const void* x, int is_bf16, int64_t n, int mode, float* part, float* out, int accumulate, hipStream_t stream) {
  using namespace optim;
  const int grid = grid_for(n / 4);
#define PK(B, M) hipLaunchKernelGGL((partial_kernel<B, M>), dim3(grid), dim3(256), 0, stream, x, n, part)
  if (is_bf16) { if (mode == 0) PK(true, 0); else PK(true, 1); }
  else { if (mode == 0) PK(false, 0); else PK(false, 1); }
#undef PK
  if (mode == 0) hipLaunchKernelGGL(final_kernel<0>, dim3(1), dim3(256), 0, stream, part, grid, out, accumulate);
  else hipLaunchKernelGGL(final_kernel<1>, dim3(1), dim3(256), 0, stream, part, grid, out, accumulate);
  return (int)hipGetLastError();
}

int adamw_flat_launch(float* p, const void* g, int g_is_bf16, float* m, float* v, void* p16, int64_t n, float lr, float beta1,
                      float beta2, float eps, float wd, float bc1, float bc2, const float* gscale_ptr, float gscale_host,
                      uint32_t sr_seed, const float* hyper, hipStream_t stream) {
  using namespace optim;
  if (n == 0) return 0;
  AdamHyper h{lr, beta1, beta2, eps, wd, bc1, bc2, sr_seed};
  // Vectors a thread, by what fills the chip: us with 1 / 2 / 4 (32-bit gradients) 64 K parameters 2.9 / 3.2 / 4.1, 1 M 5.7 /
  // 5.5 / 5.9, 2 M 9.0 / 7.9 / 7.8, 4 M 19.9 / 19.8 / 20.9, 16 M 73.4 / 72.9 / 75.0, 64 M 382 / 369 / 373; 256 M 1,457 / 1,502 /
  // 1,493, the boxes' spread.  2,048 workgroups that go on with 1 each: 2.8, 5.7, 9.0, 19.8, 77.0, 423, 1,768.
  const int u = n < (1 << 21) ? 1 : n < (1 << 26) ? 2 : 4;
  // a workgroup per block; past 2^32 parameters they go on
  const int grid = (int)std::min<int64_t>(1 << 20, std::max<int64_t>(1, (n + 1024 * u - 1) / (1024 * u)));
#define AU(B, O, U) hipLaunchKernelGGL((adamw_kernel<B, O, U>), dim3(grid), dim3(256), 0, stream, p, g, m, v, (uint16_t*)p16, n, h, gscale_ptr, gscale_host, hyper)
#define AK(B, O) do { if (u == 1) AU(B, O, 1); else if (u == 2) AU(B, O, 2); else AU(B, O, 4); } while (0)
  if (g_is_bf16) { if (p16) AK(true, true); else AK(true, false); }
  else { if (p16) AK(false, true); else AK(false, false); }
#undef AK
#undef AU
  return (int)hipGetLastError();
}

int clip_coef_launch(const float* stat, float* coef, float max_norm, int is_sumsq, hipStream_t stream) {
  hipLaunchKernelGGL(optim::clip_coef_kernel, dim3(1), dim3(1), 0, stream, stat, coef, max_norm, is_sumsq);
  return (int)hipGetLastError();
}

int scale_flat_launch(float* x, int64_t n, const float* s, hipStream_t stream) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(optim::scale_kernel, dim3(grid_for(n)), dim3(256), 0, stream, x, n, s);
  return (int)hipGetLastError();
}

}  // namespace nxd
