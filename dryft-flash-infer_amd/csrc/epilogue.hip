// Split-K plane consumers and the small epilogues between projections.
//
// The bf16 roundings land where the reference puts them:
//   reduce_planes     bf16(sum_s P[s]) in slice order      engine/kernels/cuda_fp8.py:965-981
//   residual_planes   bf16(x + bf16(sum_s P[s]))           engine/kernels/cuda_small.py:43-55
//   rms_norm          bf16(bf16(x * rsqrt(mean x^2 + eps)) * w)  engine/kernels/reference.py:13-16
//   add_rms_norm      residual then rms_norm               engine/kernels/reference.py:19-28
//   swiglu            bf16(bf16(silu(bf16 g)) * bf16 u)    engine/kernels/swiglu.py:37-53
//   add_norm_quant    residual, rms_norm, INT8 quantize    engine/kernels/cuda_int8.py:17-44
//   add_norm_fp8      residual, rms_norm, per-token e4m3 quantize (the FP8 W8A8 activation
//                     of qlx_quantize_fp8_act, from the normed row held on chip)
#include <algorithm>

#include "common.h"
#include "../../include/qlinear.h"

namespace qlx {

typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;

__global__ void __launch_bounds__(256)
reduce_planes_kernel(const float* __restrict__ p, uint16_t* __restrict__ out, size_t width, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= width) return;
  float acc = 0.f;
  for (int s = 0; s < splits; ++s) acc += p[(size_t)s * width + i];
  out[i] = f2bf(acc);
}

__global__ void __launch_bounds__(256)
residual_planes_kernel(const uint16_t* __restrict__ x, const float* __restrict__ p,
                       uint16_t* __restrict__ out, size_t width, int splits) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= width) return;
  float acc = 0.f;
  for (int s = 0; s < splits; ++s) acc += p[(size_t)s * width + i];
  out[i] = f2bf(bf2f(x[i]) + round_bf(acc));
}

__device__ __forceinline__ uint4 ld16(const uint16_t* p) {
  const u32x4 v = *gmem(reinterpret_cast<const u32x4*>(p));
  return uint4{v[0], v[1], v[2], v[3]};
}

struct NormArgs {
  const uint16_t *x, *delta;
  const float* planes;
  int splits;
  const uint16_t* w;
  uint16_t *res, *y;
  int8_t* q;
  float* qs;
  uint8_t* q8;
  float* q8s;
  int rows, n;
  float eps;
};

// What becomes of the normed row besides y.
enum { kNormOnly, kNormInt8, kNormFp8 };

// 1/sqrt(mean + eps) of a row whose squares' partial sums lie in part[0 .. waves - 1]: summed in
// fp64 (each square of a bf16 value is exact there and so is the sum of a hidden row's worth, which
// makes it independent of the order), mean rounded to fp32, + eps and 1/sqrt in fp32, as torch's
// rsqrt(mean + eps).
__device__ __forceinline__ float norm_scale(const double* part, int waves, int n, float eps) {
  double total = part[0];
  for (int w = 1; w < waves; ++w) total += part[w];
  return 1.0f / sqrtf((float)(total / (double)n) + eps);
}

// One workgroup per row of n = 8 nc values, U chunks of 8 per thread, nc <= 1024 U: the row stays in
// registers between its two passes and every load (x, delta or the planes, w) is issued before any
// is used. delta: bf16 [rows][n] or (PLANES) fp32 planes [splits][rows][n], or neither (plain
// RMSNorm, no residual written). Bound by latency, so also by the instructions that a launch fetches
// from a cold cache: the first form, eight guarded chunks per thread of 256 with every option in
// each, was 43 KB of code and took 3.9 us per call in a graph (8 rows of 2560) where this one, 2 to
// 5 KB, takes 2.7.
template <int U, bool PLANES, int QUANT>
__global__ void __launch_bounds__(1024) norm_row_kernel(NormArgs a) {
  extern __shared__ float rbuf[];  // kNormInt8: the normed row
  __shared__ double part[16];
  __shared__ float pmax[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = blockDim.x >> 6;
  const int row = blockIdx.x, nc = a.n >> 3;
  const size_t base = (size_t)row * a.n;
  const bool add = PLANES || a.delta != nullptr;
  uint4 xv[U], dv[U], wv[U];
  u32x4 pv[U][2];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = tid + u * blockDim.x;
    xv[u] = dv[u] = wv[u] = uint4{0u, 0u, 0u, 0u};
    if (c < nc) {
      xv[u] = ld16(a.x + base + 8 * c);
      if (!PLANES && add) dv[u] = ld16(a.delta + base + 8 * c);
      wv[u] = ld16(a.w + 8 * c);
    }
  }
  float d[U][8];
  if constexpr (PLANES) {  // slice-order fp32 sums
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int i = 0; i < 8; ++i) d[u][i] = 0.f;
#pragma unroll 4
    for (int sl = 0; sl < a.splits; ++sl) {
      const float* pl = a.planes + (size_t)sl * a.rows * a.n + base;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = tid + u * blockDim.x;
        if (c < nc) {
          pv[u][0] = *gmem(reinterpret_cast<const u32x4*>(pl + 8 * c));
          pv[u][1] = *gmem(reinterpret_cast<const u32x4*>(pl + 8 * c + 4));
#pragma unroll
          for (int i = 0; i < 8; ++i) d[u][i] += __uint_as_float(pv[u][i >> 2][i & 3]);
        }
      }
    }
  }
  float r[U][8];
  double ss = 0.0;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = tid + u * blockDim.x;
    const uint32_t xs[4] = {xv[u].x, xv[u].y, xv[u].z, xv[u].w};
#pragma unroll
    for (int i = 0; i < 8; ++i) r[u][i] = bf2f((xs[i >> 1] >> (16 * (i & 1))) & 0xffffu);
    if (add && c < nc) {
      const uint32_t ds[4] = {dv[u].x, dv[u].y, dv[u].z, dv[u].w};
      // bf16 rounding by the hardware's pair conversion (the integer rounding's bits for every
      // value but a NaN, which then gets the integer rounding's form).
      uint32_t rp[4], nan = 0u;
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float d0 = bf2f(ds[i >> 1] & 0xffffu), d1 = bf2f(ds[i >> 1] >> 16);
        if constexpr (PLANES) {
          const uint32_t dp = bf16_pair_hw(d[u][i], d[u][i + 1]);
          nan |= bf16_nan_bits(dp);
          d0 = bf2f(dp & 0xffffu);
          d1 = bf2f(dp >> 16);
        }
        rp[i >> 1] = bf16_pair_hw(r[u][i] + d0, r[u][i + 1] + d1);
        nan |= bf16_nan_bits(rp[i >> 1]);
      }
      if (nan != 0u) {
#pragma unroll
        for (int i = 0; i < 4; ++i) rp[i] = bf16_canonical_nan(rp[i]);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) r[u][i] = bf2f((rp[i >> 1] >> (16 * (i & 1))) & 0xffffu);
      if (a.res) *gmem(reinterpret_cast<u32x4*>(a.res + base + 8 * c)) = u32x4{rp[0], rp[1], rp[2], rp[3]};
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) ss += (double)r[u][i] * (double)r[u][i];
  }
  ss = wave_sum_last(ss);
  if (lane == 63) part[wave] = ss;
  __syncthreads();
  const float scale = norm_scale(part, waves, a.n, a.eps);
  uint32_t vp[U][4];
  float mx = 0.f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int c = tid + u * blockDim.x;
    const uint32_t ws[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
    uint32_t nan = 0u;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {  // as above
      const uint32_t t = bf16_pair_hw(r[u][i] * scale, r[u][i + 1] * scale);
      vp[u][i >> 1] = bf16_pair_hw(bf2f(t & 0xffffu) * bf2f(ws[i >> 1] & 0xffffu),
                                   bf2f(t >> 16) * bf2f(ws[i >> 1] >> 16));
      nan |= bf16_nan_bits(t) | bf16_nan_bits(vp[u][i >> 1]);
    }
    if (nan != 0u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) vp[u][i] = bf16_canonical_nan(vp[u][i]);
    }
    if (c < nc) {
      if (a.y) *gmem(reinterpret_cast<u32x4*>(a.y + base + 8 * c)) = u32x4{vp[u][0], vp[u][1], vp[u][2], vp[u][3]};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float v = bf2f((vp[u][i >> 1] >> (16 * (i & 1))) & 0xffffu);
        if constexpr (QUANT == kNormInt8) rbuf[8 * c + i] = v;
        if constexpr (QUANT == kNormFp8) mx = fmaxf(mx, fabsf(v));
      }
    }
  }
  if constexpr (QUANT == kNormFp8) {
    // per-token e4m3 quantize of the normed row: scale = max(amax / 448, 1e-12), codes e4m3(x / scale)
    mx = wave_max_last(mx);
    if (lane == 63) pmax[wave] = mx;
    __syncthreads();
    mx = pmax[0];
    for (int w = 1; w < waves; ++w) mx = fmaxf(mx, pmax[w]);
    const float sc = fmaxf(mx / 448.f, 1e-12f), yr = 1.f / sc;
    if (tid == 0) a.q8s[row] = sc;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = tid + u * blockDim.x;
      if (c < nc) {
        const uint2 e = e4m3_chunk(uint4{vp[u][0], vp[u][1], vp[u][2], vp[u][3]}, sc, yr);
        *gmem(reinterpret_cast<u32x2*>(a.q8 + base + 8 * c)) = u32x2{e.x, e.y};
      }
    }
  }
  if constexpr (QUANT == kNormInt8) {
    // INT8 activation quantize per 64-group, fragment order (cuda_int8.py:30-44).
    __syncthreads();
    const int groups = a.n / 64;
    for (int g = wave; g < groups; g += waves) {
      const int nat = (lane >> 4) * 4 + ((lane & 15) >> 2) * 16 + (lane & 3);
      const float v = rbuf[g * 64 + nat];
      const float amax = wave_max(fabsf(v));
      const float s = fmaxf(amax / 127.f, 1e-20f);
      a.q[base + g * 64 + lane] = (int8_t)(int)rintf(v / s);
      if (lane == 0) a.qs[(size_t)row * groups + g] = s;
    }
  }
}

// Rows of any length, a value at a time (n not a multiple of 8; no quantized output).
__global__ void __launch_bounds__(256) norm_row_scalar_kernel(NormArgs a) {
  extern __shared__ float rbuf[];  // the row's residual, fp32
  __shared__ double part[4];
  const int row = blockIdx.x;
  const size_t base = (size_t)row * a.n;
  double ss = 0.0;
  for (int c = threadIdx.x; c < a.n; c += 256) {
    float r = bf2f(a.x[base + c]);
    if (a.delta != nullptr || a.planes != nullptr) {
      float d;
      if (a.planes) {
        d = 0.f;
        for (int sl = 0; sl < a.splits; ++sl) d += a.planes[(size_t)sl * a.rows * a.n + base + c];
        d = round_bf(d);
      } else {
        d = bf2f(a.delta[base + c]);
      }
      r = round_bf(r + d);
      if (a.res) a.res[base + c] = f2bf(r);
    }
    rbuf[c] = r;
    ss += (double)r * (double)r;
  }
  ss = wave_sum_last(ss);
  if ((threadIdx.x & 63) == 63) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float scale = norm_scale(part, 4, a.n, a.eps);
  for (int c = threadIdx.x; c < a.n; c += 256)
    if (a.y) a.y[base + c] = f2bf(round_bf(rbuf[c] * scale) * bf2f(a.w[c]));
}

template <int U, int QUANT>
void launch_norm_row(const NormArgs& a, hipStream_t st) {
  const int nc = a.n >> 3, own = ((nc + U - 1) / U + 63) / 64 * 64;
  // INT8: the waves also share out the row's 64-value groups, one after the other; 8 rows of 512 in us per
  // call: 4.7 with the one wave that its chunks fill, 3.2 with 4, 3.1 with 8; of 1024 5.1, 3.9, 3.5
  const int threads = QUANT == kNormInt8 ? std::max(own, 64 * std::min(a.n / 64, 8)) : own;
  const size_t lds = QUANT == kNormInt8 ? a.n * sizeof(float) : 0;
  if (a.planes) norm_row_kernel<U, true, QUANT><<<a.rows, threads, lds, st>>>(a);
  else norm_row_kernel<U, false, QUANT><<<a.rows, threads, lds, st>>>(a);
}

// Threads for every chunk of a row up to 8192 values, two chunks per thread above (n <= 16384).
template <int QUANT>
void launch_norm(const NormArgs& a, hipStream_t st) {
  if (a.n % 8) norm_row_scalar_kernel<<<a.rows, 256, a.n * sizeof(float), st>>>(a);
  else if (a.n <= 8192) launch_norm_row<1, QUANT>(a, st);
  else launch_norm_row<2, QUANT>(a, st);
}

// gate_up: bf16 [rows][2I] or (planes != null) fp32 planes [splits][rows][2I].
__global__ void __launch_bounds__(256)
swiglu_kernel(const uint16_t* __restrict__ gu, const float* __restrict__ planes, int splits,
              uint16_t* __restrict__ out, int rows, int inter) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int row = blockIdx.y;
  if (c >= inter) return;
  const size_t base = (size_t)row * 2 * inter + c;
  float g, u;
  if (planes) {
    g = 0.f;
    u = 0.f;
    const size_t plane = (size_t)rows * 2 * inter;
    for (int s = 0; s < splits; ++s) {
      g += planes[s * plane + base];
      u += planes[s * plane + base + inter];
    }
    g = round_bf(g);
    u = round_bf(u);
  } else {
    g = bf2f(gu[base]);
    u = bf2f(gu[base + inter]);
  }
  const float silu = round_bf(g / (1.f + expf(-g)));
  out[(size_t)row * inter + c] = f2bf(silu * u);
}

static inline unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

}  // namespace qlx

using namespace qlx;

extern "C" {

int qlx_reduce_planes(const float* planes, void* out, long long width, int splits, void* stream) {
  QLX_REQUIRE(width > 0 && splits >= 1, "bad reduce shape");
  reduce_planes_kernel<<<blocks_for(width), 256, 0, (hipStream_t)stream>>>(planes, (uint16_t*)out,
                                                                          (size_t)width, splits);
  QLX_LAUNCH_CHECK("reduce_planes");
}

int qlx_residual_planes(const void* x, const float* planes, void* out, long long width, int splits,
                        void* stream) {
  QLX_REQUIRE(width > 0 && splits >= 1, "bad residual shape");
  residual_planes_kernel<<<blocks_for(width), 256, 0, (hipStream_t)stream>>>(
      (const uint16_t*)x, planes, (uint16_t*)out, (size_t)width, splits);
  QLX_LAUNCH_CHECK("residual_planes");
}

int qlx_add_rms_norm(const void* x, const void* delta, const float* planes, int splits, const void* w,
                     void* res, void* y, int rows, int n, float eps, void* stream) {
  QLX_REQUIRE(rows > 0 && n > 0 && n <= 16384, "rows=%d n=%d: rows must be > 0 and n in 1..16384", rows, n);
  QLX_REQUIRE(planes == nullptr || splits >= 1, "planes need splits >= 1");
  launch_norm<kNormOnly>(NormArgs{(const uint16_t*)x, (const uint16_t*)delta, planes, splits, (const uint16_t*)w, (uint16_t*)res,
                        (uint16_t*)y, nullptr, nullptr, nullptr, nullptr, rows, n, eps},
                  (hipStream_t)stream);
  QLX_LAUNCH_CHECK("add_rms_norm");
}

int qlx_add_norm_quant_int8(const void* x, const void* delta, const float* planes, int splits,
                            const void* w, void* res, void* q, float* q_scale, int rows, int n, float eps,
                            void* stream) {
  QLX_REQUIRE(rows > 0 && n > 0 && n <= 16384 && n % 64 == 0, "n=%d must be a multiple of 64 up to 16384", n);
  QLX_REQUIRE(planes == nullptr || splits >= 1, "planes need splits >= 1");
  launch_norm<kNormInt8>(NormArgs{(const uint16_t*)x, (const uint16_t*)delta, planes, splits, (const uint16_t*)w, (uint16_t*)res,
                        nullptr, (int8_t*)q, q_scale, nullptr, nullptr, rows, n, eps},
                  (hipStream_t)stream);
  QLX_LAUNCH_CHECK("add_norm_quant_int8");
}

int qlx_add_norm_quant_fp8(const void* x, const void* delta, const float* planes, int splits, const void* w,
                           void* res, void* y, void* code, float* scale, int rows, int n, float eps, void* stream) {
  QLX_REQUIRE(rows > 0 && n > 0 && n <= 16384 && n % 8 == 0, "n=%d must be a multiple of 8 up to 16384", n);
  QLX_REQUIRE(planes == nullptr || splits >= 1, "planes need splits >= 1");
  QLX_REQUIRE(code != nullptr && scale != nullptr, "codes and scales are required");
  launch_norm<kNormFp8>(NormArgs{(const uint16_t*)x, (const uint16_t*)delta, planes, splits, (const uint16_t*)w, (uint16_t*)res,
                        (uint16_t*)y, nullptr, nullptr, (uint8_t*)code, scale, rows, n, eps},
                  (hipStream_t)stream);
  QLX_LAUNCH_CHECK("add_norm_quant_fp8");
}

int qlx_swiglu(const void* gate_up, const float* planes, int splits, void* out, int rows, int inter,
               void* stream) {
  QLX_REQUIRE(rows > 0 && inter > 0, "bad swiglu shape");
  QLX_REQUIRE(gate_up != nullptr || (planes != nullptr && splits >= 1), "swiglu needs gate_up or planes");
  dim3 grid((inter + 255) / 256, rows);
  swiglu_kernel<<<grid, 256, 0, (hipStream_t)stream>>>((const uint16_t*)gate_up, planes, splits,
                                                      (uint16_t*)out, rows, inter);
  QLX_LAUNCH_CHECK("swiglu");
}

}  // extern "C"
