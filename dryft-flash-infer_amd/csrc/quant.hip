// Quantize, pack and relayout kernels (load-time work) and the library's error state.
//
// Every kernel here is bit-exact with the CPU statement of the reference:
//   quantize_weight   engine/kernels/cuda_fp8.py:1127-1151 (plus the north-star
//                     generalisations: bf16 scales, signed int8, int4 k32 words)
//   dequantize        engine/kernels/cuda_fp8.py:1154-1161
//   prepare_ref       engine/kernels/cuda_fp8.py:1117-1124, 1164-1205
//   row_major_ref     engine/kernels/cuda_fp8.py:1207-1214
//   quantize_fp8_*    engine/kernels/fp8.py:20-28 (weights; per-token activations)
//   int8_prepare      engine/kernels/cuda_int8.py:100-108
//   quantize_act_int8 engine/kernels/cuda_int8.py:58-77
#include <stdarg.h>
#include <stdio.h>

#include <type_traits>

#include "common.h"
#include "../../include/qlinear.h"

namespace qlx {

static thread_local char g_error[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

int hip_status(hipError_t e, const char* what) {
  if (e == hipSuccess) return QLX_OK;
  set_error("%s failed: %s (%d)", what, hipGetErrorString(e), (int)e);
  return QLX_EHIP;
}

// ---- weight quantize -----------------------------------------------------------------------

// Largest magnitude of 8 bf16 values (pairs in v), ignoring NaNs.
__device__ __forceinline__ float octet_amax(uint4 v, float amax) {
  const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    amax = fmaxf(amax, fabsf(bf2f(d[j] & 0xffffu)));
    amax = fmaxf(amax, fabsf(bf2f(d[j] >> 16)));
  }
  return amax;
}

// Integer codes of a group. storage: 0 = offset bytes (q + offset, uint8, one per byte), 1 = signed
// int8, 2 = int4 codes (q + 8) packed eight per int32 along K (nibble i of word j is k = 8j + i).
struct IntQuant {
  int bits, scale_fp16, nudge, storage;
  struct Group {
    float sval, y, limit, offset;  // the stored scale's value, its reciprocal
    uint16_t sbits;
    bool fast;
  };
  __device__ __forceinline__ Group group(float amax) const {
    Group g;
    g.limit = bits == 8 ? 127.f : 7.f;
    g.offset = bits == 8 ? 128.f : 8.f;
    float s = fmaxf(amax / g.limit, 1e-12f);
    if (nudge) s = s * (1.0f + 0.0009765625f);
    if (scale_fp16) {
      g.sbits = f2h(s);
      g.sval = h2f(g.sbits);
    } else {
      g.sbits = f2bf(s);
      g.sval = bf2f(g.sbits);
    }
    g.y = 1.f / g.sval;
    g.fast = g.sval >= 1e-30f && g.sval <= 3.40282347e38f;
    return g;
  }
  // 8 values at element `at` of the flat weight. The quotient of the fast path is the IEEE one
  // (quotient_by_reciprocal) wherever it can reach a code other than 0: a residual too small to
  // be exact needs |x / s| far below 1/2. A zero or infinite scale and a chunk with a NaN divide.
  __device__ __forceinline__ void store(const Group& g, uint4 v, void* data, size_t at) const {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
    uint32_t codes[8];
    if (g.fast && !(bf16_nan_bits(d[0]) | bf16_nan_bits(d[1]) | bf16_nan_bits(d[2]) | bf16_nan_bits(d[3]))) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = bf2f(e & 1 ? d[e >> 1] >> 16 : d[e >> 1] & 0xffffu);
        const float q = __builtin_amdgcn_fmed3f(rintf(quotient_by_reciprocal(x, g.sval, g.y)), -g.limit, g.limit);
        codes[e] = storage == 1 ? (uint32_t)(int32_t)q & 0xffu : (uint32_t)(q + g.offset);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = bf2f(e & 1 ? d[e >> 1] >> 16 : d[e >> 1] & 0xffffu);
        float q = clamp_keep_nan(rintf(x / g.sval), g.limit);
        if (storage == 1) {
          codes[e] = q != q ? 0u : (uint32_t)(int32_t)q & 0xffu;
        } else {
          const float b = q + g.offset;
          codes[e] = b != b ? 0u : (uint32_t)b;
        }
      }
    }
    if (storage == 2) {
      uint32_t word = 0;
#pragma unroll
      for (int e = 0; e < 8; ++e) word |= (codes[e] & 0xfu) << (4 * e);
      reinterpret_cast<uint32_t*>(data)[at >> 3] = word;
    } else {
      uint2 out;
      out.x = codes[0] | (codes[1] << 8) | (codes[2] << 16) | (codes[3] << 24);
      out.y = codes[4] | (codes[5] << 8) | (codes[6] << 16) | (codes[7] << 24);
      *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(data) + at) = out;
    }
  }
};

// e4m3 codes of a group (fp8.py:20-28): s = max(amax/448, 1e-12); code = e4m3(clamp(w/s)); scale
// out bf16(s).
struct Fp8Quant {
  struct Group {
    float sval, y;
    uint16_t sbits;
  };
  __device__ __forceinline__ Group group(float amax) const {
    const float s = fmaxf(amax / 448.f, 1e-12f);
    return Group{s, 1.f / s, f2bf(s)};
  }
  __device__ __forceinline__ void store(const Group& g, uint4 v, void* data, size_t at) const {
    *reinterpret_cast<uint2*>(reinterpret_cast<uint8_t*>(data) + at) = e4m3_chunk(v, g.sval, g.y);
  }
};

// A row's groups follow each other, so group `gid` of the weight is the flat values
// gid * group .. + group, and its scale the flat scale gid.
//
// Memory-bound (2 bytes in, 1/2 or 1 byte out per value) once every lane holds values and a value
// costs about ten instructions: one wave per 128-value group left 48 of 64 lanes idle and divided
// (IEEE division, ~30 instructions a value, and the values read twice): 151936 x 2560 to int4 in
// 1362 us, 0.7 TB/s. Groups of up to 512 values: L lanes (8 values each) per group, 4 groups per
// thread loaded before any is reduced: the same weight in 221 us, 4.4 TB/s (a large copy: 4.9 TB/s).
// Groups of 513 to 2048 values: 2 or 4 chunks a lane of a whole wave. (A block per group leaves half of its
// lanes without values: 40960 x 2048 to e4m3 in groups of 1024 68.8 us, a wave that reads the group twice
// 47.1, this 40.7; 40960 x 2080 in groups of 520 129.5, 79.1 and 57.1.)
template <class Q, int L, int CHUNKS = 1>
__global__ void __launch_bounds__(256)
quantize_segments_kernel(Q quant, const uint16_t* __restrict__ w, void* __restrict__ data,
                         uint16_t* __restrict__ scale, long long segs, int group) {
  const int lane = threadIdx.x % L, octets = group >> 3;
  constexpr int PER = 256 / L, SEGS = 4 / CHUNKS;
  const long long seg0 = (long long)blockIdx.x * (PER * SEGS) + threadIdx.x / L;
  uint4 v[SEGS][CHUNKS];
#pragma unroll
  for (int u = 0; u < SEGS; ++u) {
    const long long seg = seg0 + u * PER;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int o = lane + L * c;
      v[u][c] = uint4{0u, 0u, 0u, 0u};
      if (seg < segs && o < octets) v[u][c] = *reinterpret_cast<const uint4*>(w + (size_t)seg * group + 8 * o);
    }
  }
#pragma unroll
  for (int u = 0; u < SEGS; ++u) {
    const long long seg = seg0 + u * PER;
    float amax = 0.f;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) amax = octet_amax(v[u][c], amax);
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 64));
    if (seg >= segs) continue;
    const typename Q::Group g = quant.group(amax);
    if (lane == 0) scale[seg] = g.sbits;
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const int o = lane + L * c;
      if (o < octets) quant.store(g, v[u][c], data, (size_t)seg * group + 8 * o);
    }
  }
}

// Groups of 2049 to 256 * 8 * R values (a row per scale): a 256-thread block per group, which keeps
// its values in registers between the maximum and the codes.
template <class Q, int R>
__global__ void __launch_bounds__(256)
quantize_rows_kernel(Q quant, const uint16_t* __restrict__ w, void* __restrict__ data,
                     uint16_t* __restrict__ scale, int group) {
  __shared__ float part[4];
  const int octets = group >> 3;
  const size_t base = (size_t)blockIdx.x * group;
  uint4 v[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int o = threadIdx.x + 256 * u;
    v[u] = uint4{0u, 0u, 0u, 0u};
    if (o < octets) v[u] = *reinterpret_cast<const uint4*>(w + base + 8 * o);
  }
  float amax = 0.f;
#pragma unroll
  for (int u = 0; u < R; ++u) amax = octet_amax(v[u], amax);
  amax = wave_max(amax);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
  const typename Q::Group g = quant.group(amax);
  if (threadIdx.x == 0) scale[blockIdx.x] = g.sbits;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int o = threadIdx.x + 256 * u;
    if (o < octets) quant.store(g, v[u], data, base + 8 * o);
  }
}

// Longer groups: one wave per group, which reads the values twice.
template <class Q>
__global__ void __launch_bounds__(256)
quantize_wave_kernel(Q quant, const uint16_t* __restrict__ w, void* __restrict__ data,
                     uint16_t* __restrict__ scale, long long segs, int group) {
  const int lane = threadIdx.x & 63, octets = group >> 3;
  const long long seg = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (seg >= segs) return;
  const uint16_t* src = w + (size_t)seg * group;
  float amax = 0.f;
  for (int o = lane; o < octets; o += 64) amax = octet_amax(*reinterpret_cast<const uint4*>(src + 8 * o), amax);
  const typename Q::Group g = quant.group(wave_max(amax));
  if (lane == 0) scale[seg] = g.sbits;
  for (int o = lane; o < octets; o += 64)
    quant.store(g, *reinterpret_cast<const uint4*>(src + 8 * o), data, (size_t)seg * group + 8 * o);
}

template <class Q>
void launch_quantize(const Q& quant, const uint16_t* w, void* data, uint16_t* scale, int rows, int k, int group,
                     hipStream_t st) {
  const long long segs = (long long)rows * (k / group);
  const int octets = group >> 3;
  auto segments = [&](auto lc, auto cc) {
    constexpr int L = decltype(lc)::value, C = decltype(cc)::value, per = 256 / L * (4 / C);
    quantize_segments_kernel<Q, L, C><<<(unsigned)((segs + per - 1) / per), 256, 0, st>>>(quant, w, data, scale, segs, group);
  };
  constexpr std::integral_constant<int, 1> one{};
  if (octets <= 8) segments(std::integral_constant<int, 8>{}, one);
  else if (octets <= 16) segments(std::integral_constant<int, 16>{}, one);
  else if (octets <= 32) segments(std::integral_constant<int, 32>{}, one);
  else if (octets <= 64) segments(std::integral_constant<int, 64>{}, one);
  else if (octets <= 128) segments(std::integral_constant<int, 64>{}, std::integral_constant<int, 2>{});
  else if (octets <= 256) segments(std::integral_constant<int, 64>{}, std::integral_constant<int, 4>{});
  else if (octets <= 512) quantize_rows_kernel<Q, 2><<<(unsigned)segs, 256, 0, st>>>(quant, w, data, scale, group);
  else if (octets <= 2048) quantize_rows_kernel<Q, 8><<<(unsigned)segs, 256, 0, st>>>(quant, w, data, scale, group);
  else quantize_wave_kernel<Q><<<(unsigned)((segs + 3) / 4), 256, 0, st>>>(quant, w, data, scale, segs, group);
}

// ---- dequantize: bf16((q - offset) * float(scale)) -------------------------------------

__global__ void __launch_bounds__(256)
dequantize_kernel(const void* __restrict__ data, const uint16_t* __restrict__ scale,
                  uint16_t* __restrict__ out, int rows, int k, int groups, int bits,
                  int scale_fp16, int storage) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)rows * k) return;
  const int row = (int)(i / k), col = (int)(i % k);
  const int g = col / (k / groups);
  const uint16_t sb = scale[(size_t)row * groups + g];
  const float s = scale_fp16 ? h2f(sb) : bf2f(sb);
  float q;
  if (storage == 1) {
    q = (float)reinterpret_cast<const int8_t*>(data)[i];
  } else if (storage == 2) {
    const uint32_t word = reinterpret_cast<const uint32_t*>(data)[i >> 3];
    q = (float)((word >> (4 * (i & 7))) & 0xfu) - 8.f;
  } else {
    q = (float)reinterpret_cast<const uint8_t*>(data)[i] - (bits == 8 ? 128.f : 8.f);
  }
  out[i] = f2bf(q * s);
}

// ---- reference layouts (cuda_fp8.Prepared) --------------------------------------------------

// The prepared weight from the [rows, K] quantize output: a thread takes one 64-value block of one
// row (4 bits: the two blocks of a 128-value step) and writes the 64 bytes it becomes, which every
// layout keeps together: position 16t + 4s + i of a permuted block holds the natural value
// 16s + 2t + (0, 1, 8, 9)[i] (cuda_fp8.py:1117-1124), so dword s of the 16 bytes of t is the value
// pairs 16s + 2t and 16s + 2t + 8. (It gathered single bytes, each through six 64-bit divisions.)
// The bytes may start anywhere (a slice of a larger buffer): accesses are declared unaligned.
struct __attribute__((packed, aligned(1))) Bytes16 {
  uint32_t x, y, z, w;
};
__global__ void __launch_bounds__(256)
prepare_ref_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int rows,
                   int k, int bits, int tiled) {
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  const int per_row = k >> (bits == 4 ? 7 : 6);
  if (o >= (size_t)rows * per_row) return;
  const int r = (int)(o / per_row), blk = (int)(o - (size_t)r * per_row);
  auto block = [&](int b64, uint32_t (&out)[16]) {  // 64 values, permuted
    const Bytes16* p = reinterpret_cast<const Bytes16*>(src + (size_t)r * k + (size_t)b64 * 64);
    uint32_t d[16];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const Bytes16 v = p[i];
      d[4 * i] = v.x, d[4 * i + 1] = v.y, d[4 * i + 2] = v.z, d[4 * i + 3] = v.w;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int s = 0; s < 4; ++s)
        out[4 * t + s] = __builtin_amdgcn_perm(d[4 * s + 2 + (t >> 1)], d[4 * s + (t >> 1)],
                                               t & 1 ? 0x07060302u : 0x05040100u);
  };
  uint32_t out[16];
  size_t at;
  const size_t tile = r >> 4;
  const int half = (r >> 3) & 1, gg = r & 7;
  if (bits == 8) {
    block(blk, out);
    // tiled: [tile][K/128][half][j][g][t][16 B]
    at = tiled ? ((((tile * (k >> 7) + (blk >> 1)) * 2 + half) * 2 + (blk & 1)) * 8 + gg) * 64
               : (size_t)r * k + (size_t)blk * 64;
  } else {
    // [tile][K/128][half][g][t][16 B]; block 0 in the low nibble, block 1 in the high one
    uint32_t hi[16];
    block(2 * blk, out);
    block(2 * blk + 1, hi);
#pragma unroll
    for (int i = 0; i < 16; ++i) out[i] = (out[i] & 0x0f0f0f0fu) | ((hi[i] & 0x0f0f0f0fu) << 4);
    at = (((tile * (k >> 7) + blk) * 2 + half) * 8 + gg) * 64;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    reinterpret_cast<Bytes16*>(dst + at)[i] = Bytes16{out[4 * i], out[4 * i + 1], out[4 * i + 2], out[4 * i + 3]};
}

// Tiled 8-bit prepared weight -> fragment-permuted row-major bytes.
__global__ void __launch_bounds__(256)
row_major_ref_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst, int rows,
                     int k) {
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= (size_t)rows * k) return;
  const int r = (int)(o / k), pos = (int)(o % k);
  const int tile = r / 16, half = (r / 8) % 2, gg = r % 8;
  const int grp = pos / 128, j = (pos / 64) % 2, t = (pos / 16) % 4, byte = pos % 16;
  const size_t idx = ((((((size_t)tile * (k / 128) + grp) * 2 + half) * 2 + j) * 8 + gg) * 4 + t) * 16 + byte;
  dst[o] = src[idx];
}

// ---- FP8 e4m3 (fp8.py:20-28) ------------------------------------------------------------------

// Per-token activation quantize: a block per row, U chunks of 8 values per thread, held in registers
// between the maximum and the codes (U = 0: a loop that reads the row twice, for rows of over 16384).
template <int U>
__global__ void __launch_bounds__(1024)
quantize_fp8_act_kernel(const uint16_t* __restrict__ x, uint8_t* __restrict__ code,
                        float* __restrict__ scale, int k) {
  __shared__ float part[16];
  const int row = blockIdx.x, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const size_t base = (size_t)row * k;
  const int octets = k >> 3;
  uint4 v[U ? U : 1];
  float amax = 0.f;
  if constexpr (U > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int o = threadIdx.x + u * blockDim.x;
      v[u] = uint4{0u, 0u, 0u, 0u};
      if (o < octets) v[u] = *reinterpret_cast<const uint4*>(x + base + 8 * o);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) amax = octet_amax(v[u], amax);
  } else {
    for (int o = threadIdx.x; o < octets; o += blockDim.x)
      amax = octet_amax(*reinterpret_cast<const uint4*>(x + base + 8 * o), amax);
  }
  amax = wave_max_last(amax);
  if (lane == 63) part[threadIdx.x >> 6] = amax;
  __syncthreads();
  amax = part[0];
  for (int w = 1; w < waves; ++w) amax = fmaxf(amax, part[w]);
  const float s = fmaxf(amax / 448.f, 1e-12f), y = 1.f / s;
  if (threadIdx.x == 0) scale[row] = s;
  if constexpr (U > 0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int o = threadIdx.x + u * blockDim.x;
      if (o < octets) *reinterpret_cast<uint2*>(code + base + 8 * o) = e4m3_chunk(v[u], s, y);
    }
  } else {
    for (int o = threadIdx.x; o < octets; o += blockDim.x)
      *reinterpret_cast<uint2*>(code + base + 8 * o) = e4m3_chunk(*reinterpret_cast<const uint4*>(x + base + 8 * o), s, y);
  }
}

// Every input the FP8 quantizers can see, through e4m3_chunk and through e4m3_of_quotient: a
// finite or infinite bf16 maximum `amax` (block y), its scale max(amax / 448, 1e-12), and each
// bf16 x with |x| <= amax, plus every NaN x. counts[0] = codes that differ, counts[2 + i] the
// first 64 of them as (amax bits << 48 | x bits << 32 | fast code << 8 | reference code).
__global__ void __launch_bounds__(256) fp8_selfcheck_kernel(unsigned long long* counts) {
  const uint32_t ab = blockIdx.y;  // 0 .. 0x7f80 (+inf)
  const float amax = bf2f(ab);
  const float s = fmaxf(amax / 448.f, 1e-12f), y = 1.f / s;
  unsigned long long bad = 0;
  // 8 consecutive x bit patterns per thread: one chunk
  for (uint32_t x0 = (blockIdx.x * 256 + threadIdx.x) * 8; x0 < 0x10000u; x0 += gridDim.x * 256 * 8) {
    uint32_t pk[4];
    bool live[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t xb = x0 + e, mag = xb & 0x7fffu;
      live[e] = mag <= ab || mag > 0x7f80u;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // values outside the domain are replaced by 0 so that the chunk stays a possible input
      const uint32_t lo = live[2 * i] ? x0 + 2 * i : 0u, hi = live[2 * i + 1] ? x0 + 2 * i + 1 : 0u;
      pk[i] = lo | (hi << 16);
    }
    const uint2 f = e4m3_chunk(uint4{pk[0], pk[1], pk[2], pk[3]}, s, y);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t bits = e & 1 ? pk[e >> 1] >> 16 : pk[e >> 1] & 0xffffu;
      const uint32_t r = e4m3_of_quotient(bf2f(bits), s);
      const uint32_t fc = ((e < 4 ? f.x : f.y) >> (8 * (e & 3))) & 0xffu;
      if (fc != r) {
        ++bad;
        const unsigned long long i = atomicAdd(&counts[1], 1ull);
        if (i < 64) counts[2 + i] = ((unsigned long long)ab << 48) | ((unsigned long long)bits << 32) | (fc << 8) | r;
      }
    }
  }
  if (bad) atomicAdd(&counts[0], bad);
}

// ---- INT8 W8A8 (cuda_int8.py) ---------------------------------------------------------------

// Natural index held at INT8 fragment position p (cuda_int8.py:64).
__device__ __forceinline__ int i8_natural(int p) {
  return (p >> 4) * 4 + ((p & 15) >> 2) * 16 + (p & 3);
}

// out[r][p] = row_major_ref[r][position holding natural i8_natural(p)] ^ 128.
__global__ void __launch_bounds__(256)
int8_prepare_kernel(const uint8_t* __restrict__ src, int8_t* __restrict__ dst, int rows, int k) {
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (o >= (size_t)rows * k) return;
  const int r = (int)(o / k), pos = (int)(o % k);
  const int n = i8_natural(pos & 63);
  const int old = ((n % 8) / 2) * 16 + (n / 16) * 4 + ((n % 16) / 8) * 2 + n % 2;
  dst[o] = (int8_t)(src[(size_t)r * k + (pos & ~63) + old] ^ 128u);
}

// One wave per (row, 64-group): s = max(amax/127, 1e-20); q = rint(x/s) at fragment position.
// With q2 != null the residual x - q*s is quantized the same way (cuda_int8.py:69-74).
__global__ void __launch_bounds__(256)
quantize_act_int8_kernel(const uint16_t* __restrict__ x, int8_t* __restrict__ q,
                         float* __restrict__ scale, int8_t* __restrict__ q2, float* __restrict__ scale2,
                         int m, int k) {
  const int lane = threadIdx.x & 63;
  const long long gid = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int groups = k / 64;
  if (gid >= (long long)m * groups) return;
  const int row = (int)(gid / groups), g = (int)(gid % groups);
  const float v = bf2f(x[(size_t)row * k + g * 64 + i8_natural(lane)]);
  const float amax = wave_max(fabsf(v));
  const float s = fmaxf(amax / 127.f, 1e-20f);
  const float qv = rintf(v / s);
  q[(size_t)row * k + g * 64 + lane] = (int8_t)(int)qv;
  if (lane == 0) scale[(size_t)row * groups + g] = s;
  if (q2) {
    const float r = v - qv * s;
    const float ramax = wave_max(fabsf(r));
    const float sr = fmaxf(ramax / 127.f, 1e-20f);
    q2[(size_t)row * k + g * 64 + lane] = (int8_t)(int)rintf(r / sr);
    if (lane == 0) scale2[(size_t)row * groups + g] = sr;
  }
}

static inline unsigned blocks_for(size_t n, unsigned per) { return (unsigned)((n + per - 1) / per); }

}  // namespace qlx

using namespace qlx;

extern "C" {

const char* qlx_last_error(void) { return g_error; }

int qlx_abi_version(void) { return QLX_ABI_VERSION; }

int qlx_quantize_weight(const void* w, void* data, void* scale, int rows, int k, int group,
                        int bits, int scale_kind, int nudge, int storage, void* stream) {
  QLX_REQUIRE(bits == 8 || bits == 4, "weights are 8 or 4 bits, got %d", bits);
  QLX_REQUIRE(rows > 0 && k > 0 && group > 0 && k % group == 0, "%d is not a multiple of %d", k, group);
  QLX_REQUIRE(group % 8 == 0, "group %d must be a multiple of 8", group);
  QLX_REQUIRE(storage >= 0 && storage <= 2, "bad storage %d", storage);
  QLX_REQUIRE(storage != 2 || bits == 4, "int4 k32 packing needs bits=4");
  QLX_REQUIRE(storage != 1 || bits == 8, "signed storage needs bits=8");
  QLX_REQUIRE(scale_kind == QLX_SCALE_F16 || scale_kind == QLX_SCALE_BF16, "bad scale kind");
  launch_quantize(IntQuant{bits, scale_kind == QLX_SCALE_F16, nudge, storage}, (const uint16_t*)w, data,
                  (uint16_t*)scale, rows, k, group, (hipStream_t)stream);
  QLX_LAUNCH_CHECK("quantize_weight");
}

int qlx_dequantize(const void* data, const void* scale, void* out, int rows, int k, int groups,
                   int bits, int scale_kind, int storage, void* stream) {
  QLX_REQUIRE(rows > 0 && k > 0 && groups > 0 && k % groups == 0, "bad dequantize shape");
  QLX_REQUIRE(storage != 2 || k % 8 == 0, "k32 words need K % 8 == 0");
  dequantize_kernel<<<blocks_for((size_t)rows * k, 256), 256, 0, (hipStream_t)stream>>>(
      data, (const uint16_t*)scale, (uint16_t*)out, rows, k, groups, bits,
      scale_kind == QLX_SCALE_F16, storage);
  QLX_LAUNCH_CHECK("dequantize");
}

int qlx_prepare_ref(const void* data, void* out, int rows, int k, int bits, int tiled, void* stream) {
  QLX_REQUIRE(k % 128 == 0, "K=%d is not a multiple of 128", k);
  QLX_REQUIRE(rows % 16 == 0, "rows=%d is not a multiple of 16", rows);
  QLX_REQUIRE(bits == 8 || bits == 4, "weights are 8 or 4 bits");
  QLX_REQUIRE(bits == 8 || tiled, "4-bit weights are stored tiled");
  const size_t n = (size_t)rows * (k / (bits == 4 ? 128 : 64));
  prepare_ref_kernel<<<blocks_for(n, 256), 256, 0, (hipStream_t)stream>>>(
      (const uint8_t*)data, (uint8_t*)out, rows, k, bits, tiled);
  QLX_LAUNCH_CHECK("prepare_ref");
}

int qlx_row_major_ref(const void* weight, void* out, int rows, int k, void* stream) {
  QLX_REQUIRE(k % 128 == 0 && rows % 16 == 0, "bad row_major shape");
  row_major_ref_kernel<<<blocks_for((size_t)rows * k, 256), 256, 0, (hipStream_t)stream>>>(
      (const uint8_t*)weight, (uint8_t*)out, rows, k);
  QLX_LAUNCH_CHECK("row_major_ref");
}

int qlx_quantize_fp8_weight(const void* w, void* code, void* scale, int rows, int k, int group,
                            void* stream) {
  QLX_REQUIRE(rows > 0 && k > 0 && group > 0 && k % group == 0, "%d is not a multiple of %d", k, group);
  QLX_REQUIRE(group % 8 == 0, "group %d must be a multiple of 8", group);
  launch_quantize(Fp8Quant{}, (const uint16_t*)w, code, (uint16_t*)scale, rows, k, group, (hipStream_t)stream);
  QLX_LAUNCH_CHECK("quantize_fp8_weight");
}

int qlx_quantize_fp8_act(const void* x, void* code, float* scale, int m, int k, void* stream) {
  QLX_REQUIRE(m > 0 && k > 0 && k % 8 == 0, "activation K=%d must be a positive multiple of 8", k);
  // Threads for every 8 values of a row up to 8192, two pieces per thread to 16384: 256 threads that
  // read a row twice took 2.80 and 4.20 us per call in a graph (8 rows of 2560, 9728), these 2.38 and 2.85.
  const int octets = k >> 3, u = octets <= 1024 ? 1 : (octets <= 2048 ? 2 : 0);
  const int threads = u ? ((octets + u - 1) / u + 63) / 64 * 64 : 1024;
  const auto fn = u == 1 ? quantize_fp8_act_kernel<1> : (u == 2 ? quantize_fp8_act_kernel<2> : quantize_fp8_act_kernel<0>);
  fn<<<m, threads, 0, (hipStream_t)stream>>>((const uint16_t*)x, (uint8_t*)code, scale, k);
  QLX_LAUNCH_CHECK("quantize_fp8_act");
}

int qlx_fp8_selfcheck(unsigned long long* counts, void* stream) {
  QLX_REQUIRE(counts != nullptr, "counts is null");
  fp8_selfcheck_kernel<<<dim3(32, 0x7f81), 256, 0, (hipStream_t)stream>>>(counts);
  QLX_LAUNCH_CHECK("fp8_selfcheck");
}

int qlx_int8_prepare(const void* row_major_ref, void* out, int rows, int k, void* stream) {
  QLX_REQUIRE(k % 64 == 0 && rows > 0, "bad int8_prepare shape");
  int8_prepare_kernel<<<blocks_for((size_t)rows * k, 256), 256, 0, (hipStream_t)stream>>>(
      (const uint8_t*)row_major_ref, (int8_t*)out, rows, k);
  QLX_LAUNCH_CHECK("int8_prepare");
}

int qlx_quantize_act_int8(const void* x, void* q, float* scale, void* q2, float* scale2, int m, int k,
                          void* stream) {
  QLX_REQUIRE(m > 0 && k > 0 && k % 64 == 0, "activation K=%d must be a multiple of 64", k);
  QLX_REQUIRE(!q2 || scale2, "a second component needs its scales");
  const size_t work = (size_t)m * (k / 64);
  quantize_act_int8_kernel<<<blocks_for(work, 4), 256, 0, (hipStream_t)stream>>>(
      (const uint16_t*)x, (int8_t*)q, scale, (int8_t*)q2, scale2, m, k);
  QLX_LAUNCH_CHECK("quantize_act_int8");
}

}  // extern "C"

// ---- MI355X tile layout (load time) ------------------------------------------------------

namespace qlx {

// dst block (tile t, step s) = 2 KB ordered [j][c][r][16 B], taken from row 16t + r, bytes
// 128s + 64j + 16c of the row-major source. One thread per 16-byte chunk.
__global__ void __launch_bounds__(256)
tile_rows_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, int rows, int row_bytes) {
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  const size_t total = (size_t)rows * row_bytes / 16;
  if (o >= total) return;
  const int within = (int)(o & 127);  // 128 chunks per 2 KB block
  const size_t blk = o >> 7;
  const int steps = row_bytes >> 7;
  const int t = (int)(blk / steps), s = (int)(blk % steps);
  const int j = within >> 6, c = (within >> 4) & 3, r = within & 15;
  dst[o] = src[((size_t)(16 * t + r) * row_bytes + 128 * s + 64 * j + 16 * c) / 16];
}

}  // namespace qlx

extern "C" int qlx_tile_rows(const void* src, void* dst, int rows, int row_bytes, void* stream) {
  QLX_REQUIRE(rows > 0 && rows % 16 == 0, "rows=%d must be a positive multiple of 16", rows);
  QLX_REQUIRE(row_bytes > 0 && row_bytes % 128 == 0, "row bytes %d must be a multiple of 128", row_bytes);
  const size_t chunks = (size_t)rows * row_bytes / 16;
  qlx::tile_rows_kernel<<<(unsigned)((chunks + 255) / 256), 256, 0, (hipStream_t)stream>>>(
      (const uint4*)src, (uint4*)dst, rows, row_bytes);
  QLX_LAUNCH_CHECK("tile_rows");
}
