// Resident-activation GEMM for 1..64 tokens: y[m][n] = sum_k x[m][k] * deq(W)[n][k].
//
// The other kernels here read every activation fragment from LDS once per weight tile (1 KB for
// every 1 KB of 8-bit weights and 16 tokens, 4 KB for 4-bit ones), after a pass that stages the
// activation and a barrier, and run the code-bias chain beside the main one. Here a wave keeps one
// K range for the whole launch, so its activation fragments and code-bias totals stay in registers:
//   * a workgroup of 8 waves owns one K slice and a run of 16-row tiles; the slice's units go to
//     the waves evenly, at most U each (a unit is 1 KB of a tile: one 16-byte load per lane, 128 k
//     of 4-bit or 64 k of 8-bit codes). A wave streams its units of every tile of the run, D tiles
//     ahead of its MFMAs. Weights go from memory through registers into MFMAs; nothing else is
//     read per tile but the scales;
//   * the activation is loaded in memory order and turned into fragments through LDS, unit by
//     unit, while the first weights are on their way. This start is what bounds the calls of many
//     tokens: 2560 x 19456 W4A16 at 64 tokens 19.3 us with loads in fragment order, 18.0 now;
//     4096 x 2560 W8A16 at 32 tokens 9.5 and 9.1 (in one slice 12.3 and 9.3);
//   * the 8 partial sums of D tiles meet in LDS (two sets, one barrier per D tiles); every wave
//     adds its part of them in wave order and writes outputs;
//   * K slices (where one slice does not fit the registers, or the tiles do not fill the CUs) write
//     fp32 planes that the run's last workgroup sums in slice order;
//   * 33..64 tokens run as two blocks of 32, ids 8 apart (one XCD), the second reading the weights
//     from that XCD's L2.
// The MFMA operands are swapped against gemm.h: A rows are tokens and B columns weight rows, so a
// lane finishes one weight row and needs one scale per group. Loads past a run, a slice or the
// tokens are given offsets out of their buffer's range: they read zeros without memory traffic and
// keep the in-order memory counter exact.
#pragma once

#include "gemm_launch.h"

namespace qlx {

struct ResidentArgs {
  const void* w;
  const void* ws;
  const void* x;
  const float* xs;  // FP8: token scales
  uint16_t* y;
  float* work;
  int* tickets;
  int m, n, k, half, swiglu;
  int planes;         // the outputs are fp32 planes (K slices, or the planes themselves); 2: y is their fp32 sum
  int units, per_slice, splits;
  int ntiles, groups, tblocks;
  int strided;        // a workgroup's tiles lie `groups` apart (whole K only)
  int run, longer;    // tiles of a run: `run`, one more in the first `longer` runs
  unsigned wbytes, sbytes;
};

// What a unit of a format is: KV values of K, NF 16-byte activation fragments per 16 tokens, NG
// scale groups (0: one scale per output channel), and where its bytes lie in a tile.
template <class F>
struct Unit;
template <>
struct Unit<FmtW4> {
  static constexpr int KV = 128, NF = 4, NG = 1;
  static constexpr uint32_t BIAS = 0x43084308u;
};
template <>
struct Unit<FmtW8> {
  static constexpr int KV = 64, NF = 2, NG = 0;
  static constexpr uint32_t BIAS = 0x43004300u;
};
template <>
struct Unit<FmtFP8> {
  static constexpr int KV = 64, NF = 1, NG = 0;
  static constexpr uint32_t BIAS = 0u;
};
template <>
struct Unit<FmtRef<8>> {
  static constexpr int KV = 64, NF = 2, NG = 1;
  static constexpr uint32_t BIAS = 0x43004300u;
};
template <>
struct Unit<FmtRef<4>> {
  static constexpr int KV = 128, NF = 4, NG = 2;
  static constexpr uint32_t BIAS = 0x43084308u;
};
template <class F>
constexpr bool is_ref() {
  return std::is_same<F, FmtRef<8>>::value || std::is_same<F, FmtRef<4>>::value;
}

// Tiles a wave has in flight, and whose partial sums meet at one barrier: about 8 KB per wave (64 KB
// per CU), and LDS for two sets of partial sums (16 KB per tile and 16 tokens).
// (FmtRef<4> at two token fragments: 3 tiles of 3 units spilled registers.)
template <class F>
__host__ __device__ constexpr int resident_depth(int mt, int u) {
  if (std::is_same<F, FmtRef<4>>::value && mt == 2 && u == 3) return 2;
  return u >= 6 ? 1 : (u >= 4 ? 2 : (u == 3 ? 3 : 4));
}
// Units a wave may hold: activation fragments (4 NF registers per unit and 16 tokens), bias totals
// (4 NG) and the weights in flight within two waves per SIMD (256 registers each).
template <class F>
__host__ __device__ constexpr int resident_max_units(int mt) {
  if (std::is_same<F, FmtW4>::value) return mt == 1 ? 6 : 3;
  if (std::is_same<F, FmtRef<4>>::value) return mt == 1 ? 5 : 3;
  if (std::is_same<F, FmtRef<8>>::value) return mt == 1 ? 8 : 5;
  return mt == 1 ? 10 : 8;
}

constexpr unsigned kOutOfRange = 0x80000000u;  // or'ed into an offset of a buffer of under 2 GiB

__device__ __forceinline__ __amdgpu_buffer_rsrc_t resident_rsrc(const void* p, unsigned bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(p);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(((uint64_t)hi << 32) | lo), (short)0, (int)bytes,
                                           0x00020000);
}
__device__ __forceinline__ uint4 resident_load16(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, soff, 0);
  return uint4{v[0], v[1], v[2], v[3]};
}

// 4 x 4 transpose across the lanes 16 apart: register i of lane group c becomes what register c of
// lane group i held.
__device__ __forceinline__ void transpose_rows(uint32_t (&a)[4]) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto r = __builtin_amdgcn_permlane32_swap(a[i], a[i + 2], false, false);
    a[i] = r[0], a[i + 2] = r[1];
  }
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    const auto r = __builtin_amdgcn_permlane16_swap(a[i], a[i + 1], false, false);
    a[i] = r[0], a[i + 1] = r[1];
  }
}

// What each of the four lane groups of 16 holds in v, to all of them: out[i] = group i's value.
__device__ __forceinline__ void spread_groups(uint32_t v, uint32_t* out) {
  const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // {0, 1, 0, 1}, {2, 3, 2, 3}
  const auto a = __builtin_amdgcn_permlane16_swap(h[0], h[0], false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(h[1], h[1], false, false);
  out[0] = a[0], out[1] = a[1], out[2] = b[0], out[3] = b[1];
}

// A unit's weight codes as MFMA fragments (NF of them; exact bf16 of code + bias).
template <class F>
__device__ __forceinline__ void unit_frags(const uint4& c, uint4 (&f)[Unit<F>::NF]) {
  if constexpr (std::is_same<F, FmtW4>::value) {
    const uint32_t wd[4] = {c.x, c.y, c.z, c.w};
#pragma unroll
    for (int t = 0; t < 4; ++t) f[t] = uint4{nib_pair(wd[t], 0), nib_pair(wd[t], 4), nib_pair(wd[t], 8), nib_pair(wd[t], 12)};
  } else if constexpr (std::is_same<F, FmtRef<4>>::value) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int sh = 4 * j;
      f[2 * j] = uint4{nib_pair(c.x, sh), nib_pair(c.x, sh + 8), nib_pair(c.y, sh), nib_pair(c.y, sh + 8)};
      f[2 * j + 1] = uint4{nib_pair(c.z, sh), nib_pair(c.z, sh + 8), nib_pair(c.w, sh), nib_pair(c.w, sh + 8)};
    }
  } else {
    constexpr uint32_t flip = std::is_same<F, FmtW8>::value ? 0x80808080u : 0u;
    const uint2 p0 = bytes_to_bf16(c.x ^ flip), p1 = bytes_to_bf16(c.y ^ flip);
    const uint2 p2 = bytes_to_bf16(c.z ^ flip), p3 = bytes_to_bf16(c.w ^ flip);
    f[0] = uint4{p0.x, p0.y, p1.x, p1.y};
    f[1] = uint4{p2.x, p2.y, p3.x, p3.y};
  }
}

__device__ __forceinline__ f32x4 mfma_bf16(const uint4& a, const uint4& b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_fp8(const uint4& a, const uint4& b, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8((long)(((unsigned long)a.y << 32) | a.x),
                                                 (long)(((unsigned long)b.y << 32) | b.x), c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8((long)(((unsigned long)a.w << 32) | a.z),
                                                    (long)(((unsigned long)b.w << 32) | b.z), c, 0, 0, 0);
}

// The 16-byte chunk of a unit's row that lane group c reads as its fragment t. The reference formats
// take dwords from all chunks of a block (unit_order).
template <class F>
__device__ __forceinline__ int frag_chunk(int c, int t) {
  return is_ref<F>() ? 4 * t + c : Unit<F>::NF * c + t;
}
// A unit's fragments into the order in which the codes unpack.
template <class F>
__device__ __forceinline__ void unit_order(uint4 (&f)[Unit<F>::NF]) {
#pragma unroll
  for (int t = 0; t < Unit<F>::NF; ++t) {
    if constexpr (is_ref<F>()) {
      // The reference's permutation: lane group c of a 64-value block takes the pairs 16 s + 2 c and
      // 16 s + 2 c + 8 of every s (FmtRef::stage_chunk), dword c of each of the block's 8 chunks.
      uint32_t d[4] = {f[t].x, f[t].y, f[t].z, f[t].w};
      transpose_rows(d);
      f[t] = uint4{d[0], d[1], d[2], d[3]};
      if constexpr (std::is_same<F, FmtRef<4>>::value)
        f[t] = uint4{__builtin_amdgcn_perm(d[1], d[0], 0x05040100u), __builtin_amdgcn_perm(d[1], d[0], 0x07060302u),
                     __builtin_amdgcn_perm(d[3], d[2], 0x05040100u), __builtin_amdgcn_perm(d[3], d[2], 0x07060302u)};
    } else {
      f[t] = F::order(f[t]);
    }
  }
}

// Orders the wave's LDS accesses across its lanes, which no barrier of the workgroup does here: the
// hardware keeps a wave's LDS operations in order, this keeps the compiler from moving them (no instruction).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The code is kept small, one copy of each part: a launch of ~10 us runs it from a cold instruction
// cache. (A first version, with the epilogue inlined per tile in flight and token fragment, had 31
// to 138 KB of code and took 13.1 us where this one, 10 KB, takes 9.6: W4A16 gate_up of one token.)
template <class F, int MT, int U, int D, bool FEW>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) resident_kernel(ResidentArgs a) {
  using UT = Unit<F>;
  constexpr int NF = UT::NF, NG = UT::NG, P = D * MT;
  constexpr bool FP8 = std::is_same<F, FmtFP8>::value;
  constexpr int XB = F::XBYTES;
  extern __shared__ __align__(16) float red[];  // [2][8 waves][P][4][64]
  const int lane = threadIdx.x & 63, c = lane >> 4, r = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int bid = blockIdx.x, m0 = 0, mrows = a.m, tb_id = 0;
  if (a.tblocks == 2) {  // ids 16 q + 8 b + x: workgroup 8 q + x, tokens 32 b ..
    tb_id = (bid >> 3) & 1;
    bid = 8 * (bid >> 4) + (bid & 7);
    m0 = 32 * tb_id;
    mrows = min(32, a.m - m0);
  }
  const int g = bid, s = blockIdx.y;
  // The workgroup's tiles: t0, t0 + step, .. A run of consecutive tiles lets a CU's stores of one
  // token (32 bytes a tile, 16 with SwiGLU; 64 in a plane) fill cache lines in its own L2. Long runs
  // of whole-K calls take every groups-th tile instead, so that the CUs read one region together:
  // 151936 x 2560 W4A16 at 1 / 16 tokens 41.7 -> 38.9, 47.5 -> 45.6 us (gate_up at 64 tokens 18.4 ->
  // 20.9 that way, K slices of down at 32 tokens 12.1 -> 13.0).
  const int nt = a.run + (g < a.longer ? 1 : 0), step = a.strided ? a.groups : 1;
  const int t0 = a.strided ? g : g * a.run + min(g, a.longer);
  // The slice's units go to the waves as evenly as they can: U or U - 1 each (fewer in a short last
  // slice). `held` units of this wave, from u0.
  const int nu = min(a.per_slice, a.units - s * a.per_slice), base = nu >> 3, more = nu & 7;
  const int u0 = s * a.per_slice + wave * base + min(wave, more), held = base + (wave < more ? 1 : 0);
  unsigned idle[U];
#pragma unroll
  for (int u = 0; u < U; ++u) idle[u] = u < held ? 0u : kOutOfRange;

  const __amdgpu_buffer_rsrc_t xr =
      resident_rsrc(static_cast<const char*>(a.x) + (size_t)m0 * a.k * XB, (unsigned)mrows * (unsigned)a.k * XB);
  const __amdgpu_buffer_rsrc_t wr = resident_rsrc(a.w, a.wbytes), sr = resident_rsrc(a.ws, a.sbytes);
  const unsigned tile_bytes = (unsigned)a.units * 1024u;
  // Lane offsets of a tile's weights and scales; tiles past the run out of range.
  struct At {
    unsigned w, sc;
  };
  auto tile_at = [&](int i) __attribute__((always_inline)) {
    const unsigned past = i < nt ? 0u : kOutOfRange;
    const int t = min(t0 + i * step, a.ntiles - 1);
    // SwiGLU tiles hold gate rows 8 t .. and the matching up rows half + 8 t ..
    const int wrow = a.swiglu ? (r < 8 ? 8 * t + r : a.half + 8 * t + r - 8) : 16 * t + r;
    const int rr = wrow & 15;
    unsigned off = (unsigned)(wrow >> 4) * tile_bytes;
    if constexpr (std::is_same<F, FmtRef<8>>::value) off += (rr >> 3) * 1024 + (rr & 7) * 64 + c * 16;
    else if constexpr (std::is_same<F, FmtRef<4>>::value) off += (rr >> 3) * 512 + (rr & 7) * 64 + c * 16;
    else off += (c * 16 + rr) * 16;
    return At{off | past, (unsigned)wrow * (unsigned)(NG ? a.units * NG * 2 : 2) | past};
  };
  uint4 xf[U][MT][NF], wb[D][U];
  // A tile's scales: lane group c loads those of units c, c + 4, .. and hands them on
  // (spread_groups): a load per unit, every lane group the same 16 rows, cost as much issue as the
  // unit's weights.
  constexpr int SQ = NG ? (U + 3) / 4 : 1;
  uint32_t sb[D][SQ];
  // Scalar offsets stay inside their buffer for units past the slice too (a wave of a short last slice
  // may hold several fewer than U): whether a load is in range is decided by the lane offset alone.
  const int last_unit = a.units - 1;
  auto load_unit = [&](int d, int u, const At& at) __attribute__((always_inline)) {
    const int uu = min(u0 + u, last_unit);
    wb[d][u] = resident_load16(wr, at.w | idle[u], std::is_same<F, FmtRef<8>>::value ? (uu >> 1) * 2048 + (uu & 1) * 512 : uu * 1024);
  };
  const int su = min(u0, last_unit);
  auto load_scales = [&](int d, const At& at) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < SQ; ++q) {
      const unsigned off = at.sc | (4 * q + c < held ? 0u : kOutOfRange);
      if constexpr (NG == 1) sb[d][q] = __builtin_amdgcn_raw_buffer_load_b16(sr, (int)(off + 2 * (4 * q + c)), su * 2, 0);
      else if constexpr (NG == 2) sb[d][q] = __builtin_amdgcn_raw_buffer_load_b32(sr, (int)(off + 4 * (4 * q + c)), su * 4, 0);
      else sb[d][0] = __builtin_amdgcn_raw_buffer_load_b16(sr, (int)at.sc, 0, 0);
    }
  };
  // Activations are loaded in memory order -- load t: ROWS token rows of the unit, 16 bytes a lane along
  // a row -- and turned into fragments (lane r: token r) through the wave's part of the second set of
  // partial sums, idle until the first barrier. (Loads in fragment order, consecutive lanes in
  // consecutive rows, take the CU 4 times as long: 160 KB by 8 waves 4.6 us, in memory order 1.7.)
  // Slots of a row lie rotated by its index (exclusive or), so that reads hit every bank alike.
  constexpr int CH = 4 * NF, ROWS = 16 / NF, NL = FEW ? 1 : NF;  // 16-byte chunks of a row; rows, loads
  uint4* const turn = reinterpret_cast<uint4*>(red + 8 * P * 256) + wave * (64 * NL);
  const unsigned xoff = (unsigned)(lane / CH) * (unsigned)a.k * XB + (unsigned)(lane % CH) * 16u;
  // Unit by unit its weights of the first D tiles, then its activation fragments: the order in which
  // the first block needs them, memory's requests before the cache's.
  {
    At at[D];
#pragma unroll
    for (int d = 0; d < D; ++d) at[d] = tile_at(d);
#pragma unroll
    for (int d = 0; d < D; ++d) load_scales(d, at[d]);
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int d = 0; d < D; ++d) load_unit(d, u, at[d]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < NL; ++t)  // rows past the tokens lie past the buffer: zeros
          xf[u][mt][t] = resident_load16(xr, (xoff + (unsigned)(16 * mt + t * ROWS) * (unsigned)a.k * XB) | idle[u],
                                         min(u0 + u, last_unit) * (UT::KV * XB));
    }
  }
  // Code-bias totals: the main chain with every code at the bias, so that a zero weight cancels
  // exactly.
  constexpr int PER = NG ? NF / (NG ? NG : 1) : NF;  // fragments of one scale group
  const uint4 bias = {UT::BIAS, UT::BIAS, UT::BIAS, UT::BIAS};
  f32x4 tb[NG ? U : 1][NG ? NG : 1][MT];
#pragma unroll
  for (int u = 0; u < (NG ? U : 1); ++u)
#pragma unroll
    for (int j = 0; j < (NG ? NG : 1); ++j)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) tb[u][j][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  const unsigned plane_bytes = ((unsigned)(a.splits - 1) * (unsigned)a.m + (unsigned)mrows) * (unsigned)a.n * 4u;
  const __amdgpu_buffer_rsrc_t pr =
      resident_rsrc(a.work + (size_t)m0 * a.n, a.planes ? plane_bytes : 0u);

  int buf = 0;
  for (int it = 0; it < nt; it += D) {
    At next[D];
#pragma unroll
    for (int d = 0; d < D; ++d) next[d] = tile_at(it + D + d);
    f32x4 acc[D][MT];
    uint32_t ss[D][NG ? 4 * SQ : 1];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if constexpr (NG == 0) {
        ss[d][0] = sb[d][0];
      } else {
#pragma unroll
        for (int q = 0; q < SQ; ++q) spread_groups(sb[d][q], &ss[d][4 * q]);
      }
      load_scales(d, next[d]);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[d][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    // Activation fragments of unit u into the codes' order, and its bias totals (first block only).
    auto ready_unit = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
        for (int t = 0; t < NL; ++t) {
          const int row = t * ROWS + lane / CH;
          turn[row * CH + ((lane % CH) ^ (row / (16 / CH)))] = xf[u][mt][t];
        }
        wave_lds_order();
        const int row = FEW ? r % ROWS : r;  // rows past the tokens: others', whose products are dropped
#pragma unroll
        for (int t = 0; t < NF; ++t)
          xf[u][mt][t] = turn[row * CH + (frag_chunk<F>(c, t) ^ (row / (16 / CH)))];
        wave_lds_order();
        if constexpr (!FP8) {
          unit_order<F>(xf[u][mt]);
#pragma unroll
          for (int t = 0; t < NF; ++t) {
            f32x4& b = tb[NG ? u : 0][NG ? t / PER : 0][mt];
            b = mfma_bf16(xf[u][mt][t], bias, b);
          }
        }
      }
    };
    auto multiply = [&](int d, int u) __attribute__((always_inline)) {
      if constexpr (FP8) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[d][mt] = mfma_fp8(xf[u][mt][0], wb[d][u], acc[d][mt]);
      } else {
        uint4 wf[NF];
        unit_frags<F>(wb[d][u], wf);
        if constexpr (NG == 0) {
#pragma unroll
          for (int t = 0; t < NF; ++t)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[d][mt] = mfma_bf16(xf[u][mt][t], wf[t], acc[d][mt]);
        } else {
#pragma unroll
          for (int j = 0; j < NG; ++j) {
            const uint32_t bits = j ? ss[d][u] >> 16 : ss[d][u] & 0xffffu;
            const float sc = is_ref<F>() ? h2f((uint16_t)bits) : bf2f(bits);
            f32x4 tmp[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) tmp[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < PER; ++t)
#pragma unroll
              for (int mt = 0; mt < MT; ++mt) tmp[mt] = mfma_bf16(xf[u][mt][j * PER + t], wf[j * PER + t], tmp[mt]);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
#pragma unroll
              for (int i = 0; i < 4; ++i) acc[d][mt][i] = fmaf(sc, tmp[mt][i] - tb[u][j][mt][i], acc[d][mt][i]);
          }
        }
      }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u == U - 1 && held < U) break;  // a wave of one unit fewer
      if (it == 0) ready_unit(u);
#pragma unroll
      for (int d = 0; d < D; ++d) multiply(d, u);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int d = 0; d < D; ++d) load_unit(d, u, next[d]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = acc[d][mt][i];
          if constexpr (NG == 0) v = (FP8 ? v : v - tb[0][0][mt][i]) * bf2f(ss[d][0]);  // the channel's scale
          red[(((buf * 8 + wave) * P + d * MT + mt) * 4 + i) * 64 + lane] = v;
        }
    __syncthreads();
    // Outputs: wave w sums tokens (w & 1) and (w & 1) + 2 of each lane group's four, of the pairs
    // (tile, token fragment) p = w >> 1, + 4, ..
    for (int p = wave >> 1; p < P; p += 4) {
      const int i = it + p / MT, t = t0 + i * step;
      const int mm = 16 * (p % MT) + 4 * c + (wave & 1);  // the first token, within its block
      if (i >= nt || 16 * (p % MT) + (wave & 1) >= mrows) continue;
      const float* src = red + ((buf * 8 * P + p) * 4 + (wave & 1)) * 64 + lane;
      float v0 = src[0], v1 = src[128];
#pragma unroll
      for (int w = 1; w < 8; ++w) v0 += src[w * P * 256], v1 += src[w * P * 256 + 128];
      if constexpr (FP8) {
        v0 *= gmem(a.xs)[m0 + min(mm, mrows - 1)];
        v1 *= gmem(a.xs)[m0 + min(mm + 2, mrows - 1)];
      }
      if (a.planes) {
        const int wrow = a.swiglu ? (r < 8 ? 8 * t + r : a.half + 8 * t + r - 8) : 16 * t + r;
        const unsigned off = (((unsigned)s * (unsigned)a.m + (unsigned)mm) * (unsigned)a.n + (unsigned)wrow) * 4u;
        if (mm < mrows) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v0), pr, (int)off, 0, 16);
        if (mm + 2 < mrows) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v1), pr, (int)off, a.n * 8, 16);
      } else if (a.swiglu) {
        // Lanes r < 8 hold gate rows, r + 8 the matching up rows. Lanes r < 8 take the first token's
        // pair, lanes r >= 8 the second one's: each sends what the other half lacks, a rotation by 8
        // within 16 lanes.
        const bool lo = r < 8;
        const float x = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(lo ? v1 : v0), 0x128, 0xf, 0xf, false));
        const float o = swiglu_bf(lo ? v0 : x, lo ? x : v1);
        const float nb = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(o), 0xb1, 0xf, 0xf, false));
        const int mo = lo ? mm : mm + 2;
        if (mo < mrows && !(r & 1)) store_pair(a.y, (size_t)(m0 + mo) * a.half + 8 * t + (r & 7), o, nb);
      } else {
        // even lanes store the first token's pair of rows, odd lanes the second's
        const float x = __int_as_float(
            __builtin_amdgcn_update_dpp(0, __float_as_int(r & 1 ? v0 : v1), 0xb1, 0xf, 0xf, false));
        const int mo = r & 1 ? mm + 2 : mm;
        if (mo < mrows)
          store_pair(a.y, (size_t)(m0 + mo) * a.n + 16 * t + (r & 14), r & 1 ? x : v0, r & 1 ? v1 : x);
      }
    }
    buf ^= 1;
  }
  if (a.tickets == nullptr) return;

  // ---- K slices: the run's last workgroup sums the planes in slice order -----------------------
  __shared__ int s_last;
  publish_stores();
  if (threadIdx.x == 0) {
    int* ticket = &a.tickets[a.tblocks == 2 ? 2 * g + tb_id : g];
    const int prev = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = prev == a.splits - 1;
    if (s_last) __hip_atomic_store(ticket, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  // 4 consecutive output rows of one token per item (SwiGLU: 4 gate rows and their up rows).
  const int quads = a.swiglu ? 2 : 4, per_tok = nt * quads;
  const unsigned pstride = (unsigned)a.m * (unsigned)a.n * 4u;
  auto f4 = [](const u32x4& v) {
    return f32x4{__uint_as_float(v[0]), __uint_as_float(v[1]), __uint_as_float(v[2]), __uint_as_float(v[3])};
  };
  for (int idx = threadIdx.x; idx < per_tok * mrows; idx += 512) {
    const int mm = idx / per_tok, cc = idx - mm * per_tok;
    const int t = t0 + cc / quads, q4 = 4 * (cc % quads);
    const int row = a.swiglu ? 8 * t + q4 : 16 * t + q4;
    const unsigned off = ((unsigned)mm * (unsigned)a.n + (unsigned)row) * 4u;
    f32x4 gv = {0.f, 0.f, 0.f, 0.f}, uv = {0.f, 0.f, 0.f, 0.f};
    for (int sp0 = 0; sp0 < a.splits; sp0 += 8) {  // one round trip for up to 8 slices
      u32x4 lg[8], lu[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const unsigned po = off + (unsigned)min(sp0 + j, a.splits - 1) * pstride;
        lg[j] = __builtin_amdgcn_raw_buffer_load_b128(pr, (int)po, 0, 16);
        if (a.swiglu) lu[j] = __builtin_amdgcn_raw_buffer_load_b128(pr, (int)(po + (unsigned)a.half * 4u), 0, 16);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (sp0 + j < a.splits) {
          gv += f4(lg[j]);
          if (a.swiglu) uv += f4(lu[j]);
        }
    }
    if (a.swiglu) {
      const size_t o = (size_t)(m0 + mm) * a.half + row;
      store_pair(a.y, o, swiglu_bf(gv[0], uv[0]), swiglu_bf(gv[1], uv[1]));
      store_pair(a.y, o + 2, swiglu_bf(gv[2], uv[2]), swiglu_bf(gv[3], uv[3]));
    } else if (a.planes == 2) {
      *gmem(reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.y) + (size_t)(m0 + mm) * a.n + row)) = gv;
    } else {
      const size_t o = (size_t)(m0 + mm) * a.n + row;
      store_pair(a.y, o, gv[0], gv[1]);
      store_pair(a.y, o + 2, gv[2], gv[3]);
    }
  }
}

template <class F, int MT, int U, int D, bool FEW>
hipError_t resident_launch(const ResidentArgs& a, hipStream_t st) {
  constexpr int sums = 8 * D * MT * 1024, turn = 8 * (FEW ? 1 : Unit<F>::NF) * 1024;
  constexpr int lds = sums + (sums > turn ? sums : turn);
  static_assert(lds <= 128 * 1024, "partial sums");
  if (lds > 64 * 1024) {
    static int allowed = 64 * 1024;
    if (lds > allowed) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&resident_kernel<F, MT, U, D, FEW>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds);
      if (e != hipSuccess) return e;
      allowed = lds;
    }
  }
  resident_kernel<F, MT, U, D, FEW><<<dim3(a.groups * a.tblocks, a.splits), 512, lds, st>>>(a);
  return hipGetLastError();
}

// Runs of one tile take the instance that holds one tile (it would compute D).
template <class F, int MT, int U, bool FEW>
hipError_t resident_deep(const ResidentArgs& a, hipStream_t st) {
  if (a.run + (a.longer > 0) == 1) return resident_launch<F, MT, U, 1, FEW>(a, st);
  return resident_launch<F, MT, U, resident_depth<F>(MT, U), FEW>(a, st);
}

template <class F, int MT>
hipError_t resident_units(const ResidentArgs& a, int u, hipStream_t st) {
  constexpr int most = resident_max_units<F>(MT);
  hipError_t e = hipErrorInvalidValue;
  static_for<1, most + 1>([&](auto uc) {
    constexpr int U = decltype(uc)::value;
    if (u != U) return;
    if constexpr (MT == 1 && Unit<F>::NF > 1) {
      if (a.m <= 16 / Unit<F>::NF) {  // all of a unit's fragments in one load
        e = resident_deep<F, MT, U, true>(a, st);
        return;
      }
    }
    e = resident_deep<F, MT, U, false>(a, st);
  });
  return e;
}

// How a shape is cut: token blocks, units per wave and K slices. Returns false where the kernel
// does not serve it.
struct ResidentPlan {
  int u, splits, per_slice, groups, tblocks;
};
template <class F>
bool resident_plan(int m, int n, int k, int splits, ResidentPlan& p) {
  const int units = k / Unit<F>::KV, ntiles = n / 16;
  const int mt = m <= 16 ? 1 : 2, most = resident_max_units<F>(mt);
  p.tblocks = m > 32 ? 2 : 1;
  p.per_slice = (units + splits - 1) / splits;
  p.splits = (units + p.per_slice - 1) / p.per_slice;
  p.u = (p.per_slice + 7) / 8;
  if (p.u > most) return false;
  constexpr int cus = 256;  // one workgroup per CU
  p.groups = std::min(ntiles, std::max(1, cus / (p.splits * p.tblocks)));
  // two token blocks: whole sets of 8 workgroups, so that a pair of blocks shares an XCD
  if (p.tblocks == 2) {
    if (p.groups < 8) return false;
    p.groups &= ~7;
  }
  return true;
}

// Why the kernel cannot take a call of these sizes in `splits` K slices, nullptr where it can: its
// offsets within each operand are 32 bits, the top one of them the sign of a load out of range.
template <class F>
const char* resident_limit(int m, int n, int k, int splits) {
  constexpr long long most = 1ll << 31;
  if ((long long)(n / 16) * (k / Unit<F>::KV) * 1024 >= most) return "weights of under 2 GiB";
  if ((long long)std::min(m, 32) * k * F::XBYTES >= most) return "activations of under 2 GiB";
  if ((long long)splits * m * n * 4 >= most) return "planes of under 2 GiB";
  return nullptr;
}

template <class F>
int resident_run(const char* name, ResidentArgs a, int m, int n, int k, const qlx_plan* plan, void* stream) {
  QLX_REQUIRE(plan != nullptr, "%s: plan is NULL", name);
  QLX_REQUIRE(m >= 1 && m <= 64, "%s: m=%d must be in 1..64", name, m);
  QLX_REQUIRE(n >= 16 && n % 16 == 0 && k >= 128 && k % 128 == 0 && k % F::KSTEP == 0,
              "%s: n=%d k=%d do not fit the tiled format", name, n, k);
  QLX_REQUIRE(plan->mode >= QLX_MODE_BF16 && plan->mode <= QLX_MODE_SUM, "%s: mode %d", name, plan->mode);
  const int units = k / Unit<F>::KV;
  QLX_REQUIRE(plan->splits >= 1 && plan->splits <= units, "%s: splits must be 1..%d", name, units);
  ResidentPlan p;
  QLX_REQUIRE(resident_plan<F>(m, n, k, plan->splits, p), "%s: %d K slices leave a wave more than %d units", name,
              plan->splits, resident_max_units<F>(m <= 16 ? 1 : 2));
  const char* const limit = resident_limit<F>(m, n, k, p.splits);
  QLX_REQUIRE(limit == nullptr, "%s: %s (m=%d n=%d k=%d, %d slices)", name, limit, m, n, k, p.splits);
  // 16-byte buffer loads of weights and activations, 4-byte ones of scales
  QLX_REQUIRE(((uintptr_t)a.w | (uintptr_t)a.x) % 16 == 0 && ((uintptr_t)a.ws | (uintptr_t)a.y) % 4 == 0,
              "%s: operands must start on 16-byte boundaries (scales, outputs: 4)", name);
  QLX_REQUIRE(plan->mode != QLX_MODE_SUM || (uintptr_t)a.y % 16 == 0, "%s: fp32 outputs must start on a 16-byte boundary", name);
  const bool planes = plan->mode == QLX_MODE_PLANES, sum = plan->mode == QLX_MODE_SUM;
  QLX_REQUIRE(!planes || p.splits == plan->splits, "%s: %d splits leave %d non-empty planes", name, plan->splits, p.splits);
  QLX_REQUIRE(planes ? plan->workspace != nullptr
                     : p.splits == 1 || (plan->workspace != nullptr && plan->tickets != nullptr),
              "%s: K slices need a workspace and tickets, planes a workspace", name);
  a.m = m, a.n = n, a.k = k, a.half = n / 2, a.swiglu = plan->mode == QLX_MODE_SWIGLU;
  a.units = units, a.per_slice = p.per_slice, a.splits = p.splits;
  a.ntiles = n / 16, a.groups = p.groups, a.tblocks = p.tblocks;
  a.run = a.ntiles / a.groups, a.longer = a.ntiles % a.groups;
  a.strided = p.splits == 1 && a.run >= 12;
  a.wbytes = (unsigned)((long long)(n / 16) * units * 1024);
  a.sbytes = (unsigned)((long long)n * (Unit<F>::NG ? units * Unit<F>::NG : 1) * 2);
  a.planes = sum ? 2 : planes || p.splits > 1;
  a.work = sum && p.splits == 1 ? reinterpret_cast<float*>(a.y) : plan->workspace, a.tickets = !planes && p.splits > 1 ? plan->tickets : nullptr;
  const hipError_t e = m <= 16 ? resident_units<F, 1>(a, p.u, (hipStream_t)stream)
                               : resident_units<F, 2>(a, p.u, (hipStream_t)stream);
  return hip_status(e, name);
}

// One per format, each defined in the file that instantiates it.
int resident_w8a16(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream);
int resident_w4a16(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream);
int resident_fp8(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream);
int resident_ref8(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream);
int resident_ref4(const ResidentArgs& a, int m, int n, int k, const qlx_plan* plan, void* stream);

}  // namespace qlx
