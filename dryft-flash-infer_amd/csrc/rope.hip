// Per-head RMSNorm + RoPE of the fused QKV projection, K and V written into the cache
// (engine/kernels/rope.py:24-60 `_norm_rope`, :63-92 q/kv kernels, :125-166 the fused Q/K/V
// kernel, :169-218 the split-K planes variant, :96-122 the INT8 cache writes).
//
// Sixteen lanes per 128-value head (rope_common.h: the lane layout and the roundings, those of
// engine/kernels/reference.py:31-46). A workgroup of 256 threads covers 16 heads of one row: Q heads,
// then K heads, then V heads.
// From planes, x = bf16(sum of the fp32 planes in slice order) (rope.py:169-176).
// INT8 cache: per (token, head) scale max(amax |y|, 1e-12) / 127, codes
// clamp(floor(y / scale + 0.5), -127, 127) (rope.py:108-118).
#include "rope_common.h"
#include "../../include/qlinear.h"

namespace qlx {

struct RopeArgs {
  qlx_rope_args p;
  int heads;  // n_q + 2 n_kv
};

// 4 values of row `row` at column `col`, as bf16 pairs: read from qkv, or the planes' slice-order
// sums rounded once.
template <bool PLANES>
__device__ __forceinline__ u32x2 load4(const qlx_rope_args& p, int row, long long col) {
  if constexpr (!PLANES) {
    return *gmem(reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(p.qkv) + (size_t)row * p.stride + col));
  } else {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < p.splits; ++s) {
      const f32x4 v = *gmem(reinterpret_cast<const f32x4*>(p.planes + ((size_t)s * p.rows + row) * p.stride + col));
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] += v[i];
    }
    return u32x2{bf16_canonical_nan(bf16_pair_hw(acc[0], acc[1])), bf16_canonical_nan(bf16_pair_hw(acc[2], acc[3]))};
  }
}

__device__ __forceinline__ void unpack4(u32x2 d, float* f) {
  f[0] = bf2f(d[0] & 0xffffu), f[1] = bf2f(d[0] >> 16), f[2] = bf2f(d[1] & 0xffffu), f[3] = bf2f(d[1] >> 16);
}

// clamp(floor(f / sc + 0.5), -127, 127) of 4 values. y = 1 / sc: the quotient is the IEEE one wherever
// it can reach a code other than 0 (quotient_by_reciprocal); over an infinite scale finite values
// give 0, the others a NaN, which the clamp turns into -127.
__device__ __forceinline__ void store_int8(int8_t* dst, const float* f, float sc, float y) {
  uint32_t d = 0u;
  if (sc <= 3.40282347e38f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float c = fminf(fmaxf(floorf(quotient_by_reciprocal(f[i], sc, y) + 0.5f), -127.f), 127.f);
      d |= ((uint32_t)(int)c & 0xffu) << (8 * i);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) d |= (fabsf(f[i]) <= 3.40282347e38f ? 0u : 0x81u) << (8 * i);
  }
  *gmem(reinterpret_cast<uint32_t*>(dst)) = d;
}

// Max over the 16 lanes of a head.
__device__ __forceinline__ float head_max(float v) {
  v = fmaxf(v, __shfl_xor(v, 1, 64));
  v = fmaxf(v, __shfl_xor(v, 2, 64));
  v = fmaxf(v, __shfl_xor(v, 4, 64));
  return fmaxf(v, __shfl_xor(v, 8, 64));
}

// A lane's two groups of 4 values (bf16 pairs lo, hi: dims 4 j .., 64 + 4 j ..) into head slot `slot`
// of a bf16 cache, or quantized into an INT8 one with its scale.
template <bool INT8>
__device__ __forceinline__ void write_head(void* cache, float* scales, size_t slot, int j, const u32x2& lo, const u32x2& hi,
                                           bool writes) {
  if constexpr (INT8) {
    float fl[4], fh[4];
    unpack4(lo, fl);
    unpack4(hi, fh);
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) amax = fmaxf(amax, fmaxf(fabsf(fl[i]), fabsf(fh[i])));
    const float sc = fmaxf(head_max(amax), 1e-12f) / 127.0f, y = 1.0f / sc;
    if (!writes) return;
    int8_t* dst = reinterpret_cast<int8_t*>(cache) + slot * 128;
    store_int8(dst + 4 * j, fl, sc, y);
    store_int8(dst + 64 + 4 * j, fh, sc, y);
    if (j == 0) scales[slot] = sc;
  } else {
    if (!writes) return;
    uint16_t* dst = reinterpret_cast<uint16_t*>(cache) + slot * 128;
    *gmem(reinterpret_cast<u32x2*>(dst + 4 * j)) = lo;
    *gmem(reinterpret_cast<u32x2*>(dst + 64 + 4 * j)) = hi;
  }
}

// A launch is a chain of two memory round trips and a wave's instructions, fetched cold: one
// instance per source and cache type, 16 lanes per head (half the values, so half the instructions, of
// 8), value heads on lanes of their own. us per call in a graph at 1 / 64 rows of 32 + 8 heads: bf16
// cache 3.56 / 3.78 -> 2.45 / 2.85, INT8 4.49 / 4.76 -> 2.90 / 3.29 (8 lanes per head, all options in
// one kernel of 19 KB, a value head read by its key's lanes).
template <bool PLANES, bool INT8>
__global__ void __launch_bounds__(256) rope_kernel(RopeArgs ra) {
  const qlx_rope_args& p = ra.p;
  const int row = blockIdx.x;
  const int hh = blockIdx.y * 16 + (threadIdx.x >> 4);
  const int j = threadIdx.x & 15;
  // Lanes past the last head compute on head 0's data and store nothing (a head's 16 lanes
  // take the same branch, and no lane leaves before the shuffles).
  const bool active = hh < ra.heads;
  const int h = active ? hh : 0;
  const bool is_q = h < p.n_q, is_v = h >= p.n_q + p.n_kv;
  const int kvh = is_v ? h - p.n_q - p.n_kv : h - p.n_q;
  const long long col = is_q ? p.q_col + (long long)h * 128 : (is_v ? p.v_col : p.k_col) + (long long)kvh * 128;

  // The position first: the cos/sin rows it selects are the second of two dependent loads.
  const int tok = row % p.seq_len;
  const long long pos = p.pos_int64 ? reinterpret_cast<const long long*>(p.positions)[tok]
                                    : (long long)reinterpret_cast<const int*>(p.positions)[tok];
  u32x2 lo = load4<PLANES>(p, row, col + 4 * j), hi = load4<PLANES>(p, row, col + 64 + 4 * j);
  const bool in_table = pos >= 0 && pos < p.table_rows;
  const int seq = row / p.seq_len;
  const bool writes = active && in_table && pos < p.capacity;

  if (!is_v) {
    const uint16_t* gain = reinterpret_cast<const uint16_t*>(is_q ? p.q_norm_w : p.k_norm_w);
    const u32x2 wlr = *gmem(reinterpret_cast<const u32x2*>(gain + 4 * j)),
                whr = *gmem(reinterpret_cast<const u32x2*>(gain + 64 + 4 * j));
    const long long tp = in_table ? pos : 0;
    const uint16_t* cs = reinterpret_cast<const uint16_t*>(p.cos) + (size_t)tp * 128 + 4 * j;
    const uint16_t* sn = reinterpret_cast<const uint16_t*>(p.sin) + (size_t)tp * 128 + 4 * j;
    float cl[4], ch[4], sl[4], sh[4], xl[4], xh[4], wl[4], wh[4], yl[4], yh[4];
    unpack4(*gmem(reinterpret_cast<const u32x2*>(cs)), cl);
    unpack4(*gmem(reinterpret_cast<const u32x2*>(cs + 64)), ch);
    unpack4(*gmem(reinterpret_cast<const u32x2*>(sn)), sl);
    unpack4(*gmem(reinterpret_cast<const u32x2*>(sn + 64)), sh);
    unpack4(lo, xl);
    unpack4(hi, xh);
    unpack4(wlr, wl);
    unpack4(whr, wh);
    uint32_t ylp[2], yhp[2];
    rope_norm_rotate<4>(xl, xh, wl, wh, cl, ch, sl, sh, p.eps, yl, yh, ylp, yhp);
    lo = u32x2{ylp[0], ylp[1]}, hi = u32x2{yhp[0], yhp[1]};
    if (is_q) {
      if (!active) return;
      // a position outside the cos/sin table: the head reads as NaN
      if (!in_table) lo = hi = u32x2{0x7fc07fc0u, 0x7fc07fc0u};
      uint16_t* q = reinterpret_cast<uint16_t*>(p.q_out) + (size_t)row * p.n_q * 128 + (size_t)h * 128 + 4 * j;
      *gmem(reinterpret_cast<u32x2*>(q)) = lo;
      *gmem(reinterpret_cast<u32x2*>(q + 64)) = hi;
      return;
    }
  } else {
    lo = u32x2{bf16_canonical_nan(lo[0]), bf16_canonical_nan(lo[1])};
    hi = u32x2{bf16_canonical_nan(hi[0]), bf16_canonical_nan(hi[1])};
  }

  // The rotated K or the raw V head to slot pos of sequence row / seq_len.
  const size_t hs = (size_t)seq * p.n_kv + kvh;
  if (p.k_copy != nullptr && active) {
    uint16_t* copy = reinterpret_cast<uint16_t*>(is_v ? p.v_copy : p.k_copy) + (hs * p.seq_len + tok) * 128 + 4 * j;
    *gmem(reinterpret_cast<u32x2*>(copy)) = lo;
    *gmem(reinterpret_cast<u32x2*>(copy + 64)) = hi;
  }
  write_head<INT8>(is_v ? p.v_cache : p.k_cache, is_v ? p.v_scale : p.k_scale,
                   hs * p.capacity + (size_t)(writes ? pos : 0), j, lo, hi, writes);
}

}  // namespace qlx

using namespace qlx;

extern "C" int qlx_qkv_norm_rope(const qlx_rope_args* args, void* stream) {
  QLX_REQUIRE(args != nullptr, "norm_rope: null arguments");
  const qlx_rope_args& p = *args;
  QLX_REQUIRE(p.rows >= 0 && p.n_q >= 0 && p.n_kv >= 0 && p.n_q + p.n_kv > 0, "norm_rope: bad row or head counts");
  QLX_REQUIRE(p.seq_len >= 1 && p.rows % p.seq_len == 0, "norm_rope: rows (%d) must be a multiple of seq_len (%d)",
              p.rows, p.seq_len);
  QLX_REQUIRE((p.qkv == nullptr) != (p.planes == nullptr), "norm_rope: give qkv or planes, not both");
  QLX_REQUIRE(p.planes == nullptr || p.splits >= 1, "norm_rope: planes need splits >= 1");
  QLX_REQUIRE(p.stride > 0 && p.stride % 8 == 0, "norm_rope: row stride must be a positive multiple of 8");
  QLX_REQUIRE(p.table_rows >= 1 && p.cos && p.sin && p.positions, "norm_rope: cos/sin tables and positions needed");
  QLX_REQUIRE(p.n_q == 0 || (p.q_out && p.q_norm_w && p.q_col >= 0 && p.q_col % 8 == 0 &&
                             p.q_col + (long long)p.n_q * 128 <= p.stride),
              "norm_rope: Q heads need q_out, q_norm_w and columns inside the row");
  QLX_REQUIRE(p.n_kv == 0 || (p.k_cache && p.v_cache && p.k_norm_w && p.capacity >= 1 && p.k_col >= 0 &&
                              p.v_col >= 0 && p.k_col % 8 == 0 && p.v_col % 8 == 0 &&
                              p.k_col + (long long)p.n_kv * 128 <= p.stride &&
                              p.v_col + (long long)p.n_kv * 128 <= p.stride),
              "norm_rope: K/V heads need caches, k_norm_w, capacity and columns inside the row");
  QLX_REQUIRE((p.k_scale == nullptr) == (p.v_scale == nullptr), "norm_rope: give both cache scales or neither");
  QLX_REQUIRE((p.k_copy == nullptr) == (p.v_copy == nullptr), "norm_rope: give both bf16 copies or neither");
  if (p.rows == 0) return QLX_OK;
  RopeArgs ra{p, p.n_q + 2 * p.n_kv};
  const dim3 grid(p.rows, (ra.heads + 15) / 16);
  const auto fn = p.planes ? (p.k_scale ? rope_kernel<true, true> : rope_kernel<true, false>)
                           : (p.k_scale ? rope_kernel<false, true> : rope_kernel<false, false>);
  fn<<<grid, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(ra);
  QLX_LAUNCH_CHECK("norm_rope");
}
