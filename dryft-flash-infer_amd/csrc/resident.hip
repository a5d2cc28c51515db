// Resident-activation GEMM: the plan and the C entry point (resident.h holds the kernel).
#include "resident.h"

namespace qlx {

// K slices of a shape, 0 where the kernel does not serve it: the least of a time in microseconds,
// fitted to a sweep of 1 to 8 slices over the Qwen3-4B projections in all five formats at 1 to 64
// tokens and over 70 other shapes (n 960 to 24000, k 1024 to 13824; MI355X). A CU takes in about 25 KB
// of weights and 40 of activations per microsecond, the weights of the whole call come at 5.6 TB/s;
// slices cost their planes, a ticket and a round trip for the sum. The slices it picks take 0.3 % more
// time than the best of the eight on the Qwen3-4B projections, 1.1 % on the others (W8A16 down: 12.3
// -> 11.6 us at 24 tokens, 16.5 -> 14.3 at 64 against an earlier fit, which was 1.4 and 1.7 % off).
template <class F>
int resident_splits(int m, int n, int k) {
  const int units = k / Unit<F>::KV, ntiles = n / 16, rows = std::min(m, 32);
  int best = 0;
  double least = 0;
  for (int s = 1; s <= 8 && s <= units; ++s) {
    ResidentPlan p;
    if (!resident_plan<F>(m, n, k, s, p) || p.splits != s || resident_limit<F>(m, n, k, s)) continue;
    const int tiles = (ntiles + p.groups - 1) / p.groups;
    const double weights = std::max((double)ntiles * units / 5600, (double)tiles * p.per_slice / 25);
    const double acts = rows * (double)p.per_slice * (Unit<F>::KV * F::XBYTES / 1024.0) / 40;
    const int rounds = (tiles * 4 * rows + 511) / 512, depth = resident_depth<F>(rows > 16 ? 2 : 1, p.u);
    const double slices = s > 1 ? 0.8 + 1.2 * rounds + 0.2 * s + (double)s * m * n * 8 / 2e6 : 0;
    const double t = weights + acts + slices + 0.5 * std::min((tiles + depth - 1) / depth - 1, 2);
    if (best == 0 || t < least) best = s, least = t;
  }
  return best;
}

// Where another kernel streams a call faster, although this one serves it in `s` slices: the decode kernel
// up to 8 tokens, the skinny GEMM above. The lines are measured: both kernels at 8643 calls of 1 to 64
// tokens (n 1024 to 151936, k 1024 to 13824, distinct weights; MI355X), and at 1944 with SwiGLU; in
// brackets this kernel's time over the other's past the line (geometric mean). What they
// share is a workgroup's long run: probably as the other kernels' staging of the activation, which this one
// saves, is then spread over many tiles, while its sums over 8 waves, and planes, are paid for each.
// us per call, the other kernel / this one: 151936 x 2560 FP8 67.7 / 74.2 at one token, 68.8 / 81.6 at 16,
// W8A16 72.4 / 75.7 at 8, 67.8 / 81.2 at 16 (but 123.8 / 114.6 at 64), W4A16 37.5 / 38.9 at one token,
// 46.7 / 42.6 at 8; FP8 19456 x 2560 15.8 / 18.0 at 32; W8A16 32000 x 5120 52.7 / 61.1 at 64. FP8 of one
// token takes a launch fewer there: that kernel quantizes it itself.
static bool resident_yields(int fmt, int m, int n, int k, int s) {
  const long long bytes = (long long)n * k;
  const int tiles = n / 16;
  switch (fmt) {
    case QLX_FMT_FP8:
      if (m == 1 || bytes > (64ll << 20)) return true;
      if (m >= 9) return tiles >= 1024 || (s > 1 && tiles >= 640);  // [1.06 to 32 tokens, 1.14 above]
      return s > 1 && tiles >= (m <= 4 ? 256 : 512);                // [1.06, 1.08]
    case QLX_FMT_W8A16:
      if (m <= 32 && bytes > (64ll << 20)) return true;
      if (m >= 33) return (s > 1 || k <= 1024) && tiles > 1792;  // [1.14]
      return m >= 9 && tiles > (m <= 16 ? 1024 : 1536);          // [1.06, 1.06]
    case QLX_FMT_W4A16:
      if (m <= 4 && tiles >= 2 * 8 * 256) return true;
      // 28672 x 2560 of 16 tokens 11.5 / 14.1, but 49152 x 2560 18.9 / 17.9
      if (m >= 9 && m <= 32) return (tiles > 1536 && tiles <= 2048) || (m > 16 && s > 1 && tiles >= 4096);  // [1.05]
      return m <= 2 && s > 1 && tiles >= 256 && tiles <= 512;  // [1.04]
  }
  return false;
}

int resident_splits_of(int fmt, int m, int n, int k) {
  switch (fmt) {
    case QLX_FMT_W4A16: return resident_splits<FmtW4>(m, n, k);
    case QLX_FMT_W8A16: return resident_splits<FmtW8>(m, n, k);
    case QLX_FMT_FP8: return resident_splits<FmtFP8>(m, n, k);
    case QLX_FMT_REF8: return resident_splits<FmtRef<8>>(m, n, k);
    case QLX_FMT_REF4: return resident_splits<FmtRef<4>>(m, n, k);
  }
  return 0;
}

}  // namespace qlx

using namespace qlx;

extern "C" {

int qlx_plan_resident(int fmt, int mode, int m, int n, int k, qlx_plan* plan) {
  QLX_REQUIRE(plan != nullptr, "plan is NULL");
  const int kstep = fmt == QLX_FMT_W4A16 ? 256 : 128;
  QLX_REQUIRE(mode >= QLX_MODE_BF16 && mode <= QLX_MODE_SUM, "bad mode %d", mode);
  QLX_REQUIRE(m >= 1 && m <= 64 && n >= 16 && n % 16 == 0 && k >= kstep && k % kstep == 0,
              "shape m=%d n=%d k=%d does not fit format %d", m, n, k, fmt);
  const int s = resident_splits_of(fmt, m, n, k);
  qlx_plan p = {};
  p.mode = mode;
  p.waves = 8;
  p.kw = 8;
  p.rw = 1;
  p.splits = resident_yields(fmt, m, n, k, s) ? 0 : s;
  *plan = p;
  return QLX_OK;
}

int qlx_linear_resident(int fmt, const void* w, const void* w_scale, const void* x, const float* x_scale, void* y,
                        int m, int n, int k, const qlx_plan* plan, void* stream) {
  QLX_REQUIRE(plan != nullptr, "linear_resident: plan is NULL");
  QLX_REQUIRE(w && w_scale && x && (y || plan->mode == QLX_MODE_PLANES), "linear_resident: NULL pointer");
  QLX_REQUIRE(fmt != QLX_FMT_FP8 || x_scale, "linear_resident: FP8 W8A8 takes the token scales");
  ResidentArgs a = {};
  a.w = w;
  a.ws = w_scale;
  a.x = x;
  a.xs = x_scale;
  a.y = static_cast<uint16_t*>(y);
  switch (fmt) {
    case QLX_FMT_W4A16: return resident_w4a16(a, m, n, k, plan, stream);
    case QLX_FMT_W8A16: return resident_w8a16(a, m, n, k, plan, stream);
    case QLX_FMT_FP8: return resident_fp8(a, m, n, k, plan, stream);
    case QLX_FMT_REF8: return resident_ref8(a, m, n, k, plan, stream);
    case QLX_FMT_REF4: return resident_ref4(a, m, n, k, plan, stream);
  }
  QLX_REQUIRE(false, "linear_resident: format %d", fmt);
}

}  // extern "C"
