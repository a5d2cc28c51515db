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

// Where another kernel streams a call faster, although this one serves it (us per call over distinct
// weights, the other kernel / this one, MI355X). 8-bit weights of over 64 MiB, where both are at the
// memory's rate and the other kernels' 8 waves of whole tiles read it more evenly: 151936 x 2560 FP8
// 67.7 / 74.2 at one token, 72.3 / 78.2 at 8, 68.8 / 81.6 at 16, 102.7 / 113.5 at 64; W8A16 71.3 /
// 71.5, 72.4 / 75.7, 67.8 / 81.2 (but 123.8 / 114.6 at 64). 4-bit weights of long runs at up to 4
// tokens, where the ring kernel does (gemm.h): W4A16 37.5 / 38.9 at one token, 40.4 / 42.3 at 4,
// 46.7 / 42.6 at 8. FP8 of one token: the other kernel quantizes it itself, one launch fewer.
static bool resident_yields(int fmt, int m, int n, int k) {
  const long long bytes = (long long)n * k;
  if (fmt == QLX_FMT_FP8) return m == 1 || bytes > (64ll << 20);
  if (fmt == QLX_FMT_W8A16) return m <= 32 && bytes > (64ll << 20);
  if (fmt == QLX_FMT_W4A16) return m <= 4 && n / 16 >= 2 * 8 * 256;
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
  p.splits = resident_yields(fmt, m, n, k) ? 0 : s;
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
