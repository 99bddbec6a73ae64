// Error bookkeeping shared by every entry point of libhqekv.
#include <stdarg.h>
#include <stdio.h>
#include <atomic>
#include <chrono>
#include <random>

#include "common.h"

namespace hq {

static thread_local char g_err[512] = "";

int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_launch(const char *what) {
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) return HQEKV_OK;
  snprintf(g_err, sizeof(g_err), "%s: %s", what, hipGetErrorString(e));
  return (int)e;
}

uint64_t launch_number() {
  static std::atomic<uint64_t> next{std::random_device{}() * 0x9e3779b97f4a7c15ull ^ (uint64_t)std::chrono::steady_clock::now().time_since_epoch().count()};
  return next.fetch_add(1, std::memory_order_relaxed);
}

}  // namespace hq

extern "C" int hqekv_selftest_form(int what, int64_t a, int64_t b, int64_t c) {
  const hq::PromptForm p = hq::prompt_form(a, b);
  switch (what) {
    case 0: return 10 * p.key_shares + p.tiles + (p.reversed ? 100 : 0);
    case 1: return hq::quant_rows_form(a);
    case 2: return hq::quant_k_staged(a, b, (int)c) ? 1 : 0;
    case 3: return hq::rows_sum_lanes(a, b);
    default: return hq::fail(HQEKV_E_ARG, "selftest_form: what=%d", what);
  }
}

extern "C" int hqekv_version(void) { return 1; }
extern "C" const char *hqekv_last_error(void) { return hq::g_err; }
