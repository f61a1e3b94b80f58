// Host-side support of the launchers (runtime_support.h, split_plan.h), driven without a GPU: the HIP calls that they make are
// the ones below.  Exits with the line of the first check that fails.
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <thread>

#include "../../tvm_amd/csrc/runtime_support.h"

#define REQUIRE(cond)                                        \
  do {                                                       \
    if (!(cond)) {                                           \
      std::printf("line %d: %s\n", __LINE__, #cond);         \
      std::exit(1);                                          \
    }                                                        \
  } while (0)

static std::map<const void*, int> g_lds_bytes;
static int g_calls = 0, g_fail = 0;
extern "C" hipError_t hipFuncSetAttribute(const void* func, hipFuncAttribute, int value) {
  ++g_calls;
  if (g_fail > 0) {
    --g_fail;
    return hipErrorInvalidValue;
  }
  g_lds_bytes[func] = value;
  return hipSuccess;
}
extern "C" const char* hipGetErrorString(hipError_t) { return "refused"; }
static void* volatile g_called;
static void kernel_a(int x) { g_called = &x; }
static void kernel_b(int x) { g_called = &x + 1; }

static void dynamic_lds_is_allowed_for_every_kernel_of_a_type() {
  g_fail = 1;
  bool threw = false;
  try {
    tvmkv::allow_dynamic_lds<kernel_a>(66048);
  } catch (const tvmkv::Error&) {
    threw = true;
  }
  REQUIRE(threw && g_lds_bytes.empty());
  for (int i = 0; i < 3; ++i) {  // the call that failed is made again, the others once
    tvmkv::allow_dynamic_lds<kernel_a>(66048);
    tvmkv::allow_dynamic_lds<kernel_b>(66048);
  }
  REQUIRE(g_calls == 3);
  REQUIRE(g_lds_bytes[reinterpret_cast<const void*>(kernel_a)] == 66048);
  REQUIRE(g_lds_bytes[reinterpret_cast<const void*>(kernel_b)] == 66048);
}

static void a_buffer_is_leased_once() {
  std::recursive_mutex mutex;
  bool decode = false, prefill = false;
  auto hold = [&](bool* buffer) { return tvmkv::ScratchHold(std::unique_lock<std::recursive_mutex>(mutex), buffer); };
  auto refused = [&](bool* buffer) {
    try {
      hold(buffer);
    } catch (const tvmkv::Error&) {
      return true;
    }
    return false;
  };
  auto locked_for_others = [&] {
    bool got = false;
    std::thread([&] {
      got = mutex.try_lock();
      if (got) mutex.unlock();
    }).join();
    return !got;
  };
  {
    tvmkv::ScratchHold outer = hold(&prefill);
    REQUIRE(refused(&prefill) && prefill);  // the refused one leaves the mark alone
    {
      tvmkv::ScratchHold inner = hold(&decode);  // another buffer, the same thread
      REQUIRE(decode && refused(&decode) && refused(&prefill));
    }
    REQUIRE(!decode && prefill && locked_for_others());
    tvmkv::ScratchHold moved = std::move(outer);
    REQUIRE(prefill && refused(&prefill) && locked_for_others());
    moved = {};
    REQUIRE(!prefill && !refused(&prefill) && !locked_for_others());
  }
  REQUIRE(!decode && !prefill && !locked_for_others());
}

int main() {
  a_buffer_is_leased_once();
  dynamic_lds_is_allowed_for_every_kernel_of_a_type();
  std::printf("all checks passed\n");
  return 0;
}
