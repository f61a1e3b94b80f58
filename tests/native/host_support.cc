// Host-side support of the launchers (runtime_support.h, split_plan.h), driven without a GPU: the HIP calls that they make are
// the ones below.  Exits with the line of the first check that fails.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include <thread>

#include "../../tvm_amd/csrc/launch_mix.h"
#include "../../tvm_amd/csrc/runtime_support.h"
#include "../../tvm_amd/csrc/typed_kernels.h"

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

// Every item of either kind has one workgroup, eight neighbours are of one kind, and two groups of the second follow one of the
// first as long as there are both
static void two_kinds_of_items_are_dealt_out_once() {
  const int counts[] = {0, 1, 7, 8, 9, 15, 16, 17, 63, 64, 65, 129, 1000, 2047, 5003};
  for (int first : counts) {
    for (int others : counts) {
      const tvmkv::LaunchMix mix(first, others);
      std::set<int> seen[2];
      int in_front = 0;
      for (unsigned block = 0; block < mix.grid(); ++block) {
        bool is_first = false, group_is_first = false;
        const int item = mix.item(static_cast<int>(block), is_first);
        mix.item(static_cast<int>(block & ~7u), group_is_first);
        REQUIRE(is_first == group_is_first);
        if (item < 0) continue;
        REQUIRE(item < (is_first ? first : others) && item % 8 == static_cast<int>(block % 8));
        REQUIRE(seen[is_first].insert(item).second);
        if (!is_first && static_cast<int>(seen[1].size()) < first) in_front = std::max(in_front, item / 8 + 1);
      }
      REQUIRE(static_cast<int>(seen[1].size()) == first && static_cast<int>(seen[0].size()) == others);
      REQUIRE(first == 0 || in_front >= std::min((others + 7) / 8, 2 * ((first + 7) / 8 - 1)));
    }
  }
  for (int64_t bad : {int64_t{-1}, (int64_t{1} << 31) - 16}) {
    bool threw = false;
    try {
      tvmkv::LaunchMix(bad, 0);
    } catch (const tvmkv::Error&) {
      threw = true;
    }
    REQUIRE(threw);
  }
}

// The items of a split launch come in the order of its grid by itself: (kv heads, row tiles, shares), the first fastest
static void row_tiles_of_one_share_are_neighbours() {
  for (int h_kv : {1, 3, 8}) {
    for (int slots : {1, 2, 5}) {
      for (int shares : {1, 2, 64}) {
        int item = 0;
        const int items = h_kv * slots * shares;
        for (int share = 0; share < shares; ++share) {
          for (int slot = 0; slot < slots; ++slot) {
            for (int kvh = 0; kvh < h_kv; ++kvh) {
              const tvmkv::RowTileItem it(item++, items, h_kv, shares);
              REQUIRE(it.kvh == kvh && it.slot == slot && it.share == share);
            }
          }
        }
      }
    }
  }
}

// Decode steps over a shared prefix whose times were measured in one launch and in two
static void a_prefix_is_walked_beside_the_sequences_where_that_is_faster() {
  const auto one = [](int d, int hq, int h_kv, int64_t sequences, int64_t own) {
    return tvmkv::shared_prefix_in_one_launch(d, hq / h_kv, h_kv, sequences, sequences * own, 256);
  };
  for (int d : {64, 128}) {
    for (int64_t own : {32, 1500, 6000, 32000}) REQUIRE(one(d, 32, 8, 64, own) && one(d, 32, 8, 36, own));
    REQUIRE(one(d, 32, 8, 160, 300) && one(d, 32, 8, 200, 1500) && one(d, 8, 8, 200, 1500) && one(d, 32, 4, 110, 6000));
  }
  for (int64_t own : {3000, 6000, 10000}) {
    REQUIRE(!one(64, 32, 8, 110, own) && !one(64, 8, 8, 140, own) && !one(64, 64, 8, 200, own));
    REQUIRE(one(128, 32, 8, 110, own) && one(128, 8, 8, 140, own) && one(128, 64, 8, 200, own));
  }
  REQUIRE(!one(64, 32, 1, 64, 500) && !one(96, 32, 8, 64, 500) && !one(256, 32, 8, 64, 500));  // not built
}

int main() {
  a_prefix_is_walked_beside_the_sequences_where_that_is_faster();
  two_kinds_of_items_are_dealt_out_once();
  row_tiles_of_one_share_are_neighbours();
  a_buffer_is_leased_once();
  dynamic_lds_is_allowed_for_every_kernel_of_a_type();
  std::printf("all checks passed\n");
  return 0;
}
