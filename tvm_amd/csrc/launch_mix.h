// How the workgroups of a launch with two kinds of work are dealt out.  Host and device code.
#ifndef TVMKV_CSRC_LAUNCH_MIX_H_
#define TVMKV_CSRC_LAUNCH_MIX_H_

#include <hip/hip_runtime_api.h>

#include <cstdint>

#include "common.h"

namespace tvmkv {

// Two kinds of work items in one launch, one per workgroup.  Eight neighbouring workgroups (one per XCD) are of one kind;
// kOthers such groups of the second kind follow one of the first until a kind is used up.  (The period is odd on purpose: with
// an even number of groups a kind's workgroups land on the same compute units; measured beside
// decode_beside_prefill_kernel.)
struct LaunchMix {
  static constexpr int kOthers = 2;
  int first_items, other_items;

  LaunchMix(int64_t first, int64_t others) : first_items(static_cast<int>(first)), other_items(static_cast<int>(others)) {
    KV_CHECK(first >= 0 && others >= 0 && first + others < (int64_t{1} << 31) - 16) << "too many work items for one launch";
  }
  static __host__ __device__ int groups(int items) { return (items + 7) / 8; }
  unsigned grid() const { return 8u * static_cast<unsigned>(groups(first_items) + groups(other_items)); }

  // The item of a workgroup, -1: none
  __host__ __device__ int item(int block, bool& is_first) const {
    const int eight = block >> 3;
    const int first_groups = groups(first_items), other_groups = groups(other_items);
    const int runs = first_groups < other_groups / kOthers ? first_groups : other_groups / kOthers;
    const int run = eight / (1 + kOthers);
    int before;  // groups of the first kind in front of this one
    if (run < runs) {
      is_first = eight == run * (1 + kOthers);
      before = run + (is_first ? 0 : 1);
    } else {
      const int rest = eight - runs - other_groups;  // the others that are left come first
      is_first = rest >= 0;
      before = runs + (rest > 0 ? rest : 0);
    }
    const int at = (is_first ? before : eight - before) * 8 + (block & 7);
    return at < (is_first ? first_items : other_items) ? at : -1;
  }
};

// One item of a prefill launch: kv heads next to each other, then row tiles, then shares of the keys, as in the grid of the
// launch by itself: what runs at the same time reads the same keys.
struct RowTileItem {
  int kvh, slot, share;

  __host__ __device__ RowTileItem(int item, int items, int h_kv, int shares) {
    const int tile = item / h_kv, slots = items / (h_kv * shares);
    kvh = item - tile * h_kv;
    share = tile / slots;
    slot = tile - share * slots;
  }
};

}  // namespace tvmkv

#endif  // TVMKV_CSRC_LAUNCH_MIX_H_
