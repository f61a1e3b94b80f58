// What the attention launches of a step take, estimated on the host from its lengths alone.  The cache compares the
// routes that a step can take with it; only the differences between routes matter.
//
// A launch's workgroups own a row tile of one kv head and walk the keys of their sequence in tiles of 64.  It lasts as
// long as the longest walk of a workgroup that has its compute unit to itself, as all walks spread over the compute units,
// or as the K / V rows take at the streaming rate, whichever is longest; a launch whose keys are split pays for the
// shares' states and their merge.  The constants of each kernel are a fit to measured steps (1-40 sequences of 1-1500 new
// tokens on 0-100 000 cached ones, 8-64 query and 8-32 kv heads): 7-8 % off for the ragged kernel over gathered keys
// (598 steps), 9-17 % for the tuned kernels (383), 8-20 % for the generic ones (602 steps, fp16 and float32).
#ifndef TVMKV_CSRC_STEP_ESTIMATE_H_
#define TVMKV_CSRC_STEP_ESTIMATE_H_

#include <algorithm>
#include <cstdint>

namespace tvmkv {

struct LaunchCosts {
  int64_t rows;     // query rows of a workgroup
  double start;     // what a workgroup does before its first tile, in tiles
  double alone;     // us a tile, the workgroup alone on its compute unit
  double full;      // us a tile and compute unit, all units busy
  double full_row;  // and per 128 query rows of the tile
  double split;     // us that splitting the keys adds, beside the shares' traffic
  double stream;    // times of the K / V rows at 5 TB/s
};

// The tuned kernels (fp16) over pages, plain, and with RoPE inside: by head dim 64, 128, 256
inline LaunchCosts tuned_costs(int64_t d, bool rotating) {
  if (d <= 64) return rotating ? LaunchCosts{128, 3.2, 4.75, 2.75, 0.2, 16, 1} : LaunchCosts{128, 3, 1.15, 0.87, 0.2, 6, 1};
  if (d <= 128) return rotating ? LaunchCosts{128, 1.6, 6.9, 4.5, 1, 11, 1} : LaunchCosts{128, 3, 1.26, 1.3, 0.2, 4, 1};
  return rotating ? LaunchCosts{128, 1.3, 16, 18, 1.7, 26, 1} : LaunchCosts{128, 6, 3.4, 4, 0.7, 6, 1};
}
// The same under the mask of a layer's own window, which most of the tiles of such a launch cross
inline LaunchCosts tuned_window_costs(int64_t d) {
  return d <= 64 ? LaunchCosts{128, 4, 1.5, 1.2, 0.2, 6, 1} : LaunchCosts{128, 4, 1.65, 1.3, 0.2, 4, 1};
}
// The ragged kernel over gathered keys
inline LaunchCosts gathered_costs(int64_t d) {
  if (d <= 64) return {128, 6.6, 1.06, 0.72, 0, 0, 0};
  if (d <= 128) return {128, 7.4, 1.11, 1.06, 0, 0, 0};
  return {128, 6.1, 3.4, 4, 0.7, 0, 0};
}
// The generic kernels over pages; up to head dim 128 a row tile of 16 rows takes 0.6 of the time of one of 32
inline LaunchCosts generic_costs(int elem_bits, int64_t d, bool rotating, int64_t rows) {
  LaunchCosts c;
  if (elem_bits == 32) {
    c = d <= 64 ? LaunchCosts{rows, 2.2, 2.6, 1.97, 0, 6, 1.2} : d <= 128 ? LaunchCosts{rows, 2.4, 4.25, 3.5, 0, 9, 1.3} : LaunchCosts{rows, 2.8, 4.85, 5.85, 0, 9.6, 1.6};
  } else if (rotating) {
    c = d <= 64 ? LaunchCosts{rows, 3.1, 2.6, 0.84, 0, 9.6, 1.6} : d <= 128 ? LaunchCosts{rows, 2.9, 0.3, 1.77, 0, 11.5, 1.6} : LaunchCosts{rows, 2.9, 0.6, 3.5, 0, 20, 1.6};
  } else {
    c = d <= 64 ? LaunchCosts{rows, 2.7, 1.6, 0.59, 0, 5, 1.3} : d <= 128 ? LaunchCosts{rows, 3.8, 1.84, 0.84, 0, 10, 1.7} : LaunchCosts{rows, 1.6, 2.7, 1.8, 0, 0, 1.5};
  }
  if (d <= 128 && rows == 16) c.alone *= 0.6, c.full *= 0.6;
  return c;
}
// The same over the new tokens alone
inline LaunchCosts generic_own_costs(int elem_bits, int64_t d, bool rotating) {
  const int64_t rows = d <= 128 ? 32 : 16;
  if (elem_bits == 32) {
    return d <= 64 ? LaunchCosts{rows, 0, 3, 5.2, 0, 0, 0} : d <= 128 ? LaunchCosts{rows, 0, 0.1, 5.8, 0, 0, 0} : LaunchCosts{rows, 0, 0.1, 10, 0, 0, 0};
  }
  if (rotating) {
    return d <= 64 ? LaunchCosts{rows, 0, 0.1, 2.4, 0, 0, 0} : d <= 128 ? LaunchCosts{rows, 0, 2.1, 4, 0, 0, 0} : LaunchCosts{rows, 0, 4, 8, 0, 0, 0};
  }
  return d <= 64 ? LaunchCosts{rows, 0, 0.7, 1.4, 0, 0, 0} : d <= 128 ? LaunchCosts{rows, 0, 2.4, 1.73, 0, 0, 0} : LaunchCosts{rows, 0, 0.1, 2.6, 0, 0, 0};
}

class LaunchEstimate {
 public:
  // h_q / h_kv query rows a token and kv head; share_bytes: of an element of the shares' outputs
  LaunchEstimate(const LaunchCosts& costs, int64_t h_q, int64_t h_kv, int64_t d, int elem_bits, int cus, int splits = 1,
                 int share_bytes = 0)
      : costs_(costs), h_q_(h_q), h_kv_(h_kv), group_(h_q / h_kv), row_bytes_(2 * h_kv * d * elem_bits / 8), cus_(cus),
        splits_(splits), share_row_bytes_(h_q * d * share_bytes) {}

  // A sequence whose `tokens` queries attend to `cached` keys and, under the causal mask, to `own` new ones
  void Add(int64_t cached, int64_t own, int64_t tokens) {
    tokens_ += tokens;
    const int64_t keys = cached + own;
    if (keys == 0) return;
    const int64_t tiles = (tokens * group_ + costs_.rows - 1) / costs_.rows * h_kv_;
    const double mean = (static_cast<double>(cached) + own / 2.0) / 64;
    longest_ = std::max(longest_, (keys + 63) / 64);
    workgroups_ += tiles;
    work_ += tiles * mean;
    row_work_ += tokens * h_q_ / 128.0 * mean;
    bytes_ += static_cast<double>(keys) * row_bytes_;
  }

  double Us() const {
    if (longest_ == 0) return 0;
    const double walk = costs_.alone * (costs_.start + static_cast<double>((longest_ + splits_ - 1) / splits_));
    const double all = (costs_.full * (work_ + costs_.start * workgroups_ * splits_) + costs_.full_row * row_work_) / cus_;
    const double us = std::max({walk, all, costs_.stream * bytes_ / 5e6});
    return splits_ > 1 ? us + costs_.split + 2.0 * splits_ * tokens_ * share_row_bytes_ / 5e6 : us;
  }

 private:
  LaunchCosts costs_;
  int64_t h_q_, h_kv_, group_, row_bytes_;
  int cus_, splits_;
  int64_t share_row_bytes_;
  int64_t tokens_ = 0, longest_ = 0, workgroups_ = 0;
  double work_ = 0, row_work_ = 0, bytes_ = 0;
};

}  // namespace tvmkv

#endif  // TVMKV_CSRC_STEP_ESTIMATE_H_
