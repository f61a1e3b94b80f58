// Host-side support shared by the kernel launchers: tuning options (read from the environment once,
// changeable through tvmkv_set_option) and the scratch buffers of the split-KV kernels.
#ifndef TVMKV_CSRC_RUNTIME_SUPPORT_H_
#define TVMKV_CSRC_RUNTIME_SUPPORT_H_

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <utility>

#include "common.h"

struct tvmkv_rope_scaling;  // include/tvmkv.h

namespace tvmkv {

enum Option {
  kOptDecodeChunkPages = 0,   // pages per split-KV chunk of the decode kernel, 0 = derived from the shapes
  kOptDecodeSeparateMerge,    // != 0: merge the chunks in a second launch instead of inside the kernel
  kOptDecodeWgsPerCu,         // > 0: cap the decode grid at this many workgroups per compute unit
  kOptMlaChunkTokens,         // lower bound of the tokens per split-KV chunk of the MLA kernel, 0 = 128
  kOptMlaSeparateMerge,       // unused (the MLA chunks are always merged in a second launch)
  kOptPrefillKvSplits,        // > 0: split the keys of every row tile of a paged prefill launch this many ways, 0 = derived
  kOptNoFusedDecodeStep,      // != 0: the cache object runs a decode step as split+RoPE+append and decode, two launches
  kOptStepRoute,              // > 0: the route of the cache object's steps instead of the one that the estimate prefers, where a
                              // step can take it: 1 the general launches, 2 prompts and decoding sequences apart, 3 gathered keys
  kNumOptions
};
bool stream_is_capturing(hipStream_t stream);
int64_t option(Option id);

// Scratch memory of a split-KV launch.  A buffer belongs to one (device, stream, user): launches on
// one stream are ordered and may share it, launches on different streams (two caches, two layers in
// flight) never do.  The first `counter_bytes` bytes hold arrival counters that are not reset between
// launches: every launch gets a new `epoch`, a counter is a 64-bit word (epoch << 32 | arrivals), and a
// word left behind by an earlier launch -- also one that failed or was abandoned half way -- carries an
// older epoch and counts as zero.  The epoch is the low half of a 64-bit launch count; when it wraps
// (2^32 launches on one buffer) the counters are cleared by a kernel in stream order and the epochs
// start over at 1.
// The lease keeps the pool locked until it is destroyed: hold it until the launch that uses the buffer
// has been enqueued, so that a second host thread on the same stream cannot free the buffer in between.
// The lock lets the same thread in again, as one launch may use the buffers of two users; a second lease
// of the same buffer meanwhile, which would share it or free it, is refused.
class ScratchHold {
 public:
  ScratchHold() = default;
  // held: the mark of the buffer, which the lock guards
  ScratchHold(std::unique_lock<std::recursive_mutex> lock, bool* held) : lock_(std::move(lock)) {
    KV_CHECK(!*held) << "scratch memory is leased while a launch that uses it is being prepared";
    *held = true;
    held_ = held;
  }
  ScratchHold(ScratchHold&& other) noexcept { *this = std::move(other); }
  ScratchHold& operator=(ScratchHold&& other) noexcept {
    if (this != &other) {
      Release();
      lock_ = std::move(other.lock_);
      held_ = std::exchange(other.held_, nullptr);
    }
    return *this;
  }
  ~ScratchHold() { Release(); }

 private:
  void Release() {
    if (held_ != nullptr) *std::exchange(held_, nullptr) = false;  // in front of the unlock
    if (lock_.owns_lock()) lock_.unlock();
  }
  std::unique_lock<std::recursive_mutex> lock_;
  bool* held_ = nullptr;
};
struct ScratchLease {
  char* ptr;        // device memory, at least the requested size, 256-byte aligned
  uint32_t epoch;   // never 0
  ScratchHold hold;
};
enum ScratchUser { kScratchDecode = 0, kScratchMla = 1, kScratchPrefill = 2, kScratchGeneric = 3 };
// at_least: what a buffer that has to be allocated gets in any case
ScratchLease lease_scratch(ScratchUser user, hipStream_t stream, size_t bytes, size_t counter_bytes, size_t at_least = 0);
// Frees the buffers of (current device, stream) after synchronising the stream; a buffer whose address
// a graph under capture has recorded is kept until the process ends instead.
void release_scratch(hipStream_t stream);
// The epoch of the next launch from a 64-bit launch count (host arithmetic only).
uint32_t next_scratch_epoch(uint64_t* launches, bool* wrapped);
void zero_scratch_counters(char* ptr, size_t counter_bytes, hipStream_t stream);
// Test aid: launches of two kinds of work (launch_mix.h) since the process began
void count_joint_launch();
// Test aid: sets the launch count of every pooled buffer (to run a launch across the epoch wrap).
void debug_set_scratch_launches(uint64_t launches);

// A kernel that is launched with more dynamic shared memory than every function may have by itself (48 KB): said once per
// kernel, which is a template argument so that kernels of one type do not share the flag, and again after a call that failed.
// (The attribute is the function's, not the device's.)
template <auto kKernel>
void allow_dynamic_lds(size_t bytes) {
  static std::atomic<bool> said{false};
  if (said.load(std::memory_order_acquire)) return;
  HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kKernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)));
  said.store(true, std::memory_order_release);
}

// The table of an attention kernel's in-kernel RoPE for a frequency variant (NULL: the default
// frequencies): entries for all head_dim elements, see InlineRopeTable in kernels_common.cuh.  Host
// arithmetic only (defined next to the split-rotary kernel's tables in kernels_page.hip).
struct InlineRopeHost {
  float v[256];
  int inverse;
  int halves_differ;
  float magnitude;
};
InlineRopeHost inline_rope_table(const ::tvmkv_rope_scaling* scaling, int head_dim, double rope_theta);

// Chunk-slot arithmetic of the decode split, on the host (the device functions of the same names in
// kernels_decode.hip compute the same values; the tests compare both against a direct enumeration).
int decode_pick_chunk_pages(int64_t nnz_pages, int h_kv, int batch, int head_dim = 128);
// the same for launches whose work items carry 32 query heads (GQA groups above 16)
int decode_pick_chunk_pages_wide(int64_t nnz_pages, int h_kv, int batch, int head_blocks, int resident_items);

// Shares of the keys of a paged prefill launch (work_q query tokens in work_seqs sequences of avg_keys keys on average,
// group query heads per kv head) on a device of `cus` compute units, and the workgroups that it has unsplit.
constexpr int64_t kMinShareKeys = 512;  // eight tiles of 64 keys
int64_t prefill_workgroups(int64_t work_q, int group, int64_t work_seqs, int h_kv);
int prefill_kv_splits(int64_t work_q, int group, int64_t work_seqs, int h_kv, int64_t avg_keys, int cus);
// The same of a launch of the generic kernel, whose workgroups own generic_row_tile() query rows.
inline int generic_row_tile(int d, int64_t rows_per_sequence) { return d > 128 || rows_per_sequence <= 16 ? 16 : 32; }
int generic_kv_splits(int elem_bits, int d, int64_t work_q, int group, int64_t work_seqs, int h_kv, int64_t avg_keys, int cus);

}  // namespace tvmkv

#endif  // TVMKV_CSRC_RUNTIME_SUPPORT_H_
