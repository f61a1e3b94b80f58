// The MHA kernels behind one more argument: the storage type of q / k / v / pages / out.
//
// The reference builds every kernel for a storage dtype, a page size and a head dim
// (python/tvm/relax/frontend/nn/llm/kv_cache.py:559-736; its tests run float16 and float32 storage,
// tests/python/relax/test_runtime_builtin_paged_attention_kv_cache_cpu.py:269-276).  This library's tuned
// kernels are fp16 with pages of 16 / 32 / 64 / 128 tokens and head dims 64 / 80 / 96 / 112 / 128 / 256 (80 / 96 /
// 112 in their plain form only); everything else those factories accept -- float32 storage, any page size, any
// head dim that is a multiple of 4 (fp32) or 8 (fp16) up to 256 -- runs on the generic matrix-core kernels of
// kernels_generic.hip: float32 sums, K and V rows read straight from their pages with one page-table lookup per
// row, the sliding-window cache (length_info (3, batch)), the per-layer window mask and RoPE inside the kernel
// included.  Not built there: MLA.
//
// elem_bits is 16 or 32.  The functions return the library's error codes and leave the message in the
// thread's last-error slot, like the extern "C" launchers they stand beside; they are internal: the
// tensor-level boundary (the dtype travels in the DLTensor) and the cache object (dtype_bits) call them.
#ifndef TVMKV_CSRC_TYPED_KERNELS_H_
#define TVMKV_CSRC_TYPED_KERNELS_H_

#include <cstdint>

#include "../../include/tvmkv.h"

namespace tvmkv {

// What the tuned fp16 attention kernels are built for; anything else goes to the generic kernels.
inline bool tuned_page_size(int page_size) { return page_size == 16 || page_size == 32 || page_size == 64 || page_size == 128; }
inline bool tuned_head_dim(int d) { return d == 64 || d == 80 || d == 96 || d == 112 || d == 128 || d == 256; }

// One launcher for every MHA attention slot.  Sources: paged (pages != NULL: page_indptr, page_values,
// last_page_len (batch,), page_size) or ragged (k, v, kv_indptr).  q_indptr NULL: one query row per
// sequence (decode).  Masks: causal (query i of n sees the first kv_len - n + i + 1 keys,
// _kernel_common.py:130-135), or, with tree labels, the token-tree mask (tree_attn.py:48-65: the last
// tree_indptr[b+1] - tree_indptr[b] keys of sequence b are tree nodes, labels = (first, second) per node);
// neither: every key.
struct GenericAttention {
  int elem_bits = 16;
  const void* q = nullptr;
  const int32_t* q_indptr = nullptr;
  const void* k = nullptr;
  const void* v = nullptr;
  const int32_t* kv_indptr = nullptr;
  const void* pages = nullptr;
  const int32_t* page_indptr = nullptr;
  const int32_t* page_values = nullptr;
  const int32_t* last_page_len = nullptr;
  const int32_t* tree_indptr = nullptr;
  const int32_t* tree_labels = nullptr;
  void* out = nullptr;
  float* lse = nullptr;
  int64_t total_q = 0;
  int64_t nnz_pages = 0;
  int64_t num_pages = 0;
  int32_t batch = 0, h_q = 0, h_kv = 0, d = 0, page_size = 0;
  int32_t causal = 0;
  double sm_scale = 1.0;
  const char* what = "attention";
  // The extended form, as the tuned kernels have it.  sliding_window: last_page_len is the (3, batch) length_info of
  // a sliding-window cache (last page length, window offset, sink size; attn_utils.h:483-495), keys have logical
  // indices, the sink tokens first (_kernel_common.py:155-170); layer_window > 0 with causal on such a cache: the
  // per-layer window mask (:138-144).  rotary_mode 1: q and k are rotated inside the kernel, query token i at
  // q_rope_position[i], logical key t of sequence b at k_rope_pos_offset[b] + t (ragged with k_rope_pos_offset NULL:
  // at q_rope_position[kv_indptr[b] + t], the token-tree form, tree_attn.py:93-259), frequencies of rope_scaling
  // (NULL: the default ones).  Needs a head dim that is a multiple of 16 (fp16) or 8 (float32).
  int32_t sliding_window = 0;
  int32_t layer_window = 0;
  int64_t rotary_mode = 0;
  const int32_t* q_rope_position = nullptr;
  const int32_t* k_rope_pos_offset = nullptr;
  double rope_scale = 1.0, rope_theta = 1e4;
  const tvmkv_rope_scaling* rope_scaling = nullptr;
  // Not in the extended form:
  // rows, page_begin (paged, q_indptr NULL): sequence b's query is token rows[b] of q, q_rope_position, out and lse (NULL:
  // b), its pages start at page_values[page_begin[b]] (NULL: page_indptr[b]).  skip_single: sequences with one query
  // token are passed over; work_q / work_seqs / nnz_pages then describe the others.  merge_into: out / lse hold an
  // attention state of the rows that are computed, and this one is merged into it.
  const int32_t* rows = nullptr;
  const int32_t* page_begin = nullptr;
  int32_t skip_single = 0, merge_into = 0;
  int64_t work_q = 0, work_seqs = 0;
};
int generic_attention(const GenericAttention& args, void* stream);
// Both calls; the second merges into rows of the first.  One launch where the first has row tiles of 32 rows and the second a
// split one of 16 (generic_pair_tiles: query rows a sequence and kv head on average).
inline bool generic_pair_tiles(int d, int group, int64_t own_rows) { return d <= 128 && group <= 16 && own_rows > 16; }
int generic_attention_pair(const GenericAttention& own, const GenericAttention& decoding, void* stream);

// Slot 24 (and 24 + 13 with pages != NULL) for any even head dim up to 256 and either storage type; the
// arguments of tvmkv_fused_rope_append_scaled.
int typed_fused_rope(int elem_bits, const void* qkv, const int32_t* position_map, void* q, void* k, void* v,
                     int64_t apply_rope, const float* rope_ext_factors, const tvmkv_rope_scaling* scaling, void* pages,
                     const int32_t* append_position_map, int64_t seq_len, int32_t num_q_heads, int32_t num_kv_heads,
                     int32_t head_dim, int64_t num_pages, int32_t page_size, double rope_scale, double rope_theta,
                     void* stream);
// Slot 23 for either storage type.
int typed_merge_state_inplace(int elem_bits, void* v, float* s, const void* v_other, const float* s_other, int64_t n,
                              int32_t h, int32_t d, void* stream);

// Keys and values of a step as one run of rows per sequence (fp16): the cached tokens of sequence b in logical order
// (a sliding-window cache's sinks, then its window), then its new tokens, at rows kv_indptr[b] .. kv_indptr[b + 1] of
// k_out / v_out (rows, h_kv, d).  Keys are rotated on the way when `rotate` (rotate-half over the whole head at
// k_rope_pos_offset[b] + t for the cached ones, at q_rope_position[i] for the new ones: what the attention kernels
// do with rotary_mode 1), and q_out, when given, receives the rotated queries (total_q, h_q, d).
struct GatherKV {
  const void* pages = nullptr;
  const int32_t* page_indptr = nullptr;
  const int32_t* page_values = nullptr;
  const int32_t* length_info = nullptr;  // (batch) last page lengths, or (3, batch) with `sliding`
  const int32_t* k_rope_pos_offset = nullptr;
  const int32_t* q_indptr = nullptr;
  const int32_t* kv_indptr = nullptr;
  const int32_t* q_rope_position = nullptr;
  const void* q_new = nullptr;  // new tokens: rows of consecutive tokens are *_stride elements apart, heads d apart
  const void* k_new = nullptr;
  const void* v_new = nullptr;
  int64_t q_stride = 0, kv_stride = 0;
  void* k_out = nullptr;
  void* v_out = nullptr;
  void* q_out = nullptr;
  int64_t kv_rows = 0;  // kv_indptr[batch]
  int32_t batch = 0, h_q = 0, h_kv = 0, d = 0, page_size = 0;
  int32_t sliding = 0, rotate = 0;
  double rope_scale = 1.0, rope_theta = 1e4;
  const tvmkv_rope_scaling* rope_scaling = nullptr;
};
int gather_kv(const GatherKV& args, void* stream);

// tvmkv_batch_prefill_ragged_kv (causal, no RoPE inside) over keys that gather_kv laid out; q_token_stride != 0: the
// queries are read from the fused qkv tensor, rotated at q_rope_position with the default frequencies if apply_rope.
int prefill_over_gathered_kv(const void* q, int64_t q_token_stride, const int32_t* q_rope_position, int64_t apply_rope,
                             double rope_scale, double rope_theta, const int32_t* q_indptr, const void* k, const void* v,
                             const int32_t* kv_indptr, void* output, float* lse, double sm_scale, int32_t batch_size,
                             int64_t total_q, int32_t h_q, int32_t h_kv, int32_t d, void* stream);

// Decode attention (fp16, head dims 64 / 128 / 256, tuned page sizes) of sequences whose new token is not in the pages
// the table names: its k / v row is one more key.  rows (NULL: 0 .. batch - 1): the sequences' tokens in q, k_new,
// v_new, q_rope_position, out and lse; page_begin (NULL: page_indptr): where their pages start in page_values, with
// page_indptr[b + 1] - page_indptr[b] pages each.  rotate 1: q, the cached keys and the new one are rotated at their
// positions (default frequencies); 2: the queries alone; 0: nothing.
struct NewTokenDecode {
  const void* q = nullptr;
  const void* k_new = nullptr;
  const void* v_new = nullptr;
  int64_t q_stride = 0, new_stride = 0;  // elements between consecutive tokens
  const int32_t* rows = nullptr;
  const void* pages = nullptr;
  const int32_t* page_indptr = nullptr;
  const int32_t* page_begin = nullptr;
  const int32_t* page_values = nullptr;
  const int32_t* length_info = nullptr;  // (batch), or (3, batch) with `sliding`
  const int32_t* k_rope_pos_offset = nullptr;
  const int32_t* q_rope_position = nullptr;
  void* out = nullptr;
  float* lse = nullptr;
  int64_t rotate = 0;
  double rope_scale = 1.0, rope_theta = 1e4, sm_scale = 1.0;
  int64_t nnz_pages = 0, num_pages = 0;  // nnz_pages: page_indptr[batch]
  int32_t batch = 0, h_q = 0, h_kv = 0, d = 0, page_size = 0;
  int32_t sliding = 0;
};
struct PromptLaunch;
// beside: prompts to run in the same launch (kernels_decode.hip), or NULL
int decode_with_new_token(const NewTokenDecode& args, void* stream, const PromptLaunch* beside = nullptr);

// Prefill attention (fp16, head dims 64 / 128, tuned page sizes) of a step's sequences with more than one new token:
// cached keys, then the new ones under the causal mask.  Sequences with one new token are passed over; their rows of
// out / lse hold nothing of use afterwards.  layer_window 0: one pass over both key sets, the queries read from q with
// q_stride and rotated if apply_rope; else the per-layer window mask over the length_info (3, batch) of such a layer.
struct PromptPrefill {
  const void* q = nullptr;
  int64_t q_stride = 0;  // elements between consecutive tokens, 0: h_q * d
  const int32_t* q_rope_position = nullptr;
  int32_t apply_rope = 0;
  double rope_scale = 1.0, rope_theta = 1e4, sm_scale = 1.0;
  const int32_t* q_indptr = nullptr;
  const void* k = nullptr;
  const void* v = nullptr;
  const void* pages = nullptr;
  const int32_t* page_indptr = nullptr;
  const int32_t* page_values = nullptr;
  const int32_t* length_info = nullptr;
  int32_t layer_window = 0;
  void* out = nullptr;
  float* lse = nullptr;
  int32_t batch = 0, h_q = 0, h_kv = 0, d = 0, page_size = 0;
  int64_t total_q = 0, num_pages = 0;
  int64_t prompts = 0, prompt_tokens = 0, prompt_cached = 0;  // sequences with more than one new token: their number, new and cached tokens
};

// A step that mixes prompts and decoding sequences: both of the above, in one launch where that is built.
inline bool mixed_in_one_launch(int d, int group) { return (d == 64 || d == 128) && group <= 16; }
int attend_mixed(const PromptPrefill& prompts, const NewTokenDecode& decoding, void* stream);

// tvmkv_batch_prefill_paged_kv_scaled for a caller that knows the keys of its longest sequence (0: not known)
int prefill_paged_with_lengths(const void* q, const int32_t* q_indptr, const void* pages, const int32_t* page_indptr,
                               const int32_t* page_values, const int32_t* length_info, const int32_t* k_rope_pos_offset,
                               const int32_t* q_rope_position, void* output, float* lse, int64_t causal, int64_t rotary_mode,
                               double rope_scale, double rope_theta, double sm_scale, int32_t batch_size, int64_t total_q,
                               int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv, int32_t d, int32_t page_size,
                               int32_t sliding_window, int32_t sliding_window_size, int32_t merge_into,
                               const tvmkv_rope_scaling* rope_scaling, int64_t longest, void* stream);

// A decode step behind a shared prefix (fp16, plain cache): decode attention over the sequences' own pages, which writes
// out and lse, and paged prefill attention of all queries over the prefix, merged into them.  One launch and the merge of
// the prefix's shares where its keys are split.
struct SharedPrefixDecode {
  const void* q = nullptr;
  const void* pages = nullptr;
  void* out = nullptr;
  float* lse = nullptr;
  struct Level {
    const int32_t* page_indptr = nullptr;
    const int32_t* page_values = nullptr;
    const int32_t* length_info = nullptr;
    int32_t sequences = 0;
    int64_t nnz_pages = 0;
  } own, prefix;
  const int32_t* prefix_q_indptr = nullptr;
  int64_t longest = 0;  // keys of the longest prefix
  double sm_scale = 1.0;
  int64_t total_q = 0, num_pages = 0;
  int32_t h_q = 0, h_kv = 0, d = 0, page_size = 0;
};
int decode_with_shared_prefix(const SharedPrefixDecode& args, void* stream);  // where shared_prefix_in_one_launch
// At head dim 64 the launch of both holds three workgroups per compute unit, the decode kernel by itself five.  Where the
// sequences alone are that many items, of more than one chunk each, nothing is left to overlap with: 100-200 sequences of
// 3000-10 000 tokens behind 1100-16 000, 4-8 kv heads with 1-8 query heads each, took 0.96-1.08 times as long in two launches,
// 1.00 in the mean of 93 shapes (32 / 8 heads, 140 x 6000 behind 4096: 329 us a layer, in two 318).  Fewer or shorter ones, and
// head dim 128: 0.97-1.36, 1.07 in the mean of 387.
inline bool shared_prefix_in_one_launch(int d, int group, int h_kv, int64_t sequences, int64_t own_tokens, int cus) {
  const bool full = d == 64 && sequences * h_kv >= 3 * static_cast<int64_t>(cus) && own_tokens > 2048 * sequences;
  return mixed_in_one_launch(d, group) && !full;
}

// tvmkv_kv_cache_transpose_append with the k / v rows of consecutive tokens token_stride elements apart (the fused
// qkv tensor of the step)
int append_strided(void* pages, const void* k_data, const void* v_data, int64_t token_stride, const int32_t* position_map,
                   int64_t ntoken, int64_t num_pages, int32_t num_kv_heads, int32_t page_size, int32_t head_dim, void* stream);

// The copy kernels move rows of head_dim elements whatever they hold: float32 rows are fp16 rows of twice
// the length.
inline int32_t copy_dim(int elem_bits, int32_t head_dim) { return head_dim * (elem_bits / 16); }

}  // namespace tvmkv

#endif  // TVMKV_CSRC_TYPED_KERNELS_H_
