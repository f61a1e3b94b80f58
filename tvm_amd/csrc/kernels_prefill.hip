// Ragged and paged causal prefill attention on fp16 MFMA tiles for gfx950.
//
// Replaces batch_prefill_ragged_kv and batch_prefill_paged_kv
// (python/tvm/relax/frontend/nn/llm/_prefill_kernels.py:795-923, :217-391), whose inner
// products are scalar FMAs over 32x32 tiles on a fixed grid of 16 x h_kv blocks.  Numerics
// follow the reference macros (python/tvm/relax/frontend/nn/llm/_kernel_common.py:222-334):
// S = QK^T * sm_scale * log2(e), base-2 online softmax with initial state m = -5e4, d = 1,
// fp32 accumulation, out = O/d rounded once to fp16, lse = m + log2(d); rows are the
// (position, head-in-group) pairs of one kv head, interleaved as row = pos*group + head
// (_prefill_kernels.py:331-332); causal mask col < kv_len - qo_len + row_pos + 1
// (_kernel_common.py:130-135).
//
// Tiling: a workgroup of 4 wavefronts owns 128 rows x one kv head; each wave owns 32 rows, one
// row per lane%32, and keeps Q as MFMA B-fragments in registers.  K/V tiles of 64 tokens are
// copied from global memory straight into LDS (global_load_lds_dwordx4: no staging registers, no
// ds_write), row-major and unpadded, two stages deep, so that tile t+1 lands while tile t is
// multiplied.  Bank conflicts are avoided by an XOR swizzle of the 16-byte pieces of a row; the
// copy applies it on the source side (lane L always fills LDS piece L of the 1 KiB an
// instruction writes, and fetches the global piece that belongs there).  S^T = K Q^T and
// O^T = V^T P^T use v_mfma_f32_32x32x16_f16 with the query on the N axis: all per-query softmax
// state (m, l, the O rescale factor) is lane-local, and the S^T accumulator registers are exactly
// the B-operand of the PV product, so P never leaves registers.  The V^T A-fragments come from
// the row-major V tile through ds_read_b64_tr_b16, which hands each lane four consecutive tokens
// of one feature.
//
// Workgroup -> (sequence, row tile) without a prologue kernel: sequence b owns tile slots
//   [floor(q_indptr[b]*group/128) + b, floor(q_indptr[b+1]*group/128) + b + 1)
// found by binary search on q_indptr; the grid is floor(total_q*group/128) + B slots.
#include <cmath>
#include <type_traits>

#include "prefill_kernel.cuh"
#include "runtime_support.h"
#include "typed_kernels.h"

namespace tvmkv {

// Page sizes the paged kernels take: 16 << shift tokens, walked as 1 << shift runs of 16.  -1: not built.
static int paged_page_shift(int32_t page_size) {
  if (page_size < 16 || page_size > 128 || (page_size & (page_size - 1)) != 0) return -1;
  int shift = 0;
  while ((16 << shift) < page_size) ++shift;
  return shift;
}

static int64_t row_tile_slots(const PrefillParams& p, int64_t total_q) {
  const int64_t slots = total_q * p.group / BM + p.batch_size;
  if (slots >= 65536) throw Error(TVMKV_EINVAL, "prefill: too many row tiles for one launch");
  return slots;
}

template <int DQK, int DV, int SRC, int PS, bool EXT, bool STREAM = false, bool PAD = false, bool VARIANT = false>
static void launch_prefill_ext(const PrefillParams& p, int64_t total_q, const PrefillRopeDivisors& div,
                               hipStream_t stream) {
  const int64_t slots = row_tile_slots(p, total_q);
  constexpr size_t lds_bytes = prefill_lds_bytes(DQK, DV);
  if constexpr (lds_bytes > 48 * 1024) allow_dynamic_lds<prefill_kernel<DQK, DV, SRC, PS, EXT, STREAM, PAD, VARIANT>>(lds_bytes);
  hipLaunchKernelGGL((prefill_kernel<DQK, DV, SRC, PS, EXT, STREAM, PAD, VARIANT>),
                     dim3(p.h_kv, static_cast<unsigned>(slots), static_cast<unsigned>(std::max(1, p.kv_splits))),
                     dim3(NW * 64), lds_bytes, stream, p, div);
}

// ---- split over the keys ---------------------------------------------------------------------
// A launch with few row tiles and long key ranges (a token tree or a short chunk against long cached
// sequences) neither fills the chip nor balances it: a row tile is one workgroup that walks all its
// keys.  Such a launch is split: kv_splits workgroups share a row tile, each writes the attention state
// of its share of the key tiles (normalised output, lse) to scratch memory, and a second kernel
// merges the states of a row with the arithmetic of merge_state_inplace
// (python/tvm/relax/frontend/nn/llm/_decode_kernels.py:441-450) over kv_splits states at once.  A row
// whose states are all empty (lse = -5e4) stays the empty state: out 0, lse -5e4.
// T: the type of the shares' outputs, half_t or float (KvSplit).
template <typename T, int DV>
__global__ __launch_bounds__(256) void prefill_split_merge_kernel(const T* __restrict__ part_o,
                                                                  const float* __restrict__ part_lse, half_t* __restrict__ output,
                                                                  float* __restrict__ lse, int64_t rows, int splits,
                                                                  int merge_into) {
  constexpr int TPR = DV / 8;  // threads per row, 8 features each
  const int64_t row = static_cast<int64_t>(blockIdx.x) * (256 / TPR) + threadIdx.x / TPR;
  const int piece = threadIdx.x % TPR;
  if (row >= rows) return;
  // the shares' loads do not depend on each other: unrolled, eight are in flight at once (64 shares of a
  // 64-token chunk: 35 us as a loop of dependent round trips)
  float s_max = kNegInit;
#pragma unroll 8
  for (int i = 0; i < splits; ++i) s_max = fmaxf(s_max, part_lse[i * rows + row]);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float w_sum = 0.f;
  const bool any_share = s_max > kNegInit;
  if (merge_into) {
    // output / lse already hold a state of the same rows (the launch was asked to merge into it): it is one more
    // state of the sum; shares that are all empty count as the one empty state (out 0, lse -5e4) an unsplit
    // launch would have merged
    const float s_prev = lse[row];
    s_max = fmaxf(s_max, s_prev);
    const float w = fast_exp2(s_prev - s_max);
    const Vec16 v = ld16(output + row * DV + piece * 8);
    w_sum = w + (any_share ? 0.f : fast_exp2(kNegInit - s_max));
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = w * static_cast<float>(v.h8[e]);
  }
  if (any_share) {
#pragma unroll 8
    for (int i = 0; i < splits; ++i) {
      const float w = fast_exp2(part_lse[i * rows + row] - s_max);
      typedef T share_t __attribute__((ext_vector_type(8)));
      const share_t v = *reinterpret_cast<const share_t*>(part_o + (i * rows + row) * DV + piece * 8);
      w_sum += w;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += w * static_cast<float>(v[e]);
    }
  }
  const float inv = w_sum > 0.f ? 1.0f / w_sum : 0.f;
  Vec16 out;
#pragma unroll
  for (int e = 0; e < 8; ++e) out.h8[e] = static_cast<half_t>(acc[e] * inv);
  *reinterpret_cast<Vec16*>(output + row * DV + piece * 8) = out;
  if (piece == 0) lse[row] = w_sum > 0.f ? s_max + fast_log2(w_sum) : kNegInit;
}

// Redirects the launch described by p to scratch memory when it is to be split (prefill_kv_splits); finish() merges.
// The shares' outputs are fp16 where the launch has always been split, and float32 where it would otherwise run whole:
//  * float_shares: the prompts of a step whose decoding sequences run elsewhere (prefill_prompts);
//  * longest, the keys of the longest sequence where the caller knows them, else 0: one round of full row tiles lasts as
//    long as its longest walk, so two shares each where that is well above the mean.  How much it has to be above is what
//    the shares' traffic costs, and how many workgroups share a compute unit (one that ends early leaves its unit to the
//    others): 1.4 times the mean and 1024 keys more at head dim 64, 1.75 times and 2048 more at 128, and at 256, one
//    workgroup per unit in two rounds, none.  Measured, time whole / time in two shares, 260-512 workgroups, lengths
//    around means of 1500-8000 keys evenly spread or one long among equal ones, longest / mean 1.3 | 1.4 | 1.6 | 1.8 | 2.0:
//      64    0.87-1.10 | 0.91-1.18 | 0.96-1.24 | 1.06-1.30 | 1.20-1.34       256 (1.1-1.9)    0.84-0.94
//      128   0.82-1.06 | 0.81-1.10 | 0.84-1.16 | 0.85-1.23 | 1.00-1.34, from 2048 keys above the mean on 0.97-1.34 at 1.75-2.0
struct KvSplit {
  half_t* output;
  float* lse;
  int64_t rows;
  int splits;
  int merge_into = 0;
  ScratchLease lease{};
  // work_q, work_seqs: the query tokens and sequences that the launch works on, where they are not all (skip_single)
  KvSplit(PrefillParams& p, int64_t total_q, int64_t avg_keys, int dv, hipStream_t stream, int64_t longest = 0, int64_t work_q = 0,
          int64_t work_seqs = 0, bool float_shares = false)
      : output(p.output), lse(p.lse), rows(total_q * p.h_q), splits(1) {
    if (work_seqs == 0) work_q = total_q, work_seqs = p.batch_size;
    // at most one row tile per (sequence, kv head) on average: the paged kernels stream the K/V rows
    p.stream_kv = work_q * p.group <= work_seqs * BM;
    splits = prefill_kv_splits(work_q, p.group, work_seqs, p.h_kv, avg_keys, compute_units());
    const bool unlike = dv == 64 ? longest * 10 >= avg_keys * 14 && longest - avg_keys >= 1024
                                 : dv == 128 && longest * 4 >= avg_keys * 7 && longest - avg_keys >= 2048;
    if (splits == 1 && unlike && avg_keys >= 2 * kMinShareKeys && option(kOptPrefillKvSplits) == 0 &&
        prefill_workgroups(work_q, p.group, work_seqs, p.h_kv) <= 2 * static_cast<int64_t>(compute_units())) {
      splits = 2;
      float_shares = true;
    }
    if (dv % 64 != 0) splits = 1;  // padded head dims (80, 96, 112): the merge kernel is not built for their rows
    if (splits <= 1) return;
    const size_t o_bytes = static_cast<size_t>(splits) * rows * dv * (float_shares ? sizeof(float) : sizeof(half_t));
    const size_t lse_bytes = static_cast<size_t>(splits) * rows * sizeof(float);
    lease = lease_scratch(kScratchPrefill, stream, o_bytes + lse_bytes, 0);  // held until the merge is enqueued
    char* ws = lease.ptr;
    p.output = reinterpret_cast<half_t*>(ws);
    p.lse = reinterpret_cast<float*>(ws + o_bytes);
    p.kv_splits = splits;
    p.split_rows = rows;
    p.split_f32 = float_shares;
    merge_into = p.merge_into;  // the shares write plain states; the merge kernel folds the caller's state in
    p.merge_into = 0;
  }
  void finish(const PrefillParams& p, int dv, hipStream_t stream) const {
    if (splits <= 1) return;
    KV_LAUNCH_CHECK();
    const unsigned rows_per_block = 256 / (dv / 8);
    const dim3 grid(static_cast<unsigned>((rows + rows_per_block - 1) / rows_per_block));
    auto merge = [&](auto kernel, const auto* shares) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, shares, p.lse, output, lse, rows, splits, merge_into);
    };
    auto merge_dim = [&](auto dim) {
      constexpr int kD = decltype(dim)::value;
      if (p.split_f32) {
        merge(prefill_split_merge_kernel<float, kD>, reinterpret_cast<const float*>(p.output));
      } else {
        merge(prefill_split_merge_kernel<half_t, kD>, static_cast<const half_t*>(p.output));
      }
    };
    if (dv == 128) {
      merge_dim(std::integral_constant<int, 128>{});
    } else if (dv == 64) {
      merge_dim(std::integral_constant<int, 64>{});
    } else {
      merge_dim(std::integral_constant<int, 256>{});
    }
  }
};

// The extended kernels (sliding-window cache, per-layer window, inline RoPE) exist for the head
// dims that RoPE models use here; d_qk 192 / d_v 128 is the MLA self-attention, which has neither.
// scaling: the frequency variant of the in-kernel RoPE (NULL: default); used when the launch rotates at all
template <int DQK, int DV, int SRC, int PS>
static void launch_prefill(const PrefillParams& params, int64_t total_q, bool ext, double rope_theta, hipStream_t stream,
                           const tvmkv_rope_scaling* scaling = nullptr) {
  PrefillRopeDivisors div{};
  PrefillParams p = params;
  p.rope_magnitude = 1.0f;
  auto fill_table = [&]() {
    if constexpr (DQK <= 256) {
      const InlineRopeHost table = inline_rope_table(scaling, DQK, rope_theta);
      for (int i = 0; i < DQK; ++i) div.v[i] = table.v[i];
      p.rope_inverse = table.inverse;
      p.rope_halves_differ = table.halves_differ;
      p.rope_magnitude = table.magnitude;
    }
  };
  if (!ext) {
    if (p.q_inline_rope) fill_table();
    if constexpr (SRC == kPaged) {
      if (p.stream_kv) {
        launch_prefill_ext<DQK, DV, SRC, PS, false, true>(p, total_q, div, stream);
        return;
      }
    }
    launch_prefill_ext<DQK, DV, SRC, PS, false>(p, total_q, div, stream);
    return;
  }
  if constexpr (DQK == DV && SRC != kBoth) {
    if (p.rotary) fill_table();
    // the default frequencies (one divisor per pair, position / divisor) have the kernel without the general rotation
    const bool variant = p.rotary && (p.rope_inverse != 0 || p.rope_halves_differ != 0 || p.rope_magnitude != 1.0f);
    if constexpr (SRC == kPaged) {
      if (p.stream_kv) {
        if (variant) {
          launch_prefill_ext<DQK, DV, SRC, PS, true, true, false, true>(p, total_q, div, stream);
        } else {
          launch_prefill_ext<DQK, DV, SRC, PS, true, true>(p, total_q, div, stream);
        }
        return;
      }
    }
    if (variant) {
      launch_prefill_ext<DQK, DV, SRC, PS, true, false, false, true>(p, total_q, div, stream);
    } else {
      launch_prefill_ext<DQK, DV, SRC, PS, true>(p, total_q, div, stream);
    }
  } else {
    throw Error(TVMKV_EUNSUPPORTED, "prefill: inline RoPE / sliding window are not built for this head shape");
  }
}

// Head dims 80, 96 and 112: the head dim 128 kernel on rows of d elements (plain cache, no in-kernel RoPE)
static bool padded_head_dim(int d) { return d == 80 || d == 96 || d == 112; }

template <int SRC>
static void launch_prefill_padded(PrefillParams p, int64_t total_q, int d, bool ext, const char* what, hipStream_t stream) {
  if (ext) {
    throw Error(TVMKV_EUNSUPPORTED, std::string(what) + ": head_dim " + std::to_string(d) +
                                        " is built for the plain cache only (no sliding window, inline RoPE or token tree)");
  }
  p.d_mem = d;
  launch_prefill_ext<128, 128, SRC, 16, false, false, true>(p, total_q, PrefillRopeDivisors{}, stream);
}

}  // namespace tvmkv

using namespace tvmkv;

int tvmkv::prefill_over_gathered_kv(const void* q, int64_t q_token_stride, const int32_t* q_rope_position, int64_t apply_rope,
                                    double rope_scale, double rope_theta, const int32_t* q_indptr, const void* k, const void* v,
                                    const int32_t* kv_indptr, void* output, float* lse, double sm_scale, int32_t batch_size,
                                    int64_t total_q, int32_t h_q, int32_t h_kv, int32_t d, void* stream) {
  KV_API_BEGIN();
  KV_CHECK(batch_size > 0 && total_q > 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0) << "prefill_over_gathered_kv: bad shape";
  KV_CHECK(q && q_indptr && k && v && kv_indptr && output && lse) << "prefill_over_gathered_kv: NULL tensor";
  KV_CHECK(!apply_rope || (q_rope_position && (d == 64 || d == 128))) << "prefill_over_gathered_kv: rotation of the queries";
  PrefillParams p{};
  p.q = static_cast<const half_t*>(q);
  p.q_token_stride = q_token_stride;
  p.q_inline_rope = apply_rope != 0;
  p.q_rope_position = q_rope_position;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_indptr = q_indptr;
  p.k = static_cast<const half_t*>(k);
  p.v = static_cast<const half_t*>(v);
  p.kv_indptr = kv_indptr;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = 1;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  hipStream_t s = as_stream(stream);
  if (d == 128) {
    launch_prefill<128, 128, kRagged, 16>(p, total_q, false, rope_theta, s);
  } else if (d == 64) {
    launch_prefill<64, 64, kRagged, 16>(p, total_q, false, rope_theta, s);
  } else if (d == 256) {
    launch_prefill<256, 256, kRagged, 16>(p, total_q, false, rope_theta, s);
  } else {
    KV_UNSUPPORTED(!padded_head_dim(d)) << "prefill_over_gathered_kv: head_dim " << d;
    launch_prefill_padded<kRagged>(p, total_q, d, false, "prefill_over_gathered_kv", s);
  }
  KV_LAUNCH_CHECK();
  KV_API_END();
}

int tvmkv::prefill_prompts(const PromptPrefill& a, PromptLaunch* leave, void* stream) {
  KV_API_BEGIN();
  KV_CHECK(a.batch > 0 && a.total_q > 0 && a.prompts > 0 && a.h_q > 0 && a.h_kv > 0 && a.h_q % a.h_kv == 0) << "prefill_prompts: bad shape";
  const int page_shift = paged_page_shift(a.page_size);
  KV_UNSUPPORTED(page_shift < 0) << "prefill_prompts: page_size " << a.page_size << " is not built (16, 32, 64, 128)";
  KV_CHECK(a.num_pages < (int64_t{1} << 28)) << "prefill_prompts: page ids must stay below 2^28";
  KV_CHECK(a.q && a.q_indptr && a.k && a.v && a.pages && a.page_indptr && a.page_values && a.length_info && a.out && a.lse)
      << "prefill_prompts: NULL tensor";
  KV_CHECK(!a.apply_rope || (a.q_rope_position && a.layer_window == 0)) << "prefill_prompts: rotation of the queries";
  PrefillParams p{};
  p.skip_single = 1;
  p.page_shift = page_shift;
  p.q = static_cast<const half_t*>(a.q);
  p.q_token_stride = a.q_stride;
  p.q_inline_rope = a.apply_rope != 0;
  p.q_rope_position = a.q_rope_position;
  p.rope_scale = static_cast<float>(a.rope_scale);
  p.q_indptr = a.q_indptr;
  p.k = static_cast<const half_t*>(a.k);
  p.v = static_cast<const half_t*>(a.v);
  p.kv_indptr = a.q_indptr;
  p.pages = static_cast<const half_t*>(a.pages);
  p.page_indptr = a.page_indptr;
  p.page_values = a.page_values;
  p.last_page_len = a.length_info;
  p.output = static_cast<half_t*>(a.out);
  p.lse = a.lse;
  p.batch_size = a.batch;
  p.h_q = a.h_q;
  p.h_kv = a.h_kv;
  p.group = a.h_q / a.h_kv;
  p.causal = 1;
  p.scale_log2 = static_cast<float>(a.sm_scale) * kLog2e;
  hipStream_t s = as_stream(stream);
  auto by_dim = [&](auto run) {
    KV_UNSUPPORTED(a.d != 64 && a.d != 128) << "prefill_prompts: head_dim " << a.d << " is not built (64, 128)";
    if (a.d == 128) {
      run(std::integral_constant<int, 128>{});
    } else {
      run(std::integral_constant<int, 64>{});
    }
    KV_LAUNCH_CHECK();
  };
  // Left to the caller: a launch that writes the prompts' rows and nothing else (the merge of a split one writes every
  // sequence's; the cached keys behind a window are a second launch, which needs this one's rows)
  auto leave_out = [&](int src) {
    leave->p = p;
    leave->slots = row_tile_slots(p, a.total_q);
    leave->src = src;
  };
  if (a.layer_window == 0) {
    const KvSplit split(p, a.total_q, (a.prompt_cached + a.prompt_tokens) / a.prompts, a.d, s, 0, a.prompt_tokens, a.prompts, true);
    if (leave != nullptr && split.splits == 1) {
      leave_out(kBoth);
      return TVMKV_OK;
    }
    by_dim([&](auto d) { launch_prefill<d.value, d.value, kBoth, 16>(p, a.total_q, false, a.rope_theta, s); });
    split.finish(p, a.d, s);
  } else if (leave != nullptr && a.prompt_cached == 0) {
    leave_out(kRagged);
  } else {
    by_dim([&](auto d) { launch_prefill<d.value, d.value, kRagged, 16>(p, a.total_q, false, a.rope_theta, s); });
    if (a.prompt_cached > 0) {
      p.window_offset = a.length_info + a.batch;
      p.sink_size = a.length_info + 2 * static_cast<int64_t>(a.batch);
      p.layer_window = a.layer_window;
      p.merge_into = 1;
      const KvSplit split(p, a.total_q, std::min<int64_t>(a.prompt_cached / a.prompts, a.layer_window), a.d, s, 0, a.prompt_tokens,
                          a.prompts, true);
      by_dim([&](auto d) { launch_prefill<d.value, d.value, kPaged, 16>(p, a.total_q, true, a.rope_theta, s); });
      split.finish(p, a.d, s);
    }
  }
  KV_LAUNCH_CHECK();
  KV_API_END();
}

extern "C" {

static int ragged_prefill(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                          const int32_t* kv_indptr, const int32_t* q_rope_position,
                          const int32_t* k_rope_pos_offset, void* output, float* lse, int64_t causal,
                          int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                          int32_t batch_size, int64_t total_q, int32_t h_q, int32_t h_kv, int32_t d_qk,
                          int32_t d_v, const tvmkv_rope_scaling* scaling, void* stream) {
  // head dims the tuned kernel is not built for (80 / 96 / 112 with RoPE inside the kernel among them): the generic
  // matrix-core kernel
  if (d_qk == d_v && !(rotary_mode == 0 ? tuned_head_dim(d_qk) : (d_qk == 64 || d_qk == 128 || d_qk == 256))) {
    GenericAttention a;
    a.what = "batch_prefill_ragged_kv";
    a.rotary_mode = rotary_mode;
    a.q_rope_position = q_rope_position;
    a.k_rope_pos_offset = k_rope_pos_offset;
    a.rope_scale = rope_scale;
    a.rope_theta = rope_theta;
    a.rope_scaling = scaling;
    a.q = q;
    a.q_indptr = q_indptr;
    a.k = k;
    a.v = v;
    a.kv_indptr = kv_indptr;
    a.out = output;
    a.lse = lse;
    a.total_q = total_q;
    a.batch = batch_size;
    a.h_q = h_q;
    a.h_kv = h_kv;
    a.d = d_qk;
    a.causal = causal > 0;
    a.sm_scale = sm_scale;
    return generic_attention(a, stream);
  }
  KV_API_BEGIN();
  KV_CHECK(batch_size >= 0 && total_q >= 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0)
      << "batch_prefill_ragged_kv: bad shape";
  if (batch_size == 0 || total_q == 0) return TVMKV_OK;
  KV_CHECK(q && q_indptr && k && v && kv_indptr && output && lse) << "batch_prefill_ragged_kv: NULL tensor";
  KV_CHECK(rotary_mode == 0 || (q_rope_position && k_rope_pos_offset))
      << "batch_prefill_ragged_kv: inline RoPE needs the position arrays";
  PrefillParams p{};
  p.q = static_cast<const half_t*>(q);
  p.q_indptr = q_indptr;
  p.k = static_cast<const half_t*>(k);
  p.v = static_cast<const half_t*>(v);
  p.kv_indptr = kv_indptr;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = causal > 0;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  p.rotary = rotary_mode != 0;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_rope_position = q_rope_position;
  p.k_rope_pos_offset = k_rope_pos_offset;
  const bool ext = p.rotary != 0;
  hipStream_t s = as_stream(stream);
  if (d_qk == 128 && d_v == 128) {
    launch_prefill<128, 128, kRagged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (d_qk == 64 && d_v == 64) {
    launch_prefill<64, 64, kRagged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (d_qk == 256 && d_v == 256) {
    launch_prefill<256, 256, kRagged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (d_qk == 192 && d_v == 128) {
    launch_prefill<192, 128, kRagged, 16>(p, total_q, ext, rope_theta, s);
  } else if (d_qk == d_v && padded_head_dim(d_qk)) {
    launch_prefill_padded<kRagged>(p, total_q, d_qk, ext, "batch_prefill_ragged_kv", s);
  } else {
    KV_UNSUPPORTED(true) << "batch_prefill_ragged_kv: (d_qk, d_v) = (" << d_qk << ", " << d_v
                         << ") is not built ((64,64), (80,80), (96,96), (112,112), (128,128), (192,128), (256,256))";
  }
  KV_LAUNCH_CHECK();
  KV_API_END();
}

int tvmkv_batch_prefill_ragged_kv(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                                  const int32_t* kv_indptr, const int32_t* q_rope_position,
                                  const int32_t* k_rope_pos_offset, void* output, float* lse, int64_t causal,
                                  int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                                  int32_t batch_size, int64_t total_q, int32_t h_q, int32_t h_kv, int32_t d_qk,
                                  int32_t d_v, void* stream) {
  return ragged_prefill(q, q_indptr, k, v, kv_indptr, q_rope_position, k_rope_pos_offset, output, lse, causal, rotary_mode,
                        rope_scale, rope_theta, sm_scale, batch_size, total_q, h_q, h_kv, d_qk, d_v, nullptr, stream);
}

int tvmkv_batch_prefill_ragged_kv_scaled(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                                         const int32_t* kv_indptr, const int32_t* q_rope_position,
                                         const int32_t* k_rope_pos_offset, void* output, float* lse, int64_t causal,
                                         int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                                         int32_t batch_size, int64_t total_q, int32_t h_q, int32_t h_kv, int32_t d_qk,
                                         int32_t d_v, const tvmkv_rope_scaling* rope_scaling, void* stream) {
  return ragged_prefill(q, q_indptr, k, v, kv_indptr, q_rope_position, k_rope_pos_offset, output, lse, causal, rotary_mode,
                        rope_scale, rope_theta, sm_scale, batch_size, total_q, h_q, h_kv, d_qk, d_v, rope_scaling, stream);
}

static int paged_prefill(const void* q, const int32_t* q_indptr, const void* pages, const int32_t* page_indptr,
                         const int32_t* page_values, const int32_t* length_info, const int32_t* k_rope_pos_offset,
                         const int32_t* q_rope_position, void* output, float* lse, int64_t causal,
                         int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                         int32_t batch_size, int64_t total_q, int64_t nnz_pages, int64_t num_pages, int32_t h_q,
                         int32_t h_kv, int32_t d, int32_t page_size, int32_t sliding_window,
                         int32_t sliding_window_size, bool merge_into, void* stream,
                         const tvmkv_rope_scaling* scaling = nullptr, int64_t longest = 0,
                         const std::function<int(const PromptLaunch*)>* beside = nullptr) {
  // pages other than 16 / 32 / 64 / 128 tokens, other head dims (80 / 96 / 112 with a sliding-window cache or RoPE
  // inside the kernel among them): the generic matrix-core kernel (its caller merges states with merge_state_inplace)
  const bool plain = rotary_mode == 0 && sliding_window == 0;
  if (!merge_into && (!tuned_page_size(page_size) || !(plain ? tuned_head_dim(d) : (d == 64 || d == 128 || d == 256)))) {
    GenericAttention a;
    a.what = "batch_prefill_paged_kv";
    a.sliding_window = sliding_window;
    a.layer_window = sliding_window_size;
    a.rotary_mode = rotary_mode;
    a.q_rope_position = q_rope_position;
    a.k_rope_pos_offset = k_rope_pos_offset;
    a.rope_scale = rope_scale;
    a.rope_theta = rope_theta;
    a.rope_scaling = scaling;
    a.q = q;
    a.q_indptr = q_indptr;
    a.pages = pages;
    a.page_indptr = page_indptr;
    a.page_values = page_values;
    a.last_page_len = length_info;
    a.out = output;
    a.lse = lse;
    a.total_q = total_q;
    a.nnz_pages = nnz_pages;
    a.num_pages = num_pages;
    a.batch = batch_size;
    a.h_q = h_q;
    a.h_kv = h_kv;
    a.d = d;
    a.page_size = page_size;
    a.causal = causal > 0;
    a.sm_scale = sm_scale;
    return generic_attention(a, stream);
  }
  KV_API_BEGIN();
  KV_CHECK(batch_size >= 0 && total_q >= 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0)
      << "batch_prefill_paged_kv: bad shape";
  const int page_shift = paged_page_shift(page_size);
  KV_UNSUPPORTED(page_shift < 0) << "batch_prefill_paged_kv: page_size " << page_size << " is not built (16, 32, 64, 128)";
  KV_CHECK(num_pages < (int64_t{1} << 28)) << "batch_prefill_paged_kv: page ids must stay below 2^28";
  if (batch_size == 0 || total_q == 0) return TVMKV_OK;
  KV_CHECK(q && q_indptr && pages && page_indptr && length_info && output && lse)
      << "batch_prefill_paged_kv: NULL tensor";
  KV_CHECK(nnz_pages == 0 || page_values) << "batch_prefill_paged_kv: NULL page table";
  KV_CHECK(rotary_mode == 0 || (q_rope_position && k_rope_pos_offset))
      << "batch_prefill_paged_kv: inline RoPE needs the position arrays";
  PrefillParams p{};
  p.page_shift = page_shift;
  p.q = static_cast<const half_t*>(q);
  p.q_indptr = q_indptr;
  p.pages = static_cast<const half_t*>(pages);
  p.page_indptr = page_indptr;
  p.page_values = page_values;
  p.last_page_len = length_info;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = causal > 0;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  p.rotary = rotary_mode != 0;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_rope_position = q_rope_position;
  p.k_rope_pos_offset = k_rope_pos_offset;
  p.merge_into = merge_into;
  if (sliding_window != 0) {  // length_info is (3, B): last_page_len, window offset, sink size
    p.window_offset = length_info + batch_size;
    p.sink_size = length_info + 2 * static_cast<int64_t>(batch_size);
    p.layer_window = sliding_window_size;
  }
  const bool ext = p.rotary != 0 || sliding_window != 0;
  hipStream_t s = as_stream(stream);
  // (a launch under capture keeps the scratch memory that it has always needed)
  const KvSplit split(p, total_q, nnz_pages * page_size / batch_size, d, s, stream_is_capturing(s) ? 0 : longest);
  if (beside != nullptr) {  // the work that writes the state which this launch merges into
    const bool together = split.splits > 1 && !p.stream_kv && !ext && (d == 64 || d == 128);
    PromptLaunch shares;
    if (together) {
      shares.p = p;
      shares.slots = row_tile_slots(p, total_q);
      shares.src = kPaged;
    }
    const int code = (*beside)(together ? &shares : nullptr);
    if (code != TVMKV_OK) return code;
    if (together) {
      split.finish(p, d, s);
      KV_LAUNCH_CHECK();
      return TVMKV_OK;
    }
  }
  if (d == 128) {
    launch_prefill<128, 128, kPaged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (d == 64) {
    launch_prefill<64, 64, kPaged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (d == 256) {
    launch_prefill<256, 256, kPaged, 16>(p, total_q, ext, rope_theta, s, scaling);
  } else if (padded_head_dim(d)) {
    launch_prefill_padded<kPaged>(p, total_q, d, ext, "batch_prefill_paged_kv", s);
  } else {
    KV_UNSUPPORTED(true) << "batch_prefill_paged_kv: head_dim " << d << " is not built (64, 80, 96, 112, 128, 256)";
  }
  split.finish(p, d, s);
  KV_LAUNCH_CHECK();
  KV_API_END();
}

int tvmkv_batch_prefill_paged_kv(const void* q, const int32_t* q_indptr, const void* pages,
                                 const int32_t* page_indptr, const int32_t* page_values,
                                 const int32_t* length_info, const int32_t* k_rope_pos_offset,
                                 const int32_t* q_rope_position, void* output, float* lse, int64_t causal,
                                 int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                                 int32_t batch_size, int64_t total_q, int64_t nnz_pages, int64_t num_pages,
                                 int32_t h_q, int32_t h_kv, int32_t d, int32_t page_size, int32_t sliding_window,
                                 int32_t sliding_window_size, void* stream) {
  return paged_prefill(q, q_indptr, pages, page_indptr, page_values, length_info, k_rope_pos_offset, q_rope_position,
                       output, lse, causal, rotary_mode, rope_scale, rope_theta, sm_scale, batch_size, total_q,
                       nnz_pages, num_pages, h_q, h_kv, d, page_size, sliding_window, sliding_window_size,
                       /*merge_into=*/false, stream);
}

int tvmkv_batch_prefill_paged_kv_merge(const void* q, const int32_t* q_indptr, const void* pages,
                                       const int32_t* page_indptr, const int32_t* page_values,
                                       const int32_t* length_info, const int32_t* k_rope_pos_offset,
                                       const int32_t* q_rope_position, void* output, float* lse, int64_t causal,
                                       int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                                       int32_t batch_size, int64_t total_q, int64_t nnz_pages, int64_t num_pages,
                                       int32_t h_q, int32_t h_kv, int32_t d, int32_t page_size,
                                       int32_t sliding_window, int32_t sliding_window_size, void* stream) {
  return paged_prefill(q, q_indptr, pages, page_indptr, page_values, length_info, k_rope_pos_offset, q_rope_position,
                       output, lse, causal, rotary_mode, rope_scale, rope_theta, sm_scale, batch_size, total_q,
                       nnz_pages, num_pages, h_q, h_kv, d, page_size, sliding_window, sliding_window_size,
                       /*merge_into=*/true, stream);
}

int tvmkv_batch_prefill_paged_kv_scaled(const void* q, const int32_t* q_indptr, const void* pages,
                                        const int32_t* page_indptr, const int32_t* page_values,
                                        const int32_t* length_info, const int32_t* k_rope_pos_offset,
                                        const int32_t* q_rope_position, void* output, float* lse, int64_t causal,
                                        int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                                        int32_t batch_size, int64_t total_q, int64_t nnz_pages, int64_t num_pages,
                                        int32_t h_q, int32_t h_kv, int32_t d, int32_t page_size, int32_t sliding_window,
                                        int32_t sliding_window_size, int32_t merge_into,
                                        const tvmkv_rope_scaling* rope_scaling, void* stream) {
  return paged_prefill(q, q_indptr, pages, page_indptr, page_values, length_info, k_rope_pos_offset, q_rope_position,
                       output, lse, causal, rotary_mode, rope_scale, rope_theta, sm_scale, batch_size, total_q,
                       nnz_pages, num_pages, h_q, h_kv, d, page_size, sliding_window, sliding_window_size,
                       merge_into != 0, stream, rope_scaling);
}

}  // extern "C"

int tvmkv::prefill_paged_with_lengths(const void* q, const int32_t* q_indptr, const void* pages, const int32_t* page_indptr,
                                      const int32_t* page_values, const int32_t* length_info, const int32_t* k_rope_pos_offset,
                                      const int32_t* q_rope_position, void* output, float* lse, int64_t causal, int64_t rotary_mode,
                                      double rope_scale, double rope_theta, double sm_scale, int32_t batch_size, int64_t total_q,
                                      int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv, int32_t d, int32_t page_size,
                                      int32_t sliding_window, int32_t sliding_window_size, int32_t merge_into,
                                      const tvmkv_rope_scaling* rope_scaling, int64_t longest, void* stream) {
  return paged_prefill(q, q_indptr, pages, page_indptr, page_values, length_info, k_rope_pos_offset, q_rope_position, output, lse,
                       causal, rotary_mode, rope_scale, rope_theta, sm_scale, batch_size, total_q, nnz_pages, num_pages, h_q, h_kv, d,
                       page_size, sliding_window, sliding_window_size, merge_into != 0, stream, rope_scaling, longest);
}

int tvmkv::prefill_shared_prefix(const SharedPrefixDecode& a, const std::function<int(const PromptLaunch*)>& own, void* stream) {
  return paged_prefill(a.q, a.prefix_q_indptr, a.pages, a.prefix.page_indptr, a.prefix.page_values, a.prefix.length_info, nullptr, nullptr,
                       a.out, a.lse, /*causal=*/0, /*rotary_mode=*/0, 1.0, 1e4, a.sm_scale, a.prefix.sequences, a.total_q,
                       a.prefix.nnz_pages, a.num_pages, a.h_q, a.h_kv, a.d, a.page_size, 0, 0, /*merge_into=*/true, stream, nullptr,
                       a.longest, &own);
}

extern "C" {

static int cached_and_new(const void* q, int64_t q_token_stride, const int32_t* q_rope_position, int64_t apply_rope,
                          double rope_scale, double rope_theta, const int32_t* q_indptr, const void* k, const void* v,
                          const void* pages, const int32_t* page_indptr, const int32_t* page_values,
                          const int32_t* last_page_len, void* output, float* lse, double sm_scale, int32_t batch_size,
                          int64_t total_q, int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv, int32_t d,
                          int32_t page_size, void* stream) {
  KV_API_BEGIN();
  KV_CHECK(batch_size >= 0 && total_q >= 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0)
      << "batch_prefill_cached_and_new_kv: bad shape";
  const int page_shift = paged_page_shift(page_size);
  KV_UNSUPPORTED(page_shift < 0) << "batch_prefill_cached_and_new_kv: page_size " << page_size << " is not built (16, 32, 64, 128)";
  KV_CHECK(num_pages < (int64_t{1} << 28)) << "batch_prefill_cached_and_new_kv: page ids must stay below 2^28";
  if (batch_size == 0 || total_q == 0) return TVMKV_OK;
  KV_CHECK(q && q_indptr && k && v && pages && page_indptr && last_page_len && output && lse)
      << "batch_prefill_cached_and_new_kv: NULL tensor";
  KV_CHECK(nnz_pages == 0 || page_values) << "batch_prefill_cached_and_new_kv: NULL page table";
  KV_CHECK(apply_rope == 0 || q_rope_position) << "batch_prefill_cached_and_new_kv: RoPE needs the position array";
  PrefillParams p{};
  p.page_shift = page_shift;
  p.q = static_cast<const half_t*>(q);
  p.q_token_stride = q_token_stride;
  p.q_inline_rope = apply_rope != 0;
  p.q_rope_position = q_rope_position;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_indptr = q_indptr;
  p.k = static_cast<const half_t*>(k);
  p.v = static_cast<const half_t*>(v);
  p.kv_indptr = q_indptr;  // the new tokens are the queries' own
  p.pages = static_cast<const half_t*>(pages);
  p.page_indptr = page_indptr;
  p.page_values = page_values;
  p.last_page_len = last_page_len;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = 1;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  hipStream_t s = as_stream(stream);
  const KvSplit split(p, total_q, (nnz_pages * page_size + total_q) / batch_size, d, s);
  if (d == 128) {
    launch_prefill<128, 128, kBoth, 16>(p, total_q, false, rope_theta, s);
  } else if (d == 64) {
    launch_prefill<64, 64, kBoth, 16>(p, total_q, false, rope_theta, s);
  } else if (d == 256) {
    launch_prefill<256, 256, kBoth, 16>(p, total_q, false, rope_theta, s);
  } else {
    KV_UNSUPPORTED(true) << "batch_prefill_cached_and_new_kv: head_dim " << d << " is not built (64, 128, 256)";
  }
  split.finish(p, d, s);
  KV_LAUNCH_CHECK();
  KV_API_END();
}

int tvmkv_batch_prefill_cached_and_new_kv(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                                          const void* pages, const int32_t* page_indptr,
                                          const int32_t* page_values, const int32_t* last_page_len, void* output,
                                          float* lse, double sm_scale, int32_t batch_size, int64_t total_q,
                                          int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv,
                                          int32_t d, int32_t page_size, void* stream) {
  return cached_and_new(q, 0, nullptr, 0, 1.0, 1e4, q_indptr, k, v, pages, page_indptr, page_values, last_page_len,
                        output, lse, sm_scale, batch_size, total_q, nnz_pages, num_pages, h_q, h_kv, d, page_size,
                        stream);
}

int tvmkv_batch_prefill_cached_and_new_kv_fused_q(const void* qkv, const int32_t* q_rope_position, int64_t apply_rope,
                                                  double rope_scale, double rope_theta, const int32_t* q_indptr,
                                                  const void* k, const void* v, const void* pages,
                                                  const int32_t* page_indptr, const int32_t* page_values,
                                                  const int32_t* last_page_len, void* output, float* lse,
                                                  double sm_scale, int32_t batch_size, int64_t total_q,
                                                  int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv,
                                                  int32_t d, int32_t page_size, void* stream) {
  return cached_and_new(qkv, static_cast<int64_t>(h_q + 2 * h_kv) * d, q_rope_position, apply_rope, rope_scale,
                        rope_theta, q_indptr, k, v, pages, page_indptr, page_values, last_page_len, output, lse, sm_scale,
                        batch_size, total_q, nnz_pages, num_pages, h_q, h_kv, d, page_size, stream);
}

static int tree_attn_ragged(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                            const int32_t* kv_indptr, const int32_t* q_rope_position, const int32_t* mn_indptr,
                            const int32_t* mask, void* output, float* lse, int64_t rotary_mode, double rope_scale,
                            double rope_theta, double sm_scale, int32_t batch_size, int64_t total_q, int32_t h_q,
                            int32_t h_kv, int32_t d, const tvmkv_rope_scaling* scaling, void* stream) {
  if (d != 64 && d != 128 && d != 256) {  // the generic matrix-core kernel
    GenericAttention a;
    a.what = "batch_tree_attn";
    a.rotary_mode = rotary_mode;  // key t of sequence b sits at q_rope_position[kv_indptr[b] + t]
    a.q_rope_position = q_rope_position;
    a.rope_scale = rope_scale;
    a.rope_theta = rope_theta;
    a.rope_scaling = scaling;
    a.q = q;
    a.q_indptr = q_indptr;
    a.k = k;
    a.v = v;
    a.kv_indptr = kv_indptr;
    a.tree_indptr = mn_indptr;
    a.tree_labels = mask;
    a.out = output;
    a.lse = lse;
    a.total_q = total_q;
    a.batch = batch_size;
    a.h_q = h_q;
    a.h_kv = h_kv;
    a.d = d;
    a.sm_scale = sm_scale;
    return generic_attention(a, stream);
  }
  KV_API_BEGIN();
  KV_CHECK(batch_size >= 0 && total_q >= 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0) << "batch_tree_attn: bad shape";
  if (batch_size == 0 || total_q == 0) return TVMKV_OK;
  KV_CHECK(q && q_indptr && k && v && kv_indptr && mn_indptr && mask && output && lse) << "batch_tree_attn: NULL tensor";
  KV_CHECK(rotary_mode == 0 || q_rope_position) << "batch_tree_attn: inline RoPE needs the position array";
  PrefillParams p{};
  p.q = static_cast<const half_t*>(q);
  p.q_indptr = q_indptr;
  p.k = static_cast<const half_t*>(k);
  p.v = static_cast<const half_t*>(v);
  p.kv_indptr = kv_indptr;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = 0;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  p.rotary = rotary_mode != 0;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_rope_position = q_rope_position;
  p.k_rope_pos_offset = q_indptr;  // not used: keys take their positions from q_rope_position
  p.k_pos_from_q = 1;
  p.tree_indptr = mn_indptr;
  p.tree_order = mask;
  hipStream_t s = as_stream(stream);
  if (d == 128) {
    launch_prefill<128, 128, kRagged, 16>(p, total_q, true, rope_theta, s, scaling);
  } else if (d == 64) {
    launch_prefill<64, 64, kRagged, 16>(p, total_q, true, rope_theta, s, scaling);
  } else if (d == 256) {
    launch_prefill<256, 256, kRagged, 16>(p, total_q, true, rope_theta, s, scaling);
  } else {
    KV_UNSUPPORTED(true) << "batch_tree_attn: head_dim " << d << " is not built (64, 128, 256)";
  }
  KV_LAUNCH_CHECK();
  KV_API_END();
}

int tvmkv_batch_tree_attn(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                          const int32_t* kv_indptr, const int32_t* q_rope_position, const int32_t* mn_indptr,
                          const int32_t* mask, void* output, float* lse, int64_t rotary_mode, double rope_scale,
                          double rope_theta, double sm_scale, int32_t batch_size, int64_t total_q, int32_t h_q,
                          int32_t h_kv, int32_t d, void* stream) {
  return tree_attn_ragged(q, q_indptr, k, v, kv_indptr, q_rope_position, mn_indptr, mask, output, lse, rotary_mode, rope_scale,
                          rope_theta, sm_scale, batch_size, total_q, h_q, h_kv, d, nullptr, stream);
}

int tvmkv_batch_tree_attn_scaled(const void* q, const int32_t* q_indptr, const void* k, const void* v,
                                 const int32_t* kv_indptr, const int32_t* q_rope_position, const int32_t* mn_indptr,
                                 const int32_t* mask, void* output, float* lse, int64_t rotary_mode, double rope_scale,
                                 double rope_theta, double sm_scale, int32_t batch_size, int64_t total_q, int32_t h_q,
                                 int32_t h_kv, int32_t d, const tvmkv_rope_scaling* rope_scaling, void* stream) {
  return tree_attn_ragged(q, q_indptr, k, v, kv_indptr, q_rope_position, mn_indptr, mask, output, lse, rotary_mode, rope_scale,
                          rope_theta, sm_scale, batch_size, total_q, h_q, h_kv, d, rope_scaling, stream);
}

int tvmkv_tree_attn_paged_kv(const void* q, const int32_t* q_indptr, const void* pages, const int32_t* page_indptr,
                             const int32_t* page_values, const int32_t* length_info,
                             const int32_t* k_rope_pos_offset, const int32_t* q_rope_position, void* output,
                             float* lse, int64_t rotary_mode, double rope_scale, double rope_theta, double sm_scale,
                             const int32_t* tree_order_indptr, const int32_t* tree_order, int32_t batch_size,
                             int64_t total_q, int64_t nnz_pages, int64_t num_pages, int32_t h_q, int32_t h_kv,
                             int32_t d, int32_t page_size, int32_t sliding_window, void* stream) {
  if (rotary_mode == 0 && (!tuned_page_size(page_size) || (d != 64 && d != 128 && d != 256))) {
    GenericAttention a;  // the generic matrix-core kernel
    a.what = "tree_attn_paged_kv";
    a.sliding_window = sliding_window;
    a.q = q;
    a.q_indptr = q_indptr;
    a.pages = pages;
    a.page_indptr = page_indptr;
    a.page_values = page_values;
    a.last_page_len = length_info;
    a.tree_indptr = tree_order_indptr;
    a.tree_labels = tree_order;
    a.out = output;
    a.lse = lse;
    a.total_q = total_q;
    a.nnz_pages = nnz_pages;
    a.num_pages = num_pages;
    a.batch = batch_size;
    a.h_q = h_q;
    a.h_kv = h_kv;
    a.d = d;
    a.page_size = page_size;
    a.sm_scale = sm_scale;
    return generic_attention(a, stream);
  }
  KV_API_BEGIN();
  KV_CHECK(batch_size >= 0 && total_q >= 0 && h_q > 0 && h_kv > 0 && h_q % h_kv == 0)
      << "tree_attn_paged_kv: bad shape";
  const int page_shift = paged_page_shift(page_size);
  KV_UNSUPPORTED(page_shift < 0) << "tree_attn_paged_kv: page_size " << page_size << " is not built (16, 32, 64, 128)";
  KV_CHECK(num_pages < (int64_t{1} << 28)) << "tree_attn_paged_kv: page ids must stay below 2^28";
  // the reference kernel asserts the same (tree_attn.py:700-702)
  KV_UNSUPPORTED(rotary_mode != 0) << "tree_attn_paged_kv: inline rotary mode is not supported in tree attention";
  if (batch_size == 0 || total_q == 0) return TVMKV_OK;
  KV_CHECK(q && q_indptr && pages && page_indptr && length_info && output && lse && tree_order_indptr && tree_order)
      << "tree_attn_paged_kv: NULL tensor";
  KV_CHECK(nnz_pages == 0 || page_values) << "tree_attn_paged_kv: NULL page table";
  PrefillParams p{};
  p.page_shift = page_shift;
  p.q = static_cast<const half_t*>(q);
  p.q_indptr = q_indptr;
  p.pages = static_cast<const half_t*>(pages);
  p.page_indptr = page_indptr;
  p.page_values = page_values;
  p.last_page_len = length_info;
  p.output = static_cast<half_t*>(output);
  p.lse = lse;
  p.batch_size = batch_size;
  p.h_q = h_q;
  p.h_kv = h_kv;
  p.group = h_q / h_kv;
  p.causal = 0;
  p.scale_log2 = static_cast<float>(sm_scale) * kLog2e;
  p.rope_scale = static_cast<float>(rope_scale);
  p.q_rope_position = q_rope_position;
  p.k_rope_pos_offset = k_rope_pos_offset;
  if (sliding_window != 0) {  // length_info is (3, B): last_page_len, window offset, sink size
    p.window_offset = length_info + batch_size;
    p.sink_size = length_info + 2 * static_cast<int64_t>(batch_size);
  }
  p.tree_indptr = tree_order_indptr;
  p.tree_order = tree_order;
  hipStream_t s = as_stream(stream);
  const KvSplit split(p, total_q, nnz_pages * page_size / batch_size, d, s);
  if (d == 128) {
    launch_prefill<128, 128, kPaged, 16>(p, total_q, true, rope_theta, s);
  } else if (d == 64) {
    launch_prefill<64, 64, kPaged, 16>(p, total_q, true, rope_theta, s);
  } else if (d == 256) {
    launch_prefill<256, 256, kPaged, 16>(p, total_q, true, rope_theta, s);
  } else {
    KV_UNSUPPORTED(true) << "tree_attn_paged_kv: head_dim " << d << " is not built (64, 128, 256)";
  }
  split.finish(p, d, s);
  KV_LAUNCH_CHECK();
  KV_API_END();
}

}  // extern "C"
