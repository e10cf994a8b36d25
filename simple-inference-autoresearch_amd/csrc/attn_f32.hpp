// Float32 attention: decode calls whose q or K/V are float32 (attn_f32, on
// the vector ALUs), and prefill in float32 (attn_f32_prefill.hip, fp32 MFMAs).
//
// The reference wrappers accept any float dtype and return q's dtype
// (kernels/flash_decode_kernel.py:119-160, kernels/attention_kernel.py:235-305);
// its decode kernel computes in fp32 on vector lanes, tl.sum(q * k) and
// tl.sum(p * v) with an online softmax (kernels/flash_decode_kernel.py:85-114).
// The 16-bit MFMA kernels of this library take 16-bit or int8 operands, so
// float32 inputs run here instead, in fp32 end to end: products, sums,
// exponentials and the output (rounded to q's dtype).
//
// attn_f32 (gfx950, wave64):
//  * A work item is one (sequence, KV head), up to kF32Cols of its query heads
//    ("columns") and one split of the key range [0, kv_len).  The K/V rows of
//    the item are read once for all of its columns.
//  * D/4 lanes share a key row, 4 dimensions each (16-byte fp32 loads; 8 or 4
//    bytes for 16-bit and int8 K/V), so one load instruction of a wave reads
//    64/(D/4) whole rows.  Each lane group runs an online softmax over its
//    own keys (kF32Unroll keys per step); the dot products are completed
//    with cross-lane sums inside the group.  Groups are merged with shuffles,
//    waves through LDS.
//  * Split-K: the key range is cut into nsplit pieces of tps keys; with more
//    than one piece each item writes (m, l, acc) and attn_f32_merge combines
//    them.  The split is chosen on the host from the cache capacity (lengths
//    stay on the device), so one captured graph serves every length.
#pragma once

#include "sia_common.hpp"

namespace sia {

constexpr int kF32Cols = 8;     // columns (query heads) per work item of attn_f32
constexpr int kF32TileCols = 32;   // columns per work-group of the prefill kernel (attn_f32_prefill.hip)
constexpr int kF32Unroll = 4;   // keys per lane group per step

struct F32Args {
  const char* q; int64_t q_sb, q_sh, q_sm;           // byte strides; head_dim contiguous
  char* out; int64_t o_sb, o_sh, o_sm;
  const char* k; int64_t k_s0, k_sh, k_sn;           // s0: batch (contiguous) or page (paged)
  const char* v; int64_t v_s0, v_sh, v_sn;
  const char* ks; int64_t ks_s0, ks_sh, ks_sn;       // int8 scales (nullptr otherwise)
  const char* vs; int64_t vs_s0, vs_sh, vs_sn;
  const int32_t* bt; int64_t bt_sb, bt_sl;           // block table (element strides), nullptr = contiguous
  int64_t num_pages;
  int32_t page_size;
  const int32_t* kv_len; int32_t kv_per_seq;         // (decode)
  int32_t cap;                                       // keys addressable: S or max_blocks * page_size (decode)
  int32_t B, Hq, Hkv, G, Tq, Tk, causal;
  int32_t ncol;                                      // Tq * G columns per (sequence, KV head)
  int32_t nchunk;                                    // ceil(ncol / columns per work item)
  int32_t fold;                                      // prefill kernel: CU count, or 0 (see there)
  int32_t nsplit, tps;                               // key-range split: nsplit pieces of tps keys
  float qk_scale;                                    // sm_scale * log2(e)
  float* part;                                       // nsplit > 1: [row][split][D + 4] (acc, m, l)
};

struct F32Launch {
  F32Args a;
  int D;
  int q_dtype;       // also the output dtype
  int kv_dtype;
  int scale_dtype;   // int8 K/V only
  hipStream_t stream;
  hipEvent_t begin_event;   // optional, recorded around the main kernel
  hipEvent_t end_event;
};

// Launches attn_f32 (and attn_f32_merge when nsplit > 1); implemented in attn_f32.hip.
int launch_attn_f32(F32Launch& L);

// Prefill of float32 q, k, v on the matrix cores: nchunk = ceil(ncol /
// kF32TileCols), no split, no paging (attn_f32_prefill.hip).
int launch_attn_f32_prefill(F32Launch& L);

// attn_f32_merge alone, for split-K partials written in its layout by another
// kernel: head_dim D, output dtype out_dtype (f16 / bf16 / f32).
int launch_attn_merge(const F32Args& a, int D, int out_dtype, hipStream_t stream);

// Bytes of split-K partials for `rows` output rows, `nsplit` pieces, head_dim D.
inline size_t f32_partial_bytes(int64_t rows, int64_t nsplit, int D) {
  return (size_t)rows * (size_t)nsplit * (size_t)(D + 4) * 4;
}

}  // namespace sia
