// Host-side launcher declarations shared by the kernel translation units and the C ABI.
#pragma once
#include "fa_common.h"

namespace fa {
struct BwdKParams;
// What fa_last_kernel() reports: every attention launcher notes the kernel it enqueued (FA_KERNEL_* | flags |
// computed head dims << 16) for the calling thread.  Host-side only.
extern thread_local int32_t g_last_kernel;
inline int note_kernel(int launch_error, int id, bool dropout, bool split, int head_dims) {
    if (launch_error == 0) g_last_kernel = id | (dropout ? FA_KERNEL_FLAG_DROPOUT : 0) | (split ? FA_KERNEL_FLAG_SPLIT : 0) | (head_dims << 16);
    return launch_error;
}
#define FA_DECL_PREFILL(name) int name(const KParams& kp, hipStream_t stream);
FA_DECL_PREFILL(launch_prefill_bf16_64)
FA_DECL_PREFILL(launch_prefill_bf16_128)
FA_DECL_PREFILL(launch_prefill_bf16_256)
FA_DECL_PREFILL(launch_prefill_fp16_64)
FA_DECL_PREFILL(launch_prefill_fp16_128)
FA_DECL_PREFILL(launch_prefill_fp16_256)
#undef FA_DECL_PREFILL

int prefill_block_n(int d_bucket);   // key-tile length of the prefill kernel for a bucket
int prefill_block_m(int d_bucket);
// Query rows from which an unsplit launch takes the pipelined / ping-pong kernels instead of
// the general tiled kernel (measured on 32..511 rows x 128..16384 keys, bf16, with and without a causal mask:
// head dims 64 and 128 +15-45 % from 128 rows on, 0..+28 % at 100-127 rows, -9..+14 % at 64 rows; head dim 256
// +25-57 % from 32 rows on, +50-100 % from 128).
inline int prefill_long_rows(int d_bucket) { return d_bucket > 128 ? 32 : 96; }

// Launches with split keys or packed rows that the pipelined kernel takes (PART, fa_prefill_il.h), beyond head dim 128 those with split
// keys that the 16-rows-per-wave kernel takes (PART, fa_prefill_pp16.h); `p` is the problem as the kernels see it.  Against the general kernel, which had
// them: packed rows left whole, bf16, 70 tokens, 64 / 8 heads, 8 x 2k, d 128 84 -> 61 us, 16 x 6400, d 64 200 -> 152; split ones in `plan` (fa_api.hip).
// Packed rows stay with the general kernel where they are fewer than 16 blocks over short keys, which it takes in the same time (40 tokens, 16 / 2
// heads, one cache of 1k: 15.9 and 15.2 us at d 64 short, 17.2 and 17.6 full), and where they are fewer than 8 over long ones, whose many parts it
// starts and merges in less (12 tokens, 2 x 8 / 1 heads, 28836 keys 33 and 42; up to 8192 keys 0.88 of its time, 1.02 at worst).
inline bool prefill_parts(const fa_fwd_params& p, bool packed, int d_bucket) {
    if (p.p_dropout > 0.f || p.cu_seqlens_q || p.seqlen_q < prefill_long_rows(d_bucket)) return false;
    if (!packed || d_bucket > 128) return !packed;
    const int64_t blocks = (int64_t)((p.seqlen_q + 127) / 128) * p.h * p.b;
    return blocks >= 16 || (p.seqlen_k >= 4096 && (blocks >= 8 || p.seqlen_k <= 8192 || p.window_left >= 0));
}
// Launches of so few rows that 32 (4 waves to a group) or 64 of them (2) make no more than a workgroup per CU: waves that share 32 query
// rows and split the keys between them (KW, fa_prefill_il.h), else 1.  Up to head dim 64 not where all keys are one tile of 64: their sums
// meet for 0.5 us (packed, 4 x 24 tokens, 8 heads 5.6 us without and 6.2 with; so does a longer cache of which no more is filled: 382 rows,
// 8 heads, 70 of 564 rows filled 5.6 and 6.2, all of them 7.6 and 7.5; 43 rows, 10 x 8 heads, 181 rows, all filled 8.2 and 6.1).
inline int prefill_key_waves(const fa_fwd_params& p, bool packed, int d_bucket) {
    if (d_bucket > 128 || p.p_dropout > 0.f || packed || (d_bucket <= 64 && p.seqlen_k <= 64)) return 1;
    const int64_t heads = (int64_t)p.h * p.b;
    return (p.seqlen_q + 31) / 32 * heads <= 256 ? 4 : (p.seqlen_q + 63) / 64 * heads <= 256 ? 2 : 1;
}
// Launches for key waves whose K and V the 256 MiB of the memory-side cache do not hold, unmasked and on more than 128 (batch, head) pairs: those
// are the ping-pong kernel's, which asks for longer runs of them.  33-64 rows, full mask, ping-pong / key waves: 160 pairs, d 96, 3000 keys 54 / 38 us, 4096
// 70 / 50; d 128, 4096 (320 MiB) 84 / 101; 192 pairs, d 128, 2048 44 / 39, 4096 (384 MiB) 84 / 104; 256 pairs, d 80, 1024 24 / 21, 3000
// 56 / 41, 4096 (320 MiB) 79 / 99.
inline bool prefill_past_key_waves(const fa_fwd_params& p, int d_bucket, bool masked) {
    return d_bucket == 128 && !masked && (int64_t)p.h * p.b > 128 && (int64_t)4 * p.b * p.seqlen_k * p.h_k * p.d >= (int64_t)1 << 28;
}

int launch_decode(const KParams& kp, hipStream_t stream);      // small-q split-KV kernel
int launch_combine(const KParams& kp, hipStream_t stream);     // merge of split partials
// k_new/v_new (+rotary) -> cache; batch indices by falling cache length -> order
int launch_prepare_rows(const KParams& kp, bool append, int32_t* order, hipStream_t stream);
bool cache_order_applies(const fa_fwd_params& p);     // the attention kernel can walk such an order, and more than one round of it
int launch_attn_probs(const KParams& kp, hipStream_t stream);  // s_dmask: signed softmax probabilities (testing)
int launch_rotary(const fa_rotary_params& p, hipStream_t stream);   // standalone rotary embedding
// Packed batches: builds the work list of a forward launch of `nblocks` workgroups with row blocks of
// `block_m` rows in kp.p.work_counter and sets kp.work_items, when the batch qualifies and the caller lent
// enough words (fa_work_list_words); otherwise leaves kp.work_items NULL.
int prepare_work_list(KParams& kp, int block_m, int64_t nblocks, hipStream_t stream);
int64_t work_list_words(const fa_fwd_params& p);    // words behind work_counter that make every packed launch qualify

#define FA_DECL_BWD(name) int name(const BwdKParams& kp, hipStream_t stream);
FA_DECL_BWD(launch_bwd_bf16_64)
FA_DECL_BWD(launch_bwd_bf16_128)
FA_DECL_BWD(launch_bwd_bf16_256)
FA_DECL_BWD(launch_bwd_fp16_64)
FA_DECL_BWD(launch_bwd_fp16_128)
FA_DECL_BWD(launch_bwd_fp16_256)
#undef FA_DECL_BWD
}  // namespace fa
