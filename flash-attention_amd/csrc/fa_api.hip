// C ABI of libfa_mi355x.so: argument checks, mask normalisation, split planning and kernel
// dispatch.  Host-side counterpart of the reference's mha_fwd / mha_varlen_fwd / mha_fwd_kvcache
// bodies after tensor unpacking (csrc/flash_attn/flash_api.cpp:248-424, 426-585, 1038-1279) and of
// run_mha_fwd's dtype x head-dim dispatch (:194-204).
#include <cmath>
#include <cstdio>
#include <cstring>
#include <iterator>
#include <string>
#include <utility>
#include <vector>
#include <algorithm>
#include <functional>
#include <mutex>
#include "fa_prefill.h"
#include "fa_bwd_stream.h"
#include "fa_launch.h"

namespace fa {

static thread_local std::string g_err;
thread_local int32_t g_last_kernel = FA_KERNEL_NONE;
static thread_local int32_t g_last_bwd_kernel = FA_BWD_KERNEL_NONE;
static int fail(const char* msg) { g_err = msg; return 1; }
static int fail_hip(int e, const char* where) {
    g_err = std::string(where) + ": " + hipGetErrorString((hipError_t)e);
    return 2;
}

int prefill_block_n(int db) { return db == 64 ? PrefillTile<64>::BN : db == 128 ? PrefillTile<128>::BN : PrefillTile<256>::BN; }
int prefill_block_m(int db) { return 128 * (db == 64 ? PrefillTile<64>::RB : db == 128 ? PrefillTile<128>::RB : PrefillTile<256>::RB); }
static int bucket(int d) { return d <= 64 ? 64 : d <= 128 ? 128 : 256; }

static const int kNumCU = 256;   // MI355X
#ifndef FA_DEC_SLOTS
#define FA_DEC_SLOTS 8192       // chunk slots per launch, one workgroup per chunk
#endif
#ifndef FA_DEC_SLOTS_P
#define FA_DEC_SLOTS_P 4096     // same for the persistent, ticket-scheduled kernel
#endif
#ifndef FA_DEC_SB
#define FA_DEC_SB 8
#endif
#ifndef FA_SPLIT_BELOW
#define FA_SPLIT_BELOW 256      // row blocks x heads x batch below which the tiled kernel's keys are split
#endif
#ifndef FA_TILE_SLOTS
#define FA_TILE_SLOTS 4096      // chunk slots per launch of the ticket-scheduled tiled kernel
#endif
#ifndef FA_TILE_MINLEN
#define FA_TILE_MINLEN 2048     // its shortest chunk (keys)
#endif
#ifndef FA_DEC_MINLEN
#define FA_DEC_MINLEN 512       // shortest chunk of the decode kernel (keys) once the launch fills the CUs
#endif

// the keys are those of caches whose lengths are on the device: the plan sees their capacity
static bool cache_lengths(const fa_fwd_params& p) { return p.cu_seqlens_k && !p.is_seqlens_k_cumulative; }

// The small-q streaming kernel packs seqlen_q x (h / h_k) rows into 16 MFMA columns, or two times 16 up to head dim 128 over caches (the
// tiled kernel, whose row block is 128 rows, is what more rows take).  17-32 rows, bf16, appended with rotary, GPU time of the call,
// tiled -> decode: 4 positions, 64 / 8 heads, d 128, one cache of 8k 29.8 -> 17.0 us, 32k 41.7 -> 23.0, batch 4 x 2k 32.1 -> 17.8; 16 / 2 heads,
// 48 x 5k 51.1 -> 45.0; one position on 32 heads of 1, 8 x 8k 31.8 -> 20.5.
// 1500 drawn shapes of 17-32 rows, each cache shape with all full, an even spread, one full and all an eighth full, appended with rotary, appended and
// plain, set the lines.  What takes the call else is the tiled kernel, or with ungrouped heads up to 256 streams (batch x kv heads) and 1024-4096 keys
// the key waves; those need a launch of their own for the append, which the decode kernel does itself.  Its time over theirs:
//  * grouped heads, appended: 0.73-0.95 up to 256 streams at any length (3 tokens, 64 / 8 heads, 8 sequences of 573 18.8 / 15.9 us), 0.77-0.97 from 512 on;
//    without an append 0.55-1.0 past 1024 keys, 1.0-1.15 below;
//  * ungrouped heads: 0.87-1.01 appended up to 256 keys; 1.2-2.1 up to 512 keys, up to 1024 from 64 streams on, up to 4096 from 128 on; 0.6-0.95 past those lines;
//  * past 4096 keys 0.6-1.0 up to 256 streams; of full caches past 16384 up to 1.15, of unequal ones down to 0.4;
//  * 257-511 streams are a chunk and a bit for each of the 512 workgroups that run at once: up to 2048 keys 0.9 of unequal caches, 1.05-1.3 of full ones,
//    1.4-2 of caches an eighth full; past 2048 0.78-0.87 in the mean (0.4-0.75 unequal, 1.0-1.1 full, up to 4 an eighth full); up to 512 keys, one chunk, 0.75-0.91
//    appended, 1.0-1.16 not.  512 streams and more are 0.77-1.0 past 512 keys either way;
//  * where K and V are known to be full (no cache lengths) the tiled kernel's shorter parts win from 4096 keys on (16 streams of 22480 keys 33.9 and
//    48.0) and the key waves below (44 x 11 of 271 7.9 and 14.5);
//  * at head dims 65-128 caches that are streamed past the memory-side cache are bound by memory in both (8 streams of 262144, d 64, an eighth full
//    44.1 and 34.9);
//  * behind a left window bound split keys are mostly empty in either and the append is a launch of its own in both: up to 256 streams of more
//    than 1024 keys (0.47-0.64 at 128 streams and up to 2048 keys), ungrouped of more than 2048 (1.7-2.2 below), else 64 of more than 512.
// One position on grouped heads behind a left window bound
// takes no tiled form with the heads as rows (groups_as_rows): they are row blocks of their own there (159 x 1024 / 32 heads, 468 keys,
// d 64 1604 us and 67; where those are few, 1 x 512 / 16, 11.7 and 15.1).  Head dim 256 needs more than 512 registers (8 x 8k keys, 16 / 2 heads 60 -> 81 us).
// (Rows that stand for grouped heads come here again as rows of ungrouped ones: no line may take those where it leaves the grouped ones.)
static bool use_decode_kernel(const fa_fwd_params& p) {
    if (p.cu_seqlens_q != nullptr || p.p_dropout != 0.f) return false;
    const int64_t rows = (int64_t)p.seqlen_q * (p.h / p.h_k);
    if (rows <= 16) return true;
    if (rows > 32 || p.d > 128) return false;
    const int64_t streams = (int64_t)p.b * p.h_k;
    const bool past_cache = p.d > 64 && 4 * streams * p.seqlen_k * p.d >= kStreamKvBytes;
    if (p.seqlen_q == 1 && p.window_left >= 0) return !past_cache;
    if (!cache_lengths(p) || past_cache) return false;
    const int64_t sk = p.seqlen_k;
    const bool appended = p.k_new != nullptr, grouped = p.h > p.h_k;
    if (p.window_left >= 0) return sk > (grouped ? 1024 : 2048) ? streams < 256 : streams < 128 && sk > (streams < 64 ? 512 : 1024);
    if (streams >= 512) return appended || sk > 512;
    if (streams > 256) return sk > 2048 || (appended && sk <= 512);
    if (sk > 4096 || (grouped && sk > 1024) || (appended && (grouped || sk <= 256))) return true;
    return streams < 128 && sk > (streams < 64 ? 512 : 1024);
}

// One query position with more grouped q heads per kv head than the decode kernel packs into its 16 columns:
// the grouped heads of a kv head take the place of the query positions (the reference's
// seqlenq_ngroups_swapped, csrc/flash_attn/flash_api.cpp:1096-1104 for mha_fwd and :1265 for the kv-cache call).
// q and out are read as (batch, G rows, h_k heads, d) through their strides, so one workgroup per kv head
// serves all of its q heads and every K/V row is fetched once instead of G times (batch 16 x 64k keys, 32 q
// heads on 1 kv head: 1.6 ms -> 0.1 ms).  A single query row at the end of the keys sees all of them under a
// causal mask or a right window bound, so those are dropped; a left bound is not, and keeps the plain form.
// softmax_lse and the split accumulators need no change: (b, h, 1) and (b, h_k, G) index the same words.
static bool groups_as_rows(fa_fwd_params& q) {
    const int G = q.h_k > 0 ? q.h / q.h_k : 0;
    if (q.seqlen_q != 1 || G <= 16 || q.s_dmask || q.window_left >= 0 || q.cu_seqlens_q || q.p_dropout != 0.f || use_decode_kernel(q)) return false;
    q.seqlen_q = G;
    q.h = q.h_k;
    q.q_row_stride = q.q_head_stride;
    q.q_head_stride *= G;
    q.o_row_stride = q.o_head_stride;
    q.o_head_stride *= G;
    q.is_causal = 0;
    q.window_right = -1;
    return true;
}

// A few query positions (speculative or chunked decoding) with grouped q heads: seqlen_q x G rows would be
// G separate row blocks of the tiled kernel, each streaming the kv head's K/V for a handful of rows.  Here the
// (position, grouped head) pairs of a kv head become the rows of one problem with h_k heads (KParams::pack_g):
// row = position * G + head within the group, so a workgroup serves up to 128 of them and K/V are fetched once
// (batch 64 x 16k keys, 64 q heads on 8 kv heads, 4 positions: 4.0 -> 0.8 ms).  Up to 16 rows the decode kernel
// packs them itself; from 128 positions on a row block is full without packing.  Returns G when it applies.
static int positions_and_groups_as_rows(fa_fwd_params& q, int64_t* q_head_stride, int64_t* o_head_stride) {
    const int G = q.h_k > 0 ? q.h / q.h_k : 0;
    if (q.seqlen_q <= 1 || q.seqlen_q >= 128 || G < 2 || q.cu_seqlens_q || q.p_dropout != 0.f || q.s_dmask || use_decode_kernel(q)) return 0;
    if (q_head_stride) *q_head_stride = q.q_head_stride;
    if (o_head_stride) *o_head_stride = q.o_head_stride;
    q.seqlen_q *= G;
    q.h = q.h_k;
    q.q_head_stride *= G;
    q.o_head_stride *= G;
    return G;
}

static int check_common(const fa_fwd_params* p) {
    if (!p) return fail("params is NULL");
    if (!p->q || !p->k || !p->v || !p->o || !p->softmax_lse) return fail("q, k, v, o and softmax_lse must be set");
    if (p->dtype != FA_DTYPE_FP16 && p->dtype != FA_DTYPE_BF16) return fail("FlashAttention only support fp16 and bf16 data type");
    if (p->b <= 0) return fail("batch size must be positive");
    if (p->d <= 0 || p->d > 256) return fail("FlashAttention forward only supports head dimension at most 256");
    if (p->d % 8 != 0) return fail("head dimension must be a multiple of 8 at the C boundary (pad on the host)");
    if (p->h <= 0 || p->h_k <= 0 || p->h % p->h_k != 0) return fail("Number of heads in key/value must divide number of heads in query");
    if (p->seqlen_q < 0 || p->seqlen_k < 0) return fail("sequence lengths must be non-negative");
    if (p->num_splits < 0 || p->num_splits > FA_MAX_SPLITS) return fail("num_splits > 128 not supported");
    // every global access is a 16-byte piece of a row
    const void* ptrs[] = {p->q, p->k, p->v, p->o, p->k_new, p->v_new};
    for (const void* q : ptrs) if ((uintptr_t)q % 16 != 0) return fail("q, k, v, o, k_new and v_new must be 16-byte aligned");
    const int64_t strides[] = {p->q_batch_stride, p->q_row_stride, p->q_head_stride, p->k_batch_stride, p->k_row_stride,
                               p->k_head_stride, p->v_batch_stride, p->v_row_stride, p->v_head_stride, p->o_batch_stride,
                               p->o_row_stride, p->o_head_stride, p->knew_batch_stride, p->knew_row_stride,
                               p->knew_head_stride, p->vnew_batch_stride, p->vnew_row_stride, p->vnew_head_stride};
    for (int64_t st : strides) if (st % 8 != 0) return fail("strides must be multiples of 8 elements (16-byte rows)");
    // the long-sequence kernels add a 32-bit lane byte offset (up to 64 rows) to a 64-bit tile base
    if (p->k_row_stride < 0 || p->k_row_stride >= ((int64_t)1 << 23) || p->v_row_stride < 0 || p->v_row_stride >= ((int64_t)1 << 23))
        return fail("k and v row strides must be below 2^23 elements");
    if (!(p->p_dropout >= 0.f && p->p_dropout < 1.f)) return fail("p_dropout must be in [0, 1)");
    if (p->p_dropout > 0.f && !p->rng_state) return fail("rng_state is required when p_dropout > 0");
    if (p->s_dmask && (p->sdm_rows < p->seqlen_q || p->sdm_cols < p->seqlen_k)) return fail("s_dmask is smaller than (seqlen_q, seqlen_k)");
    return 0;
}

// elements from the first to one past the last element of a (b, s, h, d) tensor with non-negative strides
static int64_t span_elems(int64_t b, int64_t s, int64_t h, int64_t d, int64_t bs, int64_t rs, int64_t hs) {
    return (b - 1) * bs + (s - 1) * rs + (h - 1) * hs + d;
}
static bool spans_overlap(const void* a, int64_t a_elems, const void* b, int64_t b_elems) {
    const uintptr_t a0 = (uintptr_t)a, a1 = a0 + (uintptr_t)a_elems * 2, b0 = (uintptr_t)b, b1 = b0 + (uintptr_t)b_elems * 2;
    return a0 < b1 && b0 < a1;
}

// No two (entry, row, head) of a (b, s, h, d) tensor share an element: from the smallest stride up, each dimension steps over
// all that the smaller ones span.  (Sufficient, and true of every layout that is a permuted or cut dense one; not of a tensor
// expanded over a dimension.)
static bool rows_apart(int64_t b, int64_t s, int64_t h, int64_t d, int64_t bs, int64_t rs, int64_t hs) {
    std::pair<int64_t, int64_t> dims[] = {{bs, b}, {rs, s}, {hs, h}};       // stride, size
    std::sort(std::begin(dims), std::end(dims));
    int64_t span = d;
    for (const auto& [stride, size] : dims) {
        if (size <= 1) continue;
        if (stride < span) return false;
        span += (size - 1) * stride;
    }
    return true;
}

// the caller lent enough zeroed words for the persistent decode kernel
static bool counters_ok(const fa_fwd_params& p) {
    return p.work_counter != nullptr && p.work_counter_len >= FA_WORK_COUNTER_WORDS && (uintptr_t)p.work_counter % 8 == 0;
}
// epoch of the next launch's ticket counters (epoch_counter_next, fa_common.h): never zero, never the same twice
// in a row within a process
static uint32_t next_epoch() {
    static std::atomic<uint32_t> g_epoch{0};
    uint32_t e = g_epoch.fetch_add(1, std::memory_order_relaxed) + 1;
    if (e == 0) e = g_epoch.fetch_add(1, std::memory_order_relaxed) + 1;
    return e;
}

// Split planning for 256 CUs.
struct SplitPlan {
    int splits = 1;        // partial slots (what the caller allocates)
    int len = 0;           // keys per chunk
    int persistent = 0;    // ticket-scheduled decode kernel
    int sa = 0, sb = 0, sub = 0;
};

// Keys that a row block of 128 rows sees at most: all of them, or what a window leaves (a split by all keys left most parts empty).
static int64_t visible_keys(const fa_fwd_params& p, int sk) {
    if (p.window_left < 0) return sk;
    const int64_t right = p.is_causal ? 0 : p.window_right < 0 ? sk : p.window_right;
    return std::min<int64_t>(sk, (int64_t)p.window_left + right + 128);
}

static SplitPlan plan(const fa_fwd_params& p_in, bool allow_split) {
    SplitPlan r;
    fa_fwd_params p = p_in;
    // what runs is the problem with the grouped heads as rows (no change when it already is)
    const bool packed = !groups_as_rows(p) && positions_and_groups_as_rows(p, nullptr, nullptr) > 0;
    const int sk = p.seqlen_k;
    const int db = bucket(p.d);
    const bool dec = use_decode_kernel(p);
    const int64_t rows = (int64_t)p.seqlen_q * (p.h / p.h_k);
    // The tiled kernel under the persistent schedule of the decode kernel (prefill_persistent_kernel): one row
    // block per (batch, kv head) with every q head of the kv head in it, over a cache whose lengths are on the
    // device.  Chunks of FA_TILE_MINLEN keys or more (about FA_TILE_SLOTS per launch; down to 512 keys in launches too
    // small to fill the CUs otherwise), their remainders in halves, quarters or eighths of a chunk (see sb below).
    const int64_t wgs = (int64_t)((p.seqlen_q + prefill_block_m(db) - 1) / prefill_block_m(db)) * p.h * p.b;
    int64_t tile_chunk = 0;
    const bool wide_parts = !dec && db > 128 && prefill_parts(p, packed, db);
    // Few rows, by waves that split the keys among themselves (KW, fa_prefill_il.h): whole up to 4096 keys, where splitting them over more
    // workgroups costs more than it gives; earlier where there are few of those.  bf16 GPU time, split on the general kernel -> whole:
    // 128 tokens, 32 / 8 heads, cache of 4096 (full / an eighth), d 128 40.3 -> 34.0 / 35.0 -> 15.3 us; 100 tokens, 16 heads, 1024 33 -> 18;
    // 1024 x 4096, 8 heads, d 64 35 -> 21; 256 x 1500, 16 heads 18 -> 11.  Whole at 16 blocks of 4096 keys, d 128: 28.3 against 26.1; at 4: 28.7
    // against 19.0.
    // Up to 32 rows a (batch, head) pair is one workgroup of them, a quarter of what more rows make: 2500 keys at 24 pairs, d 128 25.1 against
    // 20.4 split on the general kernel, 2824 at 64, d 96 25.5 and 22.9; 2000 keys 0.39-0.46 of it.  Caches that the ping-pong kernel would take instead
    // (fa_prefill_inst.hip) are split: 30 x 256 / 8 heads, 3633 keys, one full among short ones 64 us whole, 48 split.
    const int64_t kw_wgs = p.seqlen_q <= 32 ? wgs / 4 : wgs;
    const bool key_waves_here = prefill_key_waves(p, packed, db) > 1 && !(cache_lengths(p) && prefill_past_key_waves(p, db, p.window_left >= 0 || p.is_causal || p.window_right >= 0));
    const bool whole_by_key_waves = !dec && key_waves_here && visible_keys(p, sk) <= (kw_wgs >= 24 ? 4096 : kw_wgs >= 12 ? (p.seqlen_q <= 32 ? 2560 : 3072) : 2048);
    if (!dec && allow_split && p.num_splits == 0 && p.p_dropout == 0.f && counters_ok(p) && !p.cu_seqlens_q && cache_lengths(p) &&
        p.seqlen_q <= prefill_block_m(db) && p.h == p.h_k) {
        // (launches too small to give every resident workgroup a chunk of FA_TILE_MINLEN keys take shorter ones,
        // down to 512: one sequence of 16k keys on 8 kv heads is 64 chunks of 2048 keys, a quarter of the CUs)
        const int64_t fill = ((int64_t)sk * wgs / (2 * kNumCU) + 511) / 512 * 512;
        const int64_t minlen = std::min<int64_t>(FA_TILE_MINLEN, std::max<int64_t>(512, fill));
        const int64_t len = (std::max<int64_t>(minlen, (int64_t)sk * wgs / FA_TILE_SLOTS) + 511) / 512 * 512;
        // (launches that fill the CUs without a split keep the plain form up to 8192 keys: two or three chunks per
        // sequence do not pay for the merge)
        // (Rows that are plain query positions, enough of them for the pipelined kernels, in a launch that fills the
        // CUs: left whole, on those kernels -- 96-128 rows, 256-2048 row blocks, caches of 8k-32k: +5-57 % at head
        // dims 64 / 128 and +30-85 % at 256 on equal and on short lengths, -6..-11 % on lengths drawn from the
        // whole range at 512 row blocks; with 64 row blocks the ticket schedule is 2-4 x as fast.)
        const bool whole_is_fast = (!packed && p.seqlen_q >= prefill_long_rows(db) && wgs >= kNumCU) || whole_by_key_waves;
        if (sk >= 2 * len && (wgs < kNumCU || sk >= 8192) && !whole_is_fast && !wide_parts) tile_chunk = len;
    }
    const int gran = dec ? 128 : tile_chunk ? 512 : prefill_block_n(db);
    auto rup = [](int64_t x, int64_t m) { return (int)((x + m - 1) / m * m); };
    int splits = 1;
    bool automatic = false;
    if (p.p_dropout > 0.f) allow_split = false;      // as the reference (flash_api.cpp:380)
    if (allow_split && sk > 0) {
        if (p.num_splits > 1) {
            splits = p.num_splits;
        } else if (p.num_splits == 0) {
            automatic = true;
            if (dec) {
                // ~8k chunk slots over the whole launch (16 per resident workgroup), chunks of at
                // least 256 to 512 keys: measured best trade between per-workgroup start-up cost and
                // the tail left by ragged cache lengths on 256 CUs x 2 resident groups.
                // With the caller's scratch word the kernel is persistent and takes longer chunks
                // (4096 keys at batch 64 x 8 kv heads x 32k), their ragged remainders in pieces of 512+ keys.
                const int64_t streams = (int64_t)p.b * p.h_k;
                // Chunks shorter than 512 keys are mostly start-up and merge (batch 4 x 32k: +22 % with
                // 512 over 256); 256 only while 512-key chunks would leave resident slots empty.
                // 17-32 rows leave twice the partial results: 256 only while such chunks all run at once and the merge weighs no more than 32
                // of them, as many as its lanes hold (64 where they leave half of the resident slots empty).  bf16, d 128, 256 / 512: 1 x 8
                // streams of 8k 17.0 / 19.8 us, 48 of 5k on one kv head 36.3 / 29.9; time of 256 over 512, full and an eighth full: up to 256
                // chunks 0.86 and 0.88 up to 8192 keys, 1.0 and 0.82 up to 16384, 1.10 and 0.87 beyond; 257-512 chunks 1.05 and 0.82, 1.11 and 0.81, 1.2 and 0.85.
                const int64_t c256 = (sk + 255) / 256;
                const bool short_chunks = rows <= 16 ? streams * ((sk + FA_DEC_MINLEN - 1) / FA_DEC_MINLEN) < 2 * kNumCU
                                                     : streams * c256 <= (c256 <= 32 ? 2 * kNumCU : c256 <= 64 ? kNumCU : 0);
                const int64_t minlen = short_chunks ? 256 : FA_DEC_MINLEN;
                int64_t len = rup(std::max<int64_t>(minlen, (int64_t)sk * streams / FA_DEC_SLOTS), 128);
                if (counters_ok(p)) {
                    const int64_t lp = rup(std::max<int64_t>(256, (int64_t)sk * streams / FA_DEC_SLOTS_P), 128);
                    // (at least 2048 keys once persistent: batch 4 x 128k keys x 8 kv heads +9 % over 1024-key chunks)
                    if (lp >= 1024) len = std::max<int64_t>(lp, 2048);
                }
                // (17-32 rows leave twice the partial results: whole streams that fill the resident slots are not split up to
                // 4096 keys.  bf16, 4 positions, 16 / 2 heads, d 64, 256 x 1024 keys split 36.7, whole 23.2 us, 256 x 3000 75 and 62; 15 positions,
                // 2 / 1 heads, 529 x 3136, an eighth full 54 and 21.)
                if (rows > 16 && streams >= 2 * kNumCU && sk <= 4096) len = rup(sk, 128);
                splits = (int)((sk + len - 1) / len);
                // (17-32 rows fill twice the partial results, also in launches that the tiled kernel did not split: no more of
                // them than the no-allocation entry point has room for, with eight slots for remainders)
                if (rows > 16) {
                    const int64_t slot_bytes = (int64_t)p.b * p.h * p.seqlen_q * (4 + 4 * ((p.d + 31) / 32 * 32));
                    const int64_t most = ((int64_t)FA_NOALLOC_SCRATCH_BYTES - (128 << 10)) / slot_bytes - 8;
                    splits = (int)std::max<int64_t>(1, std::min<int64_t>(splits, most));
                }
            } else if (tile_chunk) {
                splits = (int)((sk + tile_chunk - 1) / tile_chunk);
            } else {
                const int64_t keys = visible_keys(p, sk);
                if (wide_parts) {
                    // Head dims 129-256, one workgroup a CU: parts that fill the CUs (PART, fa_prefill_pp16.h), where a row block is long enough to
                    // pay for the merge.  bf16, before (split on the general kernel, its tickets, or whole) -> now, d 192 (256): 466 rows on 6068 keys, 32
                    // blocks 84 -> 40 us (89 -> 49); 512 on 2048, 64 blocks 53 -> 34 (62 -> 40); 2048 on 4096, 128 blocks 97 -> 73 (115 -> 86); caches, 64
                    // rows, 8 heads: 1 x 32k 107 -> 46 (111 -> 56), 4 x 4k full 62 -> 30 (63 -> 37), an eighth full 53 -> 20 (54 -> 25), 8 x 8k of even
                    // spread 162 -> 59 (165 -> 78).  Whole against two parts: 900 keys at 80 blocks 30 / 36, 1152 at 112 35 / 39,
                    // 1024 at 64 31 / 30, 2471 at 160 64 / 69.
                    // Of caches the plan sees the capacity.  Of one row block the general kernel's tickets (which took 24 x 8k full 445 us where whole takes
                    // 215, and an even spread 297 and 176) dealt the one full cache among short ones to all CUs, so a part must not be long: past 6144 keys
                    // parts of 4608, up to twice as many parts as else, or four.  One full, tickets / as else / so: 21 x 54 tokens, 8 heads, 16212 rows, d 256
                    // 157 / 365 / 143 us (all full 789 / 477 / 524), 13 x 38, 32771 rows, d 224 161 / 215 / 157, 22 x 50, 13551, d 192 164 / 278 / 140.
                    // More row blocks, from 64 or 96 of them on, were left whole, and parts of a short cache cost more than they gain: up to 8192 keys they still
                    // are (4 x 488 tokens, 8 heads, 2049 rows, d 224 all full 48 whole, 51 in two, an eighth full 15 and 29; 3 x 508, 8 heads, 4214, d 256 105 and 76,
                    // 22 and 34; past the line 2 x 142, 32 heads, 16850, d 256 449 and 259, 75 and 73), and on more than half of the CUs at any length (3 x 220, 32 heads,
                    // 17609, d 160 all full 352 and 410, an eighth 55 and 75, though one full among short ones takes 351 and 207).
                    const bool cache = cache_lengths(p), one_block = p.seqlen_q <= prefill_block_m(db) && p.h == p.h_k;
                    const int more = cache && keys >= 16384 ? 2 : 1;
                    int64_t want = wgs <= kNumCU / 2 ? std::max<int64_t>(kNumCU / wgs, 2 * more) : wgs < kNumCU ? more : 1;
                    if (cache && one_block && p.b > 1 && keys > 6144 * want && wgs < kNumCU) want = std::min<int64_t>((keys + 4607) / 4608, std::max<int64_t>(2 * want, 4));
                    const bool whole = cache && !one_block && wgs >= (keys <= 2048 ? 64 : 96) && (keys <= 8192 || wgs > kNumCU / 2);
                    const int64_t row_bytes = 4 + 4 * ((p.d + 31) / 32 * 32), most = ((int64_t)FA_NOALLOC_SCRATCH_BYTES - (128 << 10)) / (row_bytes * p.b * p.h * p.seqlen_q);
                    if (!whole && keys > (wgs <= 32 ? 640 : wgs <= 64 ? 1024 : 2047)) splits = (int)std::max<int64_t>(1, std::min({want, keys / 256, most}));
                } else if (prefill_parts(p, packed, db)) {
                    // The pipelined kernel takes the split form (PART, fa_prefill_il.h) as well as the whole one; a split adds the merge
                    // and the partial rows in 32 bits (2 parts of 128 row blocks of 512 tokens at 1024 keys: 20 us whole, 32 split), so
                    // it pays where few row blocks see many keys.  Parts: as many as fill the resident slots, of four tiles or more.
                    // bf16 GPU time, split on the general kernel by the capacity of the cache -> now: 512 tokens on a cache of 32k,
                    // 32 / 8 heads, d 128 343 -> 274 us (one of an eighth of that 176 -> 64); 213 tokens, 8 / 1 heads, 5 x 25k, d 64
                    // 109 -> 82; 24 tokens, 64 / 8 heads, 16 x 6400, d 128 178 -> 115; 3 x 874 rows on 9981 keys, window 256, d 80 54 -> 15.
                    // Packed rows over long caches are split up to 255 blocks (78 tokens, 53 x 4 / 2 heads, one full cache of 19703 rows among short ones 293 whole,
                    // 127 in three parts; all full 386 and 395), in one part more than fill the slots from 64 blocks on (24 tokens, 14 x 16 / 2, 8319 rows, one full
                    // 58.4 and 55.5), and below in 16 at most (69 tokens, 10 x 4 / 1, 17861 rows 67.9 in 17, 59.6; 51 tokens, 5 x 4 / 1, 28479 keys, d 64 42.0 in 76, 33.4).
                    const int64_t split_below = packed && keys > 4096 ? kNumCU : keys <= (db <= 64 ? 2048 : 1024) ? 64 : keys <= 2048 ? 96 : 192;
                    const int64_t slots = (db <= 64 ? 3 : 2) * kNumCU, parts = !packed ? slots / wgs : wgs >= 64 ? (slots + wgs - 1) / wgs : std::min<int64_t>(slots / wgs, 16);
                    // (one part more than fill the slots: no more partial rows than the no-allocation entry point has room for, 255 full blocks at d 128)
                    const int64_t row_bytes = 4 + 4 * ((p.d + 31) / 32 * 32), most = ((int64_t)FA_NOALLOC_SCRATCH_BYTES - (128 << 10)) / (row_bytes * p.b * p.h * p.seqlen_q);
                    if (wgs < split_below && keys > 640 && !whole_by_key_waves) splits = (int)std::max<int64_t>(1, std::min({parts, keys / 256, most}));
                } else {
                    if (wgs < FA_SPLIT_BELOW && !whole_by_key_waves) {
                        const int64_t want = (2 * kNumCU + wgs - 1) / wgs;
                        splits = (int)std::min<int64_t>(want, (sk + 255) / 256);
                    }
                }
                // From 256 row blocks on nothing is split here, also where every (batch, head) is one row block
                // over long keys: the plan sees the capacity of a cache, not the lengths in it, and chunks cut for
                // the capacity are mostly empty workgroups when the sequences are short (batch 64, 4096 keys in
                // caches of 32768, 4 positions on 8 kv heads: 0.28 ms split against 0.19).
            }
        }
        splits = std::max(1, std::min(splits, FA_MAX_SPLITS));
        splits = std::min(splits, (sk + gran - 1) / gran);   // never more chunks than tiles
        splits = std::max(1, splits);
    }
    int len = rup((sk + splits - 1) / std::max(1, splits), gran);
    if (len <= 0) len = gran;
    splits = std::max(1, (sk + len - 1) / len);               // drop chunks the rounding emptied
    r.splits = splits;
    r.len = len;
    // Persistent two-pass schedule: complete chunks first, then each sequence's ragged remainder in
    // up to eight pieces of a chunk, drawn from a ticket counter.  Needs the caller's scratch word.
    // The pieces of a remainder stay at 512 keys or more (halves of a 1024-key chunk, quarters of a
    // 2048-key one, eighths from 4096 on): shorter pieces are mostly start-up and merge (measured
    // +6 % at batch 256 x 4k and at batch 64 x 8k with 16 grouped heads, nothing lost at config 5).
    // (The tiled kernel pays more per item -- its Q rows, a first tile nothing overlaps, up to 128 partial rows to
    // write: about what 160 keys take -- so its chunks below 4096 keys are only halved: pieces of 1024 keys or more for
    // chunks of FA_TILE_MINLEN, 256 at the least for the 512-key chunks of a launch that would not fill the CUs.)
    // Halves, quarters or eighths of a multiple of 512: whole tiles.
    const int sb = tile_chunk ? (len < 4096 ? 2 : len < 8192 ? 4 : FA_DEC_SB) : len < 2048 ? 2 : len < 4096 ? 4 : FA_DEC_SB;
    if ((dec || tile_chunk) && automatic && splits > 1 && counters_ok(p) && len >= (dec ? 1024 : 512) && splits + sb <= FA_MAX_SPLITS) {
        r.persistent = 1;
        r.sa = splits;
        r.sb = sb;
        r.sub = len / sb;
        r.splits = r.sa + r.sb;
    }
    return r;
}

// A window bound as the kernels use it: they add it to row and key positions in 32 bits.  Bounds this far out mask nothing.
static int32_t window_bound(int32_t w) { return std::min(w, (int32_t)1 << 29); }

static void fill_kparams(KParams& kp, const fa_fwd_params& p) {
    kp.p = p;
    fa_fwd_params& q = kp.p;
    // mask normalisation (flash_api.cpp:111-114, 296-297)
    if (q.is_causal) q.window_right = 0;
    q.window_left = window_bound(q.window_left);
    q.window_right = window_bound(q.window_right);
    kp.has_left = q.window_left >= 0;
    kp.has_right = q.window_right >= 0;
    kp.scale_log2 = q.softmax_scale * (float)M_LOG2E;
    kp.d_rounded = (q.d + 31) / 32 * 32;
    kp.num_splits = 1;
    kp.split_len = 0;
    kp.num_m_blocks = 0;
    kp.rotary_q = 0;
    kp.dec_persistent = kp.dec_sa = kp.dec_sb = kp.dec_sub = kp.dec_append = kp.dec_compact = 0;
    kp.work_counter = q.work_counter;
    kp.epoch = next_epoch();
    kp.work_items = nullptr;
    kp.cache_order = nullptr;
    kp.rng_out = nullptr;
    kp.rng_seed = kp.rng_offset = 0;
    kp.pack_g = 0;
    kp.pack_q_hs = kp.pack_o_hs = 0;
    // K + V, 16-bit elements; seqlen_k is the cache capacity (or the longest packed sequence): an upper bound
    kp.stream_kv = (int64_t)4 * q.b * q.seqlen_k * q.h_k * q.d >= kStreamKvBytes;
}

static int run_attention(KParams& kp, hipStream_t stream) {
    const fa_fwd_params& p = kp.p;
    int e;
    if (use_decode_kernel(p)) {
        e = launch_decode(kp, stream);
        if (e) return fail_hip(e, "decode kernel launch");
    } else {
        const bool bf = p.dtype == FA_DTYPE_BF16;
        switch (bucket(p.d)) {
            case 64: e = bf ? launch_prefill_bf16_64(kp, stream) : launch_prefill_fp16_64(kp, stream); break;
            case 128: e = bf ? launch_prefill_bf16_128(kp, stream) : launch_prefill_fp16_128(kp, stream); break;
            default: e = bf ? launch_prefill_bf16_256(kp, stream) : launch_prefill_fp16_256(kp, stream); break;
        }
        if (e) return fail_hip(e, "prefill kernel launch");
    }
    if (kp.num_splits > 1) {
        e = launch_combine(kp, stream);
        if (e) return fail_hip(e, "combine kernel launch");
    }
    if (p.s_dmask) {
        e = launch_attn_probs(kp, stream);
        if (e) return fail_hip(e, "attention probability kernel launch");
    }
    return 0;
}

// `p` is the problem as the caller described it (before grouped heads become rows): plan() applies those
// transforms itself, so what it answers here is what fa_plan_splits answered for the same params.
static int resolve_splits(KParams& kp, const fa_fwd_params& p, bool allow_split) {
    const SplitPlan r = plan(p, allow_split);
    const int s = r.splits;
    kp.num_splits = s;
    kp.split_len = r.len;
    kp.dec_persistent = r.persistent;
    kp.dec_sa = r.sa; kp.dec_sb = r.sb; kp.dec_sub = r.sub;
    kp.dec_compact = r.persistent && !kp.has_left && p.b <= kDecCompactMaxBatch;
    if (s > 1 && (!p.o_accum || !p.lse_accum)) return fail("o_accum and lse_accum are required when the key range is split (see fa_plan_splits)");
    return 0;
}

// One pass or two (fa_bwd_stream.h / fa_bwd.h).  A workgroup of the one-pass kernel takes a whole (batch, kv head) with all its
// grouped heads, two workgroups per CU, while the two-pass grids have a workgroup per 128 rows of every head: what they gain
// from formed-once products one pass loses where pairs are too few to fill the CUs, the more so the longer a pair takes.
// `fill` is the share of the 512 slots that work over the launch: one workgroup of a CU runs 3/2 as fast alone as next to
// another, and a last round that fills no more than one per CU takes two thirds of a whole one.  The launch takes one pass
// from the fill of `kFill` on, by the whole 64 x 128 tiles of a pair and the heads grouped on a kv head, set at the largest
// fill at which one pass lost more than 3 % in any of causal / full, with / without dropout (5485 calls drawn over all that the
// rule takes: 0.55 of the two-pass time in the mean, 16 of them 1.04-1.29).  bf16, d 64, one pass / two passes, full mask:
//   256 tokens, 1 head per group: 128 pairs 28 / 23 us, 160 28 / 35, 512 44 / 74; 8 heads: 256 pairs 1.11 of the two-pass time
//   with dropout, 384 0.74-0.88.  512 tokens: 192 pairs 85 / 78, 256 89 / 99, 520 (a second round that is nearly empty) 210 / 202,
//   768 224 / 273; 8 heads: 128 pairs 1.9, 320 1.1, 512 0.8.  1024 tokens: 128 pairs 290 / 167, 384 418 / 459, 640 788 / 758;
//   32 heads: 32 pairs 7.6.  2048 tokens lose at any fill (the fp32 dQ tiles that go out and come back between key blocks).
// Packed sequences of unequal length fill the slots by themselves (longest first, snake order), but the launch lasts as long
// as the longest takes: what counts is how many pairs of that length the tokens would make, `kPairs`, again set by the worst of
// several distributions (even, one of 4 or 16 or a single one long, exponential).  512 tokens at most, one of 16 sequences
// that long and the rest an eighth of it: 512 pairs 0.97-1.03, 1024 0.57-0.64; 1024 at most: 512 pairs 1.4-2.1, 2048 0.5-0.7;
// a single one among short ones, 128 pairs: up to 6.
constexpr int64_t kMaxBwdScratch = (int64_t)1 << 29;
static bool bwd_one_pass_fits(const fa_bwd_params& p, int64_t total_q, int64_t total_k) {
    if (p.d > 64 || p.b <= 0 || p.h_k <= 0 || p.h % p.h_k != 0 || p.seqlen_q <= 0 || p.seqlen_k <= 0) return false;
    // (it fetches rows of `out` too, by 32-bit offsets like those of q, k, v and dout, which run_bwd checks)
    if (p.o_row_stride < 0 || p.o_row_stride >= ((int64_t)1 << 23)) return false;
    const int64_t pairs = (int64_t)p.b * p.h_k, area = (int64_t)((p.seqlen_q + 63) / 64 * 64) * ((p.seqlen_k + 127) / 128 * 128);
    const int G = p.h / p.h_k;
    if (std::max(p.seqlen_q, p.seqlen_k) > 1024 || pairs < 128) return false;
    // (up to twice the bytes of dq where every slot is in use, more where packed sequences are shorter than the declared maximum;
    // past the 256 MB of the memory-side cache it costs the gain: 3 or 4 heads, 800-1000 tokens, full mask: 1.09-1.30)
    if (bwd_stream_slot_bytes(p) * bwd_stream_slots(p) > kMaxBwdScratch) return false;
    int l = 0;
    for (int64_t most : {64 * 128, 128 * 128, 256 * 256, 384 * 384, 512 * 512, 768 * 768}) l += area > most;
    const int g = G == 1 ? 0 : G == 2 ? 1 : G <= 4 ? 2 : 3;
    // per cent; {1, 2, up to 4, more} heads per group
    static const int kFill[7][4] = {{0, 0, 0, 0}, {0, 0, 57, 76}, {40, 40, 64, 82}, {50, 64, 80, 85}, {62, 70, 85, 85}, {80, 85, 91, 93}, {85, 91, 91, 96}};
    static const int kPairs[4][2] = {{62, 250}, {80, 310}, {85, 310}, {85, 390}};      // at no tokens, and more at 1024
    const int64_t rounds = pairs / kBwdStreamSlots, rest = pairs % kBwdStreamSlots;
    const int64_t time = rounds * 768 + (rest == 0 ? 0 : rest <= 256 ? 512 : rest + 256);      // 768: a round of both workgroups of a CU
    const bool filled = pairs * 150 >= time * kFill[l][g];
    if (!p.cu_seqlens_q) return filled;
    if (l < 2) return filled && (G <= 2 || pairs > 256);      // (8 heads, 192-256 pairs: 0.99-1.22)
    if (total_q <= 0 || total_k <= 0) return false;
    const int64_t whole = (int64_t)(p.h_k * std::min((double)total_q / p.seqlen_q, (double)total_k / p.seqlen_k));
    // (sequences that are nearly all of one length run in rounds like a dense batch)
    if (whole < kPairs[g][0] + (int64_t)(kPairs[g][1] * std::sqrt((double)area) / 1024)) return false;
    if (whole * 5 >= pairs * 4) return filled;
    return l < 3 || p.b <= kBwdStreamOrdered;       // (more than that the kernel takes as they come: up to 2.0 at 500-1000 tokens)
}

// Whether two workgroups share a key block that is not cut, half of the head dimension each: 6 tile products' worth of work for 4,
// but twice the workgroups, for launches that leave CUs idle.  Up to head dim 128 by the count of key blocks (fa_bwd_inst.hip),
// at 193-256, and with dropout at 129-256, by it and by their weight: the steps of all of them over those of the heaviest one.
//   Dense, and packed of fewer than 8 streams: up to 128 blocks or, masked, a weight of 85.  bf16, whole backward, whole / shared: 2048 tokens, 2 kv heads, d 256, 96 blocks
//   1.08 causal and 1.09 full, 128 blocks 1.13 and 1.02; 200 drawn calls of more blocks: weight 70-85 1.02 in the mean (0.78-1.26),
//   85-96 0.98, 96-112 0.90, 123-160 0.75-0.96 (10 x 1681 tokens, 4 heads on 1, causal, weight 71 1.19; 10 x 2087, 88 0.90).
//   Packed, 8 (sequence, kv head) streams and more: each runs on one XCD (xcd_strided), whose 32 CUs hold the halves of 16 blocks at
//   a time.  So the longest sequence alone must not weigh more than 14 (16 under a mask), and the batch, past 128 blocks, not more
//   than 80, 10 to an XCD, counted as sequences of the declared maximum that its tokens would make (lengths are on the device).
//   764 drawn calls of more than 128 blocks by the maximum, whole / shared: the 230 shared by this rule 1.06 in the mean, 20 of them
//   0.72-0.97; the 534 others 0.85, 45 of them 1.03-1.24.  19 sequences, one of 1349 tokens, 4 heads on 1, d 256, causal 286 us shared,
//   322 whole; 4 of up to 3966, 8 on 2, full mask 2110 and 1602.
static bool bwd_halves(const fa_bwd_params& p, int64_t total_k) {
    const int D = bucket(p.d);
    const int64_t n = ((int64_t)p.seqlen_k + kBwdKeyBlock - 1) / kBwdKeyBlock, blocks = n * p.b * p.h_k;
    if (D <= 128) return blocks < 256 && p.seqlen_q >= 1024;
    if (p.d <= 192 && !(p.p_dropout > 0.f)) return false;
    const bool packed = p.cu_seqlens_q != nullptr;
    const int wl = window_bound(p.window_left), wr = p.is_causal ? 0 : window_bound(p.window_right);
    const bool masked = wl >= 0 || wr >= 0, strided = xcd_strided(packed, p.b, p.h_k);
    if (!strided && (blocks <= 128 || !masked)) return blocks <= 128;       // (no mask: the weight is the count, or unknown)
    if (n > 256) return false;
    int64_t sum = 0, most = 0;
    for (int64_t i = 0; i < n; i++) {
        int t_lo;
        const int64_t t = bwd_block_tiles((int)i * kBwdKeyBlock, p.seqlen_q, p.seqlen_k, wl >= 0, wl, wr >= 0, wr, bwd_dkv_rows(D), t_lo);
        sum += t;
        most = std::max(most, t);
    }
    const double sequences = packed && total_k > 0 ? std::min((double)p.b, (double)total_k / p.seqlen_k) : p.b;
    if (!strided) return sequences * p.h_k * sum <= 85.0 * most;
    return sum <= (masked ? 16 : 14) * most && (blocks <= 128 || sequences * p.h_k * sum <= 80.0 * most);
}

// How the dK/dV pass of a dense batch cuts the steps of its key blocks (BwdKParams::split_steps, split_pieces); no joins: not at all.
// A CU runs one workgroup at a time, so the pass lasts as long as the busiest of 256 CUs.  With fewer key blocks than CUs (few kv
// heads), or little more than one each under a causal mask, where the first one takes as long as all of a stream's average twice
// over, most of the chip is idle at the end.  Cutting a block costs: each piece starts up anew (kStart, in steps, fetch of its
// key rows and the first tile) and passes its sums on (kJoin).  The plan plays the launch through for limits of 1, 3/4 .. 1/16 of
// the longest block's steps, pieces in the order of the launch, each to the CU that is free first, and takes the
// shortest if it beats the uncut one by 15 %.  Of 110 drawn calls that it cuts the whole backward takes 0.70 of the uncut time in
// the mean, the worst 1.03 (d 160, 639 x 983 tokens, 8 heads: 72 us).  dK/dV pass, bf16, uncut -> cut (us):
//   causal: b 1, 2048 tokens, 8 heads on 1, d 128 352 -> 50; 8192 tokens 1375 -> 338, d 64 923 -> 202; 16k 3090 -> 1208;
//   2 x 4367, 12 on 3 580 -> 325; 2 x 1024, 16 on 2 182 -> 47; 16 x 512, 16 on 2 112 -> 57; 4 x 2039, 16 on 4, d 256 439 -> 342;
//   2 x 3797, 16 on 16, d 128 243: best cut 253, left whole.  Full mask: 1 x 4096, 32 on 4 811 -> 516; 1 x 5702, 8 on 8 320 -> 295.
// (uncut: two workgroups to a key block, half of the head dimension each, where the launch takes that form, bwd_halves)
// Streams that neither divide over the 8 XCDs nor are few enough to be dealt out unit by unit stay whole under a mask: an XCD's
// pieces are then not in falling order (xcd_stream_unit), and cutting loses (1 x 2998, 12 heads 84 -> 103).
struct BwdSplit { int steps, pieces; int64_t joins, bytes; };
static BwdSplit bwd_split_search(const fa_bwd_params& p) {
    const BwdSplit whole = {0, 0, 0, 0};
    if (p.cu_seqlens_q || p.b <= 0 || p.h_k <= 0 || p.h <= 0 || p.h % p.h_k != 0 || p.seqlen_q <= 0 || p.seqlen_k <= 0 || p.d <= 0) return whole;
    const int D = bucket(p.d), BM = bwd_dkv_rows(D);
    constexpr int kMaxBlocks = 2048;                                       // (8 key blocks to a CU)
    const int64_t n = ((int64_t)p.seqlen_k + kBwdKeyBlock - 1) / kBwdKeyBlock, streams = (int64_t)p.b * p.h_k;
    if (n > kMaxBlocks || n * streams > kMaxBlocks) return whole;
    const int wl = window_bound(p.window_left), wr = p.is_causal ? 0 : window_bound(p.window_right);
    const int64_t G = p.h / p.h_k;
    if ((wl >= 0 || wr >= 0) && streams > 8 && streams % 8 != 0) return whole;
    // in steps, from launches cut and uncut: at head dim 128 10 us to start and 5 to join, 1.9 a step; 256 1.7 a step
    const int kStart = D == 256 ? 6 : 5, kJoin = D == 256 ? 8 : 3;
    int64_t most = 0, work = 0;
    int64_t steps[kMaxBlocks];
    for (int64_t i = 0; i < n; i++) {
        int t_lo;
        steps[i] = G * bwd_block_tiles((int)i * kBwdKeyBlock, p.seqlen_q, p.seqlen_k, wl >= 0, wl, wr >= 0, wr, BM, t_lo);
        most = std::max(most, steps[i]);
        work += (steps[i] + kStart) * streams;
    }
    if (most > INT32_MAX / 2) return whole;
    typedef std::pair<int64_t, int64_t> Free;        // time at which CUs are free, and how many: a heap, the earliest in front
    Free heap[256 + 1];
    int free_times;
    auto push = [&](int64_t at, int64_t cus) { heap[free_times++] = Free(at, cus); std::push_heap(heap, heap + free_times, std::greater<Free>()); };
    // time of a launch whose block i is `parts(steps[i])` workgroups of `cost(steps[i], parts)` each; once that is known to be `bound`
    // or more, `bound`
    auto play = [&](int64_t bound, auto&& parts, auto&& cost) {
        int64_t time = 0, load = 0;
        for (int64_t i = 0; i < n; i++) {
            const int64_t c = parts(steps[i]);
            load += cost(steps[i], c) * c * streams;
        }
        if (load >= bound * 256) return bound;       // (of 256 CUs one has the mean or more)
        free_times = 0;
        push(0, 256);
        for (int64_t i = 0; i < n; i++) {
            const int64_t c = parts(steps[i]), piece = cost(steps[i], c);
            for (int64_t left = c * streams; left > 0;) {
                std::pop_heap(heap, heap + free_times, std::greater<Free>());
                const Free f = heap[--free_times];
                const int64_t m = std::min(left, f.second);
                left -= m;
                if (f.second > m) push(f.first, f.second - m);
                push(f.first + piece, m);
                time = std::max(time, f.first + piece);
                if (time >= bound) return bound;
            }
        }
        return time;
    };
    const int64_t forever = (int64_t)1 << 50;
    const int64_t uncut = play(forever, [](int64_t) { return (int64_t)1; }, [&](int64_t t, int64_t) { return t + kStart; });
    if (uncut * 256 * 10 < work * 11) return whole;      // the CUs are within 10 % of evenly loaded as it is
    BwdSplit best = whole;
    int64_t best_time = uncut * (p.d > 192 && n * streams <= 128 ? 15 : 17) / 20;
    for (int k : {12, 10, 8, 7, 6, 5, 4, 3, 2, 1}) {
        const int limit = (int)((most * k + 15) / 16);
        if (limit < 4) break;
        auto parts_of = [&](int64_t t) { return (int64_t)bwd_block_parts((int)t, limit); };
        int64_t pieces = 0;
        for (int64_t i = 0; i < n; i++) pieces += parts_of(steps[i]);
        const int64_t joins = (pieces - n) * streams, bytes = 2 * joins * bwd_partial_bytes(D) + joins * 4;
        if (bytes > kMaxBwdScratch) break;
        const int64_t time = play(best_time, parts_of, [&](int64_t t, int64_t parts) { return (t + parts - 1) / parts + kStart + (parts > 1 ? kJoin : 0); });
        if (time < best_time) {
            best_time = time;
            best = {limit, (int)pieces, joins, bytes};
        }
    }
    if (D == 256 && best.joins) {
        // Cutting blocks of few steps, 16-30, in four or more costs more than the search above says: a join takes longer the more
        // levels the tree has, 24 of them take a step's time of the memory (two partial sums out and in, 0.5 MB), and uncut two
        // workgroups may share a block, which then takes nine tenths of its steps.  Of 254 drawn calls that the search cuts this
        // leaves 39 whole, whose backward took 0.97-1.20 (1.04 in the mean) of the uncut time (6 x 666 tokens, 1 head, d 224, full
        // 68 us uncut, 82 cut; 2 x 340, 16 on 8, 61 and 71); the others 0.74 in the mean, the worst three 1.04-1.07.
        const bool columns = p.d > 192 || p.p_dropout > 0.f;      // all 256 of them, not 160 or 192
        const int kFirst = columns ? 8 : 6, kLevel = columns ? 3 : 2;
        const int64_t left = bwd_halves(p, 0) ? play(forever, [](int64_t) { return (int64_t)2; }, [&](int64_t t, int64_t) { return (t * 9 + 9) / 10 + kStart; }) : uncut;
        const int64_t cut = best.joins / 24 + play(left, [&](int64_t t) { return (int64_t)bwd_block_parts((int)t, best.steps); }, [&](int64_t t, int64_t parts) {
            int levels = 0;
            while (((int64_t)1 << levels) < parts) levels++;
            return (t + parts - 1) / parts + kStart + (levels ? kFirst + (levels - 1) * kLevel : 0);
        });
        if (cut >= left) return whole;
    }
    return best;
}

// The plan of a shape is asked for twice a call, for the room that is lent and at the launch, and again by the next layer and step:
// a thread keeps its last one.  It costs 1-6 us on most drawn calls, up to 230 on a long sequence of few heads (1 x 32768 tokens,
// 8 heads on 1 191 us; twice 210 when it was played through for every limit, each time it was asked for; 3 x 30140, 2 on 1 19, twice 421).
static BwdSplit bwd_split_plan(const fa_bwd_params& p) {
    struct Shape { int32_t b, h, h_k, d, sq, sk, wl, wr, causal, dropout, packed; };
    const Shape shape = {p.b, p.h, p.h_k, p.d, p.seqlen_q, p.seqlen_k, p.window_left, p.window_right, p.is_causal, p.p_dropout > 0.f, p.cu_seqlens_q != nullptr};
    static thread_local struct { Shape shape; BwdSplit split; } last;       // (zero: a batch of none, which has no plan)
    if (memcmp(&last.shape, &shape, sizeof(shape)) != 0) {
        last.split = bwd_split_search(p);
        last.shape = shape;
    }
    return last.split;
}

// What a backward runs when it is lent `lent` bytes.
struct BwdForm { bool one_pass, halves; BwdSplit split; };
static BwdForm bwd_form(const fa_bwd_params& p, int64_t total_q, int64_t total_k, int64_t lent) {
    const bool fits = bwd_one_pass_fits(p, total_q, total_k);
    BwdForm f = {fits && lent >= bwd_stream_slot_bytes(p) * bwd_stream_slots(p), false, {0, 0, 0, 0}};
    if (f.one_pass) return f;
    if (lent > 0 && !fits) {      // (lent less than the one-pass kernel asks for: as without)
        f.split = bwd_split_plan(p);
        if (f.split.bytes > lent) f.split = {0, 0, 0, 0};
    }
    f.halves = !f.split.joins && bwd_halves(p, total_k);
    return f;
}

// Backward: host-side counterpart of mha_bwd / mha_varlen_bwd after tensor unpacking
// (flash_api.cpp:609-832, 834-1036) and of run_mha_bwd's dispatch (:587-607).
static int run_bwd(const fa_bwd_params* p, bool varlen, int64_t total_q, int64_t total_k, void* scratch, int64_t scratch_bytes, hipStream_t stream) {
    if (!p) return fail("params is NULL");
    if (!p->dout || !p->q || !p->k || !p->v || !p->out || !p->softmax_lse || !p->dq || !p->dk || !p->dv || !p->softmax_d)
        return fail("dout, q, k, v, out, softmax_lse, dq, dk, dv and softmax_d must be set");
    if (p->dtype != FA_DTYPE_FP16 && p->dtype != FA_DTYPE_BF16) return fail("FlashAttention only support fp16 and bf16 data type");
    if (p->b <= 0) return fail("batch size must be positive");
    if (p->d <= 0 || p->d > 256) return fail("FlashAttention backward only supports head dimension at most 256");
    if (p->d % 8 != 0) return fail("head_size should be a multiple of 8");
    if (p->h <= 0 || p->h_k <= 0 || p->h % p->h_k != 0) return fail("Number of heads in key/value must divide number of heads in query");
    if (p->seqlen_q < 0 || p->seqlen_k < 0) return fail("sequence lengths must be non-negative");
    if (p->seqlen_q_rounded < p->seqlen_q) return fail("seqlen_q_rounded must be at least seqlen_q");
    if (varlen && (!p->cu_seqlens_q || !p->cu_seqlens_k)) return fail("fa_varlen_bwd needs cu_seqlens_q and cu_seqlens_k");
    if (!varlen && (p->cu_seqlens_q || p->cu_seqlens_k)) return fail("fa_bwd takes dense batches; use fa_varlen_bwd");
    if (!(p->p_dropout >= 0.f && p->p_dropout < 1.f)) return fail("p_dropout must be in [0, 1)");
    if (p->p_dropout > 0.f && !p->rng_state) return fail("rng_state is required when p_dropout > 0");
    const int64_t strides[] = {p->q_row_stride, p->q_head_stride, p->k_row_stride, p->k_head_stride, p->v_row_stride,
                               p->v_head_stride, p->o_row_stride, p->o_head_stride, p->do_row_stride, p->do_head_stride,
                               p->dq_row_stride, p->dq_head_stride, p->dk_row_stride, p->dk_head_stride,
                               p->dv_row_stride, p->dv_head_stride, p->q_batch_stride, p->k_batch_stride, p->v_batch_stride,
                               p->o_batch_stride, p->do_batch_stride, p->dq_batch_stride, p->dk_batch_stride, p->dv_batch_stride};
    for (int64_t st : strides) if (st % 8 != 0) return fail("strides must be multiples of 8 elements (16-byte rows)");

    const void* ptrs[] = {p->dout, p->q, p->k, p->v, p->out, p->dq, p->dk, p->dv, scratch};
    for (const void* q : ptrs) if ((uintptr_t)q % 16 != 0) return fail("dout, q, k, v, out, dq, dk, dv and scratch must be 16-byte aligned");
    // the tile movers add a 32-bit lane byte offset (up to 128 rows) to a 64-bit tile base
    const int64_t row_strides[] = {p->q_row_stride, p->k_row_stride, p->v_row_stride, p->do_row_stride};
    for (int64_t st : row_strides) if (st < 0 || st >= ((int64_t)1 << 23)) return fail("row strides must be below 2^23 elements");

    BwdKParams kp;
    kp.p = *p;
    if (kp.p.is_causal) kp.p.window_right = 0;     // flash_api.cpp:627
    kp.p.window_left = window_bound(kp.p.window_left);
    kp.p.window_right = window_bound(kp.p.window_right);
    kp.has_left = kp.p.window_left >= 0;
    kp.has_right = kp.p.window_right >= 0;
    kp.scale_log2 = p->softmax_scale * (float)M_LOG2E;
    kp.slot_bytes = bwd_stream_slot_bytes(*p);
    kp.scratch = static_cast<char*>(scratch);
    const BwdForm form = bwd_form(*p, total_q, total_k, scratch ? scratch_bytes : 0);
    kp.one_pass = form.one_pass;
    kp.halves = form.halves;
    kp.split_steps = 0;
    if (form.split.joins) {
        kp.split_steps = form.split.steps;
        kp.split_pieces = form.split.pieces;
        kp.split_joins = form.split.joins;
        kp.split_counters = reinterpret_cast<int32_t*>(kp.scratch + 2 * form.split.joins * bwd_partial_bytes(bucket(p->d)));
    }
    const bool bf = p->dtype == FA_DTYPE_BF16;
    int e = 0;
    switch (bucket(p->d)) {
        case 64: e = bf ? launch_bwd_bf16_64(kp, stream) : launch_bwd_fp16_64(kp, stream); break;
        case 128: e = bf ? launch_bwd_bf16_128(kp, stream) : launch_bwd_fp16_128(kp, stream); break;
        default: e = bf ? launch_bwd_bf16_256(kp, stream) : launch_bwd_fp16_256(kp, stream); break;
    }
    if (e) return fail_hip(e, "backward kernel launch");
    g_last_bwd_kernel = kp.one_pass ? FA_BWD_KERNEL_ONE_PASS : FA_BWD_KERNEL_TWO_PASS;
    return 0;
}

}  // namespace fa

using namespace fa;

// ------------------------------------------------------------------------------------------------
// Device memory owned by the library, for the one entry point that must not allocate
// (fa_fwd_kvcache_noalloc): the ticket word, lse_accum and o_accum of a split launch live in this array
// instead of caller-provided buffers.  Every GPU the library runs on holds its own copy at its own
// address until the process ends; `scratch` itself is only the host-side name of the symbol, the
// address kernels may use is looked up once per device.
// ------------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[FA_NOALLOC_SCRATCH_BYTES];

static const int kMaxDevices = 64;
static void* g_scratch_ptr[kMaxDevices];          // device address of `scratch`, per device (0: not looked up yet)
static std::mutex g_scratch_mutex;

// address of the current device's copy of `scratch`, or nullptr (g_err says why)
static unsigned char* scratch_of_current_device() {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) { fail_hip((int)e, "hipGetDevice"); return nullptr; }
    if (dev < 0 || dev >= kMaxDevices) { fail("device index out of range for the no-allocation entry point"); return nullptr; }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));      // resolves the symbol on the CURRENT device
        if (e != hipSuccess || !ptr) { fail_hip((int)e, "hipGetSymbolAddress(scratch)"); return nullptr; }
        g_scratch_ptr[dev] = ptr;
    }
    return static_cast<unsigned char*>(g_scratch_ptr[dev]);
}

// A work list or order is written by one launch and read by the next.  Callers that lend the same words from several threads
// for launches on one stream must not get another thread's launch between the two: held while both are enqueued (one of 64, by
// the words, so that different words rarely wait for each other; the fast path of calls without a list takes none).
struct ListGuard {
    std::unique_lock<std::mutex> lock;
    ListGuard(const int32_t* words, bool list) {
        static std::mutex mutexes[64];
        if (list) lock = std::unique_lock<std::mutex>(mutexes[((uintptr_t)words >> 9) % 64]);
    }
};

static __global__ void set_rng_state_kernel(uint64_t* dst, uint64_t seed, uint64_t offset) {
    if (threadIdx.x == 0) { dst[0] = seed; dst[1] = offset; }
}

// fa_fwd_rng, fa_varlen_fwd_rng: the attention kernel writes the words (rng_publish), except where there is none to launch.
static void rng_words(KParams& kp, const uint64_t* rng) {
    if (!rng || kp.p.p_dropout <= 0.f) return;
    kp.rng_out = const_cast<uint64_t*>(kp.p.rng_state);
    kp.rng_seed = rng[0];
    kp.rng_offset = rng[1];
}
static int rng_words_only(const fa_fwd_params* p, const uint64_t* rng, void* hip_stream) {
    return rng && p->p_dropout > 0.f ? fa_set_rng_state(const_cast<uint64_t*>(p->rng_state), rng[0], rng[1], hip_stream) : 0;
}

extern "C" {

const char* fa_last_error(void) { return g_err.c_str(); }
int32_t fa_version(void) { return (0 << 16) | 1; }
int32_t fa_last_kernel(void) { return g_last_kernel; }

int32_t fa_last_bwd_kernel(void) { return g_last_bwd_kernel; }
int32_t fa_sizeof_params(void) { return (int32_t)sizeof(fa_fwd_params); }

int fa_num_splits_heuristic_reference(int32_t batch_nheads_mblocks, int32_t num_sms, int32_t num_n_blocks, int32_t max_splits) {
    if (batch_nheads_mblocks >= 0.8f * num_sms) return 1;
    max_splits = std::min({max_splits, num_sms, num_n_blocks});
    auto cdiv = [](int a, int b) { return (a + b - 1) / b; };
    auto eligible = [&](int s) { return s == 1 || cdiv(num_n_blocks, s) != cdiv(num_n_blocks, s - 1); };
    std::vector<float> eff(std::max(max_splits, 0) + 1, 0.f);
    float best = 0.f;
    for (int s = 1; s <= max_splits; s++) {
        if (!eligible(s)) continue;
        const float waves = float(batch_nheads_mblocks * s) / num_sms;
        eff[s] = waves / std::ceil(waves);
        best = std::max(best, eff[s]);
    }
    for (int s = 1; s <= max_splits; s++)
        if (eligible(s) && eff[s] >= 0.85f * best) return s;
    return 1;
}

int fa_plan_splits(const fa_fwd_params* p, int32_t api, int32_t* num_splits) {
    g_err.clear();
    if (int r = check_common(p)) return r;
    if (!num_splits) return fail("num_splits is NULL");
    if (api != 0 && api != 2) return fail("api must be 0 (fa_fwd) or 2 (fa_fwd_kvcache)");
    *num_splits = plan(*p, true).splits;
    return 0;
}

int64_t fa_work_list_words(const fa_fwd_params* p) {
    if (!p || p->h_k <= 0 || p->h <= 0 || p->h % p->h_k != 0) return FA_WORK_COUNTER_WORDS;
    const int64_t w = work_list_words(*p);
    return w > FA_WORK_COUNTER_WORDS ? w : FA_WORK_COUNTER_WORDS;
}

static int fwd(const fa_fwd_params* p, const uint64_t* rng, void* hip_stream) {
    if (int r = check_common(p)) return r;
    if (p->cu_seqlens_q || p->cu_seqlens_k) return fail("fa_fwd takes dense batches; use fa_varlen_fwd or fa_fwd_kvcache");
    if (p->k_new || p->v_new || p->rotary_cos || p->cache_batch_idx) return fail("fa_fwd does not append or rotate; use fa_fwd_kvcache");
    if (p->seqlen_q == 0) return rng_words_only(p, rng, hip_stream);
    KParams kp;
    fill_kparams(kp, *p);
    rng_words(kp, rng);
    kp.p.seqlen_knew = 0;
    kp.p.rotary_dim = 0;
    if (groups_as_rows(kp.p)) kp.has_right = 0;
    else kp.pack_g = positions_and_groups_as_rows(kp.p, &kp.pack_q_hs, &kp.pack_o_hs);
    if (int r = resolve_splits(kp, *p, true)) return r;
    return run_attention(kp, (hipStream_t)hip_stream);
}

static int varlen_fwd(const fa_fwd_params* p, const uint64_t* rng, void* hip_stream) {
    if (int r = check_common(p)) return r;
    if (!p->cu_seqlens_q || !p->cu_seqlens_k) return fail("cu_seqlens_q and cu_seqlens_k are required");
    if (!p->is_seqlens_k_cumulative) return fail("cu_seqlens_k must be cumulative for fa_varlen_fwd");
    if (p->k_new || p->v_new || p->rotary_cos || p->cache_batch_idx) return fail("fa_varlen_fwd does not append or rotate");
    if (p->seqlen_q == 0) return rng_words_only(p, rng, hip_stream);
    KParams kp;
    fill_kparams(kp, *p);
    rng_words(kp, rng);
    kp.p.seqlen_knew = 0;
    kp.p.rotary_dim = 0;
    kp.p.num_splits = 1;
    if (int r = resolve_splits(kp, kp.p, false)) return r;
    const ListGuard guard(p->work_counter, p->work_counter && p->work_counter_len > FA_WORK_COUNTER_WORDS);
    return run_attention(kp, (hipStream_t)hip_stream);
}

int fa_fwd(const fa_fwd_params* p, void* hip_stream) {
    g_err.clear();
    return fwd(p, nullptr, hip_stream);
}

int fa_fwd_rng(const fa_fwd_params* p, uint64_t seed, uint64_t offset, void* hip_stream) {
    g_err.clear();
    const uint64_t rng[2] = {seed, offset};
    return fwd(p, rng, hip_stream);
}

int fa_varlen_fwd(const fa_fwd_params* p, void* hip_stream) {
    g_err.clear();
    return varlen_fwd(p, nullptr, hip_stream);
}

int fa_varlen_fwd_rng(const fa_fwd_params* p, uint64_t seed, uint64_t offset, void* hip_stream) {
    g_err.clear();
    const uint64_t rng[2] = {seed, offset};
    return varlen_fwd(p, rng, hip_stream);
}

int fa_fwd_kvcache(const fa_fwd_params* p, void* hip_stream) {
    g_err.clear();
    if (int r = check_common(p)) return r;
    if (p->cu_seqlens_q) return fail("fa_fwd_kvcache takes a dense q batch");
    if (p->p_dropout != 0.f || p->s_dmask) return fail("fa_fwd_kvcache has no dropout");
    if (p->cu_seqlens_k && p->is_seqlens_k_cumulative) return fail("cache_seqlens must be per-batch lengths, not prefix sums");
    const bool has_new = p->k_new != nullptr;
    if (has_new) {
        if (!p->v_new) return fail("If key is supplied, value must also be passed in");
        if (!p->cu_seqlens_k) return fail("If key is supplied, seqlens_k must also be passed in");
        if (p->seqlen_knew <= 0) return fail("seqlen_knew must be positive when k_new is given");
        if (p->seqlen_q > p->seqlen_k) return fail("If key is supplied, it must have seqlen <= the seqlen of the KV cache");
    } else if (p->v_new) {
        return fail("If value is supplied, key must also be passed in");
    }
    if (p->rotary_cos || p->rotary_sin) {
        if (!has_new) return fail("If rotary cos/sin are provided, new key / value to be appended to KV cache must also be provided");
        if (!p->rotary_cos || !p->rotary_sin) return fail("If rotary cos is provided, rotary sin must also be provided");
        if (p->rotary_dim <= 0 || p->rotary_dim > p->d) return fail("rotary_dim must be <= headdim");
        if (p->rotary_dim % 16 != 0) return fail("Only rotary dimensions divisible by 16 are currently supported");
    }
    if (p->seqlen_q == 0) return 0;
    KParams kp;
    fill_kparams(kp, *p);
    if (!has_new) kp.p.seqlen_knew = 0;
    if (!p->rotary_cos) kp.p.rotary_dim = 0;
    kp.rotary_q = kp.p.rotary_dim > 0;
    // (q rotary: without a mask every row is rotated to the position of the first new token, as the one row was)
    if (groups_as_rows(kp.p)) kp.has_right = 0;
    else kp.pack_g = positions_and_groups_as_rows(kp.p, &kp.pack_q_hs, &kp.pack_o_hs);
    if (int r = resolve_splits(kp, *p, true)) return r;
    hipStream_t stream = (hipStream_t)hip_stream;
    // (of the call as it came: packed rows step over positions and heads)
    const int64_t o_span = span_elems(p->b, p->seqlen_q, p->h, p->d, p->o_batch_stride, p->o_row_stride, p->o_head_stride);
    // The decode kernels append the new rows themselves: the item that reaches them writes them, which saves a launch
    // (one chunk per workgroup, 1-13 caches of a few hundred keys: the call 30.6-32.1 -> 27.2-28.3 us).
    // The append stays a launch of its own, as for every other kernel,
    //  * with a left window bound: some new rows may lie outside every query's window and would not be visited;
    //  * where batch entries can share cache rows (cache_batch_idx may name one twice, a cache may be expanded over the
    //    batch): all rows are appended before any entry attends, and no workgroup waits for another one's stores;
    //  * where the kernel itself writes o (nothing is split) and o's memory meets that of k_new or v_new: a workgroup may
    //    write results over rows that another one has yet to append.
    const bool own_rows = (kp.p.b == 1 || !p->cache_batch_idx) &&
        rows_apart(kp.p.b, p->seqlen_k, p->h_k, p->d, p->k_batch_stride, p->k_row_stride, p->k_head_stride) &&
        rows_apart(kp.p.b, p->seqlen_k, p->h_k, p->d, p->v_batch_stride, p->v_row_stride, p->v_head_stride);
    const bool new_meets_o = has_new &&
        (spans_overlap(p->k_new, span_elems(kp.p.b, p->seqlen_knew, p->h_k, p->d, p->knew_batch_stride, p->knew_row_stride, p->knew_head_stride), kp.p.o, o_span) ||
         spans_overlap(p->v_new, span_elems(kp.p.b, p->seqlen_knew, p->h_k, p->d, p->vnew_batch_stride, p->vnew_row_stride, p->vnew_head_stride), kp.p.o, o_span));
    kp.dec_append = has_new && use_decode_kernel(kp.p) && !kp.has_left && own_rows && (kp.num_splits > 1 || !new_meets_o);
    const bool append = has_new && !kp.dec_append;
    // Every attention kernel rotates the q rows while it loads them.  The pipelined / ping-pong kernels read them from a rotated copy
    // before, which a pass of its own wrote to o: chunks of 512 tokens, 32 / 8 heads, d 128, batch 8 on caches of up to 16k 467-470
    // -> 462 us; 447 tokens, 64 / 8 heads, batch 36 on caches of 7-125 rows 411 -> 351; 163 tokens, 64 / 8 heads, batch 4 25.9 -> 20.3
    // (drawn calls, and the ones that lose: rotate_rows).  Where q's memory meets that of o the general kernel runs, and the tests of
    // such calls hold it to that.  With o == q that is a choice: the others too read only the rows that they write, before they write
    // any, and calls without rotary take them so.  Views of one tensor that meet otherwise are outside what the header allows.
    const bool disjoint = !kp.rotary_q || !spans_overlap(
        p->q, span_elems(p->b, p->seqlen_q, p->h, p->d, p->q_batch_stride, p->q_row_stride, p->q_head_stride), p->o, o_span);
    // (Few rows, which the plan left whole for waves that split the keys, run on those, or on the ping-pong kernel.)
    if (!disjoint && (kp.num_splits > 1 || prefill_key_waves(kp.p, kp.pack_g > 1, bucket(kp.p.d)) == 1)) kp.rotary_q = kRotaryTiled;
    const bool long_rows = kp.num_splits <= 1 && kp.pack_g <= 1 && !use_decode_kernel(kp.p) && disjoint && kp.p.seqlen_q >= prefill_long_rows(bucket(kp.p.d));
    // Caches of unequal length, in more than a round of workgroups: the row blocks of the longest first (xcd_cache_item).
    int32_t* order = nullptr;
    if (long_rows && cache_order_applies(kp.p) && p->work_counter && p->work_counter_len >= FA_WORK_COUNTER_WORDS + kp.p.b)
        order = p->work_counter + FA_WORK_COUNTER_WORDS;
    const ListGuard guard(order, order != nullptr);
    if (append || order) {
        if (int e = launch_prepare_rows(kp, append, order, stream)) return fail_hip(e, "append launch");
    }
    kp.cache_order = order;
    return run_attention(kp, stream);
}

// 17-32 packed rows up to head dim 128 whose split count is the library's to choose are launched whole where the partial results have no room: whichever
// kernel use_decode_kernel names, the same calls are taken (the decode kernel's plan stays within the room, the tickets of the tiled one may not).
static bool whole_where_no_room(const fa_fwd_params& p) {
    const int64_t rows = (int64_t)p.seqlen_q * (p.h / p.h_k);
    return p.num_splits == 0 && rows > 16 && rows <= 32 && p.d <= 128;
}

int fa_fwd_kvcache_noalloc(const fa_fwd_params* p, void* hip_stream) {
    g_err.clear();
    if (!p) return fail("params is NULL");
    unsigned char* base = scratch_of_current_device();
    if (!base) return 2;
    // layout inside the array: [0, kCounterBytes) the persistent decode kernel's counters (zero when the
    // library is loaded, left zero by every launch), then lse_accum, then o_accum (256-byte aligned)
    constexpr size_t kCounterBytes = 64u << 10;
    fa_fwd_params q = *p;
    q.work_counter = reinterpret_cast<int32_t*>(base);
    q.work_counter_len = (int32_t)(kCounterBytes / sizeof(int32_t));
    q.o_accum = nullptr;
    q.lse_accum = nullptr;
    if (int r = check_common(&q)) return r;
    const int splits = plan(q, q.p_dropout == 0.f).splits;
    if (splits > 1) {
        auto up256 = [](size_t x) { return (x + 255) / 256 * 256; };
        const size_t rows = (size_t)q.b * q.h * q.seqlen_q;
        const size_t lse_bytes = up256((size_t)splits * rows * sizeof(float));
        const size_t o_bytes = (size_t)splits * rows * (size_t)((q.d + 31) / 32 * 32) * sizeof(float);
        if (kCounterBytes + lse_bytes + o_bytes <= (size_t)FA_NOALLOC_SCRATCH_BYTES) {
            q.lse_accum = reinterpret_cast<float*>(base + kCounterBytes);
            q.o_accum = reinterpret_cast<float*>(base + kCounterBytes + lse_bytes);
        } else if (whole_where_no_room(q)) {
            q.num_splits = 1;
        } else {
            return fail("fa_fwd_kvcache_noalloc: the split accumulators of this problem exceed FA_NOALLOC_SCRATCH_BYTES; "
                        "use fa_fwd_kvcache with caller-provided o_accum / lse_accum, or request num_splits = 1");
        }
    }
    return fa_fwd_kvcache(&q, hip_stream);
}

int fa_set_rng_state(uint64_t* rng_state, uint64_t seed, uint64_t offset, void* hip_stream) {
    g_err.clear();
    if (!rng_state) return fail("rng_state is NULL");
    hipLaunchKernelGGL(set_rng_state_kernel, dim3(1), dim3(64), 0, (hipStream_t)hip_stream, rng_state, seed, offset);
    if (int e = (int)hipGetLastError()) return fail_hip(e, "rng state launch");
    return 0;
}

int32_t fa_sizeof_rotary_params(void) { return (int32_t)sizeof(fa_rotary_params); }

int fa_rotary(const fa_rotary_params* p, void* hip_stream) {
    g_err.clear();
    if (!p) return fail("null parameters");
    if (!p->x || !p->out || !p->cos || !p->sin) return fail("x, out, cos and sin are required");
    if (p->dtype != FA_DTYPE_FP16 && p->dtype != FA_DTYPE_BF16) return fail("rotary only supports fp16 and bf16 data");
    if (p->cs_dtype != FA_DTYPE_FP16 && p->cs_dtype != FA_DTYPE_BF16 && p->cs_dtype != FA_DTYPE_FP32) return fail("cos/sin must be fp16, bf16 or fp32");
    if (p->b < 0 || p->seqlen < 0 || p->h < 0 || p->d <= 0) return fail("negative size");
    if (p->rotary_dim <= 0 || p->rotary_dim > p->d) return fail("rotary_dim must be <= headdim");
    if (p->rotary_dim % 2 != 0) return fail("rotary_dim must be even");
    if (p->seqlen_ro < 0) return fail("negative table length");
    // (16-byte granules when rotary_dim is a multiple of 16, the head dim and all strides multiples of 8 elements
    // and the pointers 16-byte aligned; anything else takes the element-wise kernel)
    if (int e = launch_rotary(*p, (hipStream_t)hip_stream)) return fail_hip(e, "rotary kernel launch");
    return 0;
}

int64_t fa_bwd_scratch_bytes(const fa_bwd_params* p, int64_t total_q, int64_t total_k) {
    return p && bwd_one_pass_fits(*p, total_q, total_k) ? bwd_stream_slot_bytes(*p) * bwd_stream_slots(*p) : 0;
}

int64_t fa_bwd_lend_bytes(const fa_bwd_params* p, int64_t total_q, int64_t total_k) {
    if (!p) return 0;
    return bwd_one_pass_fits(*p, total_q, total_k) ? bwd_stream_slot_bytes(*p) * bwd_stream_slots(*p) : bwd_split_plan(*p).bytes;
}

int32_t fa_bwd_plan_form(const fa_bwd_params* p, int64_t total_q, int64_t total_k, int64_t scratch_bytes) {
    if (!p || p->b <= 0 || p->h <= 0 || p->h_k <= 0 || p->h % p->h_k != 0 || p->d <= 0 || p->d > 256 || p->seqlen_q <= 0 || p->seqlen_k <= 0) return FA_BWD_FORM_NONE;
    const BwdForm f = bwd_form(*p, total_q, total_k, scratch_bytes);
    return f.one_pass ? FA_BWD_FORM_ONE_PASS : f.split.joins ? FA_BWD_FORM_PARTS : f.halves ? FA_BWD_FORM_HALVES : FA_BWD_FORM_WHOLE;
}

int32_t fa_sizeof_bwd_params(void) { return (int32_t)sizeof(fa_bwd_params); }

int fa_bwd(const fa_bwd_params* p, void* hip_stream) {
    g_err.clear();
    return run_bwd(p, false, 0, 0, nullptr, 0, (hipStream_t)hip_stream);
}

int fa_varlen_bwd(const fa_bwd_params* p, void* hip_stream) {
    g_err.clear();
    return run_bwd(p, true, 0, 0, nullptr, 0, (hipStream_t)hip_stream);
}

int fa_bwd_lent(const fa_bwd_params* p, int64_t total_q, int64_t total_k, void* scratch, int64_t scratch_bytes, void* hip_stream) {
    g_err.clear();
    return run_bwd(p, p && p->cu_seqlens_q, total_q, total_k, scratch, scratch_bytes, (hipStream_t)hip_stream);
}

}  // extern "C"
