// Small memory-bound kernels around the attention kernels:
//  * combine: log-sum-exp weighted merge of split-KV partials
//    (reference: combine_attn_seqk_parallel, csrc/flash_attn/src/flash_fwd_kernel.h:1169-1327);
//  * prepare_rows: copy of k_new / v_new (new keys rotated) into the cache rows
//    [cache_seqlens[b], cache_seqlens[b] + seqlen_knew) of cache row cache_batch_idx[b]
//    (reference: the Append_KV prologue, flash_fwd_kernel.h:763-852, copy_w_min_idx /
//    copy_rotary_* in csrc/flash_attn/src/utils.h:358-517).
#include <algorithm>
#include "fa_common.h"
#include "fa_launch.h"

namespace fa {

// L lanes per output row (b, h, i): combine_row (fa_common.h).
template <typename T, int L>
__global__ void __launch_bounds__(256) combine_kernel(const KParams kp) {
    const int64_t nrows = (int64_t)kp.p.b * kp.p.h * kp.p.seqlen_q;
    const int64_t row = (int64_t)blockIdx.x * (256 / L) + threadIdx.x / L;
    // (lanes past the end read the last row again, and leave it alone)
    combine_row<T, L>(kp, min(row, nrows - 1), threadIdx.x & 63, row < nrows);
}

int launch_combine(const KParams& kp, hipStream_t stream) {
    const int64_t nrows = (int64_t)kp.p.b * kp.p.h * kp.p.seqlen_q;
    if (nrows == 0) return 0;
    auto launch = [&](auto lanes) {
        constexpr int L = decltype(lanes)::value;
        const dim3 grid((unsigned)((nrows + 256 / L - 1) / (256 / L))), block(256);
        if (kp.p.dtype == FA_DTYPE_BF16) hipLaunchKernelGGL((combine_kernel<__bf16, L>), grid, block, 0, stream, kp);
        else hipLaunchKernelGGL((combine_kernel<_Float16, L>), grid, block, 0, stream, kp);
    };
    if (kp.d_rounded <= 64) launch(std::integral_constant<int, 16>());
    else if (kp.d_rounded <= 128) launch(std::integral_constant<int, 32>());
    else launch(std::integral_constant<int, 64>());
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------------------------------
// Work list of a packed (variable-length) forward launch.
//
// The hardware hands the workgroups that fall to an XCD to its 4 shader engines in strict rotation and in
// order (see xcd_stream_unit).  The arithmetic order of packed batches cannot follow that rule well: it
// does not know the lengths, so the row blocks a short sequence does not have are empty workgroups in the
// middle of the order, and streams of unequal length run side by side.  This kernel reads cu_seqlens_q on
// the device and writes, per XCD, the list the attention kernel then walks: sequences by falling length
// (so neighbouring streams cost about the same), four streams at a time, row block by row block from the
// last (heaviest under a causal mask) down, and nothing for row blocks that do not exist.  The slots of
// the grid past the end of a list exit at once, after all work has been handed out.
// XCD x owns q heads of kv-head parts x, x + 8, ... of every sequence (h_k * parts is a multiple of 8), as
// in the arithmetic order.  One workgroup per XCD.
// ------------------------------------------------------------------------------------------------
struct WorkListParams {
    const int32_t* cu_seqlens_q;
    int32_t b, h_k, G, parts, block_m, nmb, per_xcd;
    int32_t* out;            // kWorkListHeaderWords counts, then 8 lists of per_xcd two-word slots
};
__global__ void __launch_bounds__(1024) work_list_kernel(const WorkListParams w) {
    __shared__ int len_s[kWorkListMaxBatch];
    __shared__ int order_s[kWorkListMaxBatch];       // rank -> batch index
    __shared__ int scan_s[256];
    const int x = blockIdx.x, t = threadIdx.x, nb = w.b;
    for (int i = t; i < nb; i += 1024) len_s[i] = max(w.cu_seqlens_q[i + 1] - w.cu_seqlens_q[i], 0);
    __syncthreads();
    for (int i = t; i < nb; i += 1024) {
        const int li = len_s[i];
        int r = 0;
        for (int j = 0; j < nb; j++) r += (len_s[j] > li || (len_s[j] == li && j < i)) ? 1 : 0;
        order_s[r] = i;
    }
    __syncthreads();
    const int Gp = w.G / w.parts, E = (w.h_k * w.parts / 8) * Gp;     // streams per sequence on this XCD
    const int ns = nb * E, ng = (ns + 3) / 4;
    // (a length beyond the seqlen_q the grid was sized for is the caller's error; it must not overrun the list)
    auto units = [&](int s) { return s < ns ? min((len_s[order_s[s / E]] + w.block_m - 1) / w.block_m, w.nmb) : 0; };
    // Four threads per owner: owner o holds groups [o * gpt, (o + 1) * gpt), thread j of it writes stream j of
    // each.  Items before an owner's groups: inclusive scan over the owners' totals.
    const int o = t >> 2, jj = t & 3;
    const int gpt = (ng + 255) / 256;
    const int g_lo = min(o * gpt, ng), g_hi = min(g_lo + gpt, ng);
    int mine = 0;
    for (int g = g_lo; g < g_hi; g++) mine += units(4 * g) + units(4 * g + 1) + units(4 * g + 2) + units(4 * g + 3);
    if (jj == 0) scan_s[o] = mine;
    __syncthreads();
    const int owners = min(256, (ng + gpt - 1) / gpt);      // owners with work; the others hold zero
    for (int d = 1; d < owners; d <<= 1) {
        const int v = (jj == 0 && o >= d) ? scan_s[o - d] : 0;
        __syncthreads();
        if (jj == 0) scan_s[o] += v;
        __syncthreads();
    }
    int off = scan_s[o] - mine;
    if (t == 0) w.out[x] = owners > 0 ? scan_s[owners - 1] : 0;
    int32_t* list = w.out + kWorkListHeaderWords + (size_t)x * w.per_xcd * 2;
    for (int g = g_lo; g < g_hi; g++) {
        int u[4];
        for (int j = 0; j < 4; j++) u[j] = units(4 * g + j);
        const int s = 4 * g + jj;
        if (s < ns) {
            const int bb = order_s[s / E], e = s % E;
            const int hkp = x + 8 * (e / Gp);
            const int head = (hkp / w.parts) * w.G + (hkp % w.parts) * Gp + e % Gp;
            const int mine_u = u[jj];
            for (int un = 0; un < mine_u; un++) {
                // unit-major inside the group; lengths fall with the stream index, so the streams that still
                // have unit `un` are a prefix of the group
                const int pos = off + min(u[0], un) + min(u[1], un) + min(u[2], un) + min(u[3], un) + jj;
                list[2 * pos] = bb;
                list[2 * pos + 1] = (int32_t)(((uint32_t)head << 16) | (uint32_t)(mine_u - 1 - un));
            }
        }
        off += u[0] + u[1] + u[2] + u[3];
    }
}

static bool work_list_applies(const fa_fwd_params& p) {
    if (!p.cu_seqlens_q || p.b <= 0 || p.b > kWorkListMaxBatch || p.h >= 65536) return false;
    const uint32_t G = (uint32_t)(p.h / p.h_k), parts = xcd_parts(true, true, (uint32_t)p.h_k, G);
    return ((uint32_t)p.h_k * parts) % 8u == 0u;
}
int64_t work_list_words(const fa_fwd_params& p) {
    if (cache_order_applies(p) && p.seqlen_q >= prefill_long_rows(p.d <= 128 ? 128 : 256)) return FA_WORK_COUNTER_WORDS + p.b;
    // (key waves: no more than a workgroup per CU, all at once whatever their order)
    if (!work_list_applies(p) || prefill_key_waves(p, false, p.d <= 64 ? 64 : p.d <= 128 ? 128 : 256) > 1) return 0;
    // the smallest row block of the kernels that take one (128 rows) gives the longest lists
    const int64_t nmb = (p.seqlen_q + 127) / 128;
    return FA_WORK_COUNTER_WORDS + kWorkListHeaderWords + 2 * xcd_rows_grid(true, p.cu_seqlens_q != nullptr, p.b, p.h_k, p.h / p.h_k, nmb);
}
int prepare_work_list(KParams& kp, int block_m, int64_t nblocks, hipStream_t stream) {
    const fa_fwd_params& p = kp.p;
    kp.work_items = nullptr;
    if (!work_list_applies(p) || !kp.work_counter || nblocks <= 0 || (nblocks & 7) != 0) return 0;
    if ((p.seqlen_q + block_m - 1) / block_m >= 65536) return 0;
    if ((int64_t)p.work_counter_len < FA_WORK_COUNTER_WORDS + kWorkListHeaderWords + 2 * nblocks) return 0;
    WorkListParams w;
    w.cu_seqlens_q = p.cu_seqlens_q;
    w.b = p.b; w.h_k = p.h_k; w.G = p.h / p.h_k;
    w.parts = (int32_t)xcd_parts(true, true, (uint32_t)p.h_k, (uint32_t)w.G);
    w.block_m = block_m;
    w.nmb = (p.seqlen_q + block_m - 1) / block_m;
    w.per_xcd = (int32_t)(nblocks / 8);
    w.out = kp.work_counter + FA_WORK_COUNTER_WORDS;
    hipLaunchKernelGGL(work_list_kernel, dim3(8), dim3(1024), 0, stream, w);
    if (int e = (int)hipGetLastError()) return e;
    kp.work_items = w.out;
    return 0;
}

// What a kv-cache call needs done to its rows before the attention kernel, in one launch; each part is optional.
//  * append: k_new (rotated) and v_new into the cache rows behind the cached keys;
//  * order: the batch indices by falling cache length (ties by index), for xcd_cache_item (fa_common.h).
// Blocks: `order_blocks` that rank, then per batch entry `append_blocks` of whole token rows.  HBM-bound.  32-bit index arithmetic
// inside a block.  A thread of a large launch loads four chunks before it uses any; where that would leave CUs without a block,
// one (with four a chunk of 132 tokens, batch 24, 8 / 1 heads took 11.1 us).  The attention kernels rotate q while they load it.
struct PrepRows { int32_t order_blocks, append_blocks, append_rows; int32_t* order; };

// Chunks of 8 elements at d0[j] of the rows src[j], rotated to pos[j], to dst[j] where ok[j]; all of them loaded before any is
// used.  Same arithmetic as rotary8; columns past rotary_dim are copied.
template <typename T, int N>
FA_DEV void rotate_chunks(const KParams& kp, const T* const (&src)[N], T* const (&dst)[N], const int (&d0)[N], const int (&pos)[N], const bool (&ok)[N]) {
    const fa_fwd_params& p = kp.p;
    const int rd = p.rotary_dim, half = rd / 2;
    u32x4 raw[N];
    if (rd == 0) {
#pragma unroll
        for (int j = 0; j < N; j++) raw[j] = ld_global16(src[j] + d0[j]);
    } else if (p.is_rotary_interleaved) {
        u32x2_any c[N], s[N];
#pragma unroll
        for (int j = 0; j < N; j++) {
            raw[j] = ld_global16(src[j] + d0[j]);
            const int64_t at = (int64_t)pos[j] * half + (d0[j] < rd ? d0[j] / 2 : 0);
            c[j] = *reinterpret_cast<const u32x2_any*>(reinterpret_cast<const T*>(p.rotary_cos) + at);
            s[j] = *reinterpret_cast<const u32x2_any*>(reinterpret_cast<const T*>(p.rotary_sin) + at);
        }
#pragma unroll
        for (int j = 0; j < N; j++) {
            float x[8], c8[8], s8[8];
            unpack8<T>(raw[j], x);
            unpack8<T>((u32x4){c[j][0], c[j][1], 0, 0}, c8);
            unpack8<T>((u32x4){s[j][0], s[j][1], 0, 0}, s8);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float x0 = x[2 * e], x1 = x[2 * e + 1];
                x[2 * e] = x0 * c8[e] - x1 * s8[e];
                x[2 * e + 1] = x0 * s8[e] + x1 * c8[e];
            }
            if (d0[j] < rd) raw[j] = pack8<T>(x);
        }
    } else {
        u32x4 praw[N];
        u32x4_any c[N], s[N];
#pragma unroll
        for (int j = 0; j < N; j++) {
            raw[j] = ld_global16(src[j] + d0[j]);
            praw[j] = ld_global16(src[j] + (d0[j] >= rd ? d0[j] : d0[j] < half ? d0[j] + half : d0[j] - half));
            const int64_t at = (int64_t)pos[j] * half + (d0[j] >= rd ? 0 : d0[j] < half ? d0[j] : d0[j] - half);
            c[j] = *reinterpret_cast<const u32x4_any*>(reinterpret_cast<const T*>(p.rotary_cos) + at);
            s[j] = *reinterpret_cast<const u32x4_any*>(reinterpret_cast<const T*>(p.rotary_sin) + at);
        }
#pragma unroll
        for (int j = 0; j < N; j++) {
            float x[8], y[8], c8[8], s8[8];
            unpack8<T>(raw[j], x);
            unpack8<T>(praw[j], y);
            unpack8<T>((u32x4)c[j], c8);
            unpack8<T>((u32x4)s[j], s8);
#pragma unroll
            for (int e = 0; e < 8; e++) x[e] = d0[j] < half ? (x[e] * c8[e] - y[e] * s8[e]) : (x[e] * c8[e] + y[e] * s8[e]);
            if (d0[j] < rd) raw[j] = pack8<T>(x);
        }
    }
#pragma unroll
    for (int j = 0; j < N; j++)
        if (ok[j]) st_global16(dst[j] + d0[j], raw[j]);
}

// N: chunks of a thread in flight
template <typename T, int N>
__global__ void __launch_bounds__(256) prepare_rows_kernel(const KParams kp, const PrepRows w) {
    const fa_fwd_params& p = kp.p;
    const int tid = threadIdx.x;
    uint32_t blk = blockIdx.x;
    if (blk < (uint32_t)w.order_blocks) {
        __shared__ int len_s[kWorkListMaxBatch];
        const int nb = p.b;
        for (int i = tid; i < nb; i += 256) len_s[i] = p.cu_seqlens_k[i];
        __syncthreads();
        const int i = (int)blk * 256 + tid;
        if (i >= nb) return;
        const int li = len_s[i];
        int r = 0;
        for (int j = 0; j < nb; j++) r += (len_s[j] > li || (len_s[j] == li && j < i)) ? 1 : 0;
        w.order[r] = i;
        return;
    }
    blk -= (uint32_t)w.order_blocks;
    const int b = (int)(blk / (uint32_t)w.append_blocks);
    const uint32_t x = blk % (uint32_t)w.append_blocks, cpr = (uint32_t)p.d / 8u;
    const SeqInfo si = seq_info(p, b);
    // (rows past the cache capacity are never written)
    const int t0 = (int)x * w.append_rows;
    const int rows = min(min(w.append_rows, p.seqlen_knew - t0), p.seqlen_k - (si.sk_cache + t0));
    const uint32_t per_row = cpr * (uint32_t)p.h_k, n = (uint32_t)max(rows, 0) * per_row;
    for (uint32_t base = (uint32_t)tid; base < n; base += 256u * N) {
        const T *ks[N], *vs[N];
        T *kd[N], *vd[N];
        int d0[N], pos[N];
        bool ok[N];
        u32x4 v[N];
#pragma unroll
        for (int j = 0; j < N; j++) {
            const uint32_t idx = min(base + 256u * (uint32_t)j, n - 1u), tr = idx / per_row, rest = idx % per_row;
            const int t = t0 + (int)tr, hk = (int)(rest / cpr);
            ok[j] = base + 256u * (uint32_t)j < n;
            d0[j] = (int)(rest % cpr) * 8;
            pos[j] = si.sk_cache + t;
            ks[j] = reinterpret_cast<const T*>(p.k_new) + (int64_t)b * p.knew_batch_stride + (int64_t)t * p.knew_row_stride + (int64_t)hk * p.knew_head_stride;
            vs[j] = reinterpret_cast<const T*>(p.v_new) + (int64_t)b * p.vnew_batch_stride + (int64_t)t * p.vnew_row_stride + (int64_t)hk * p.vnew_head_stride;
            kd[j] = reinterpret_cast<T*>(const_cast<void*>(p.k)) + si.k_off + (int64_t)pos[j] * p.k_row_stride + (int64_t)hk * p.k_head_stride;
            vd[j] = reinterpret_cast<T*>(const_cast<void*>(p.v)) + si.v_off + (int64_t)pos[j] * p.v_row_stride + (int64_t)hk * p.v_head_stride;
            v[j] = ld_global16(vs[j] + d0[j]);
        }
#pragma unroll
        for (int j = 0; j < N; j++)
            if (ok[j]) st_global16(vd[j] + d0[j], v[j]);
        rotate_chunks<T, N>(kp, ks, kd, d0, pos, ok);
    }
}

int launch_prepare_rows(const KParams& kp, bool append, int32_t* order, hipStream_t stream) {
    const fa_fwd_params& p = kp.p;
    PrepRows w = {0, 0, 1, order};
    if (order) w.order_blocks = (p.b + 255) / 256;
    // whole token rows; four chunks of 16 bytes per thread where that leaves blocks enough for the CUs, one otherwise
    const int64_t per_row = (int64_t)p.h_k * (p.d / 8), chunks = append ? (int64_t)p.b * p.seqlen_knew * per_row : 0;
    const int64_t per_block = chunks >= (int64_t)2048 * 1024 ? 1024 : 256;
    if (append && p.seqlen_knew > 0) {
        w.append_rows = (int32_t)std::max<int64_t>(1, per_block / std::max<int64_t>(1, per_row));
        w.append_blocks = (p.seqlen_knew + w.append_rows - 1) / w.append_rows;
    }
    const int64_t blocks = w.order_blocks + (int64_t)p.b * w.append_blocks;
    if (blocks == 0) return 0;
    if (blocks > 0x7fffffffLL) return -2;
    dim3 grid((unsigned)blocks), block(256);
    const bool bf = p.dtype == FA_DTYPE_BF16, four = per_block > 256;
    auto kern = bf ? (four ? prepare_rows_kernel<__bf16, 4> : prepare_rows_kernel<__bf16, 1>)
                   : (four ? prepare_rows_kernel<_Float16, 4> : prepare_rows_kernel<_Float16, 1>);
    hipLaunchKernelGGL(kern, grid, block, 0, stream, kp, w);
    return (int)hipGetLastError();
}

bool cache_order_applies(const fa_fwd_params& p) {
    if (p.cu_seqlens_q || !p.cu_seqlens_k || p.is_seqlens_k_cumulative || p.b < 2 || p.b > kWorkListMaxBatch) return false;
    const uint32_t G = (uint32_t)(p.h / p.h_k), parts = xcd_parts(true, true, (uint32_t)p.h_k, G);
    // (up to 256 row blocks, of 128 rows: a workgroup per CU at most, in any order)
    return ((uint32_t)p.h_k * parts) % 8u == 0u && (int64_t)((p.seqlen_q + 127) / 128) * p.h * p.b > 256;
}

// Testing aid behind return_softmax (the reference's S_dmask, csrc/flash_attn/flash_api.cpp:351-357):
// s_dmask[b, h, i, j] = exp(scale q_i . k_j - lse_i), negated where dropout removed the entry, 0 where
// the mask hides it or outside (seqlen_q, seqlen_k).  Runs after the attention kernel, so lse is
// final and the value is the normalised probability.  One thread per entry, scalar dot product.
template <typename T>
__global__ void __launch_bounds__(256) attn_probs_kernel(const KParams kp) {
    const fa_fwd_params& p = kp.p;
    const int b = blockIdx.z / p.h, head = blockIdx.z % p.h;
    const int i = blockIdx.y * 16 + (threadIdx.x >> 4);
    const int j = blockIdx.x * 16 + (threadIdx.x & 15);
    if (i >= p.sdm_rows || j >= p.sdm_cols) return;
    const SeqInfo si = seq_info(p, b);
    const int hk = head / (p.h / p.h_k);
    const int shift = si.sk - si.sq;
    bool vis = i < si.sq && j < si.sk;
    if (kp.has_right) vis = vis && j <= i + shift + p.window_right;
    if (kp.has_left) vis = vis && j >= i + shift - p.window_left;
    float val = 0.f;
    if (vis) {
        const T* q = reinterpret_cast<const T*>(p.q) + si.q_off + (int64_t)i * p.q_row_stride + (int64_t)head * p.q_head_stride;
        const T* k = reinterpret_cast<const T*>(p.k) + si.k_off + (int64_t)j * p.k_row_stride + (int64_t)hk * p.k_head_stride;
        float dot = 0.f;
        for (int c = 0; c < p.d; c += 8) {
            float a[8], bb[8];
            unpack8<T>(ld_global16(q + c), a);
            unpack8<T>(ld_global16(k + c), bb);
#pragma unroll
            for (int e = 0; e < 8; e++) dot += a[e] * bb[e];
        }
        const float lse = p.softmax_lse[((int64_t)b * p.h + head) * p.seqlen_q + i];
        val = __expf(dot * p.softmax_scale - lse);
        if (p.p_dropout > 0.f) {
            const Drop drop = drop_init(p.rng_state, p.p_dropout, b, head, p.h);
            if (!drop_keep(drop, i, j)) val = -val;
        }
    }
    reinterpret_cast<T*>(p.s_dmask)[(((int64_t)b * p.h + head) * p.sdm_rows + i) * p.sdm_cols + j] = (T)val;
}

int launch_attn_probs(const KParams& kp, hipStream_t stream) {
    const fa_fwd_params& p = kp.p;
    if (p.sdm_rows <= 0 || p.sdm_cols <= 0) return 0;
    dim3 grid((unsigned)((p.sdm_cols + 15) / 16), (unsigned)((p.sdm_rows + 15) / 16), (unsigned)(p.b * p.h));
    if (p.dtype == FA_DTYPE_BF16) hipLaunchKernelGGL(attn_probs_kernel<__bf16>, grid, dim3(256), 0, stream, kp);
    else hipLaunchKernelGGL(attn_probs_kernel<_Float16>, grid, dim3(256), 0, stream, kp);
    return (int)hipGetLastError();
}


}  // namespace fa
