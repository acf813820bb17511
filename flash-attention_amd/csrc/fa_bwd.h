// Backward kernels for gfx950: dQ by one pass over query tiles, dK / dV by one pass over key tiles (short sequences at head
// dims up to 64: one pass, fa_bwd_stream.h).
// Counterpart of the reference's compute_dq_dk_dv_1colblock (csrc/flash_attn/src/flash_bwd_kernel.h:
// 79-780) and its dot_do_o / convert_dQ passes (flash_bwd_preprocess_kernel.h), re-designed so that
// nothing is accumulated through global atomics and no fp32 dq buffer exists:
//
//   D_i   = sum_d dO[i,d] O[i,d]                                   (the dQ pass)
//   P     = exp(scale * Q K^T - lse),   dP = dO V^T,   dS = P o (dP - D)
//   dQ    = scale * dS K                                           (bwd_dq_kernel / bwd_dq2_kernel: per query tile)
//   dV    = P^T dO,   dK = scale * dS^T Q                          (bwd_dkv3_kernel: per key tile)
//
// All keep the forward kernels' register geometry: every product is computed TRANSPOSED with
// v_mfma_f32_32x32x16 so that the accumulator gives each lane ONE row of the resident operand (a
// query row in the dQ kernel, a key row in the dK/dV kernel) and 16 rows of the streamed tile; the
// accumulator layout is then already the B-operand layout of the next product, so P and dS never
// leave registers.  Streamed tiles are read from LDS twice, row-wise (ds_read_b128) as the A operand
// of the score-shaped products and transposed (ds_read_b64_tr_b16) as the A operand of the
// gradient-shaped ones; one swizzle (swz_u) keeps both conflict free.  The sum of dK / dV over the
// query heads of a GQA group is a loop inside the key-tile kernel.
#pragma once
#include "fa_common.h"

namespace fa {

struct BwdKParams {
    fa_bwd_params p;
    float scale_log2;             // softmax_scale * log2(e)
    int32_t has_left, has_right;  // window bounds active (after causal normalisation)
    bool one_pass;                // the one-pass kernel runs (fa_bwd_stream.h)
    char* scratch;                // its scratch, slot_bytes per workgroup
    int64_t slot_bytes;
    // dK/dV pass of a dense batch: key blocks of more than split_steps steps (0: none) are cut in parts, a workgroup each; a
    // (batch, kv head) has split_pieces parts, and partial sums meet in scratch (join_parts)
    int32_t split_steps, split_pieces;
    int32_t* split_counters;      // one for each join, zeroed by the dQ pass
    int64_t split_joins;
    bool halves;                  // two workgroups share a key block of that pass, half of the head dimension each
};

constexpr int kBwdKeyBlock = 128;        // keys of a dK/dV workgroup
// query rows per dK/dV step: at head dim 64 a 64-row step holds too few products to cover its fixed cost (tile requests,
// barrier), and the fp16 hand-over leaves room for 128 rows
constexpr __host__ __device__ int bwd_dkv_rows(int D) { return D == 64 ? 128 : D == 128 ? 64 : 32; }
// steps of a key block: the tiles of BM query rows (first t_lo) that see any of its keys, of each of the G grouped heads
__host__ __device__ inline int bwd_block_tiles(int n0, int sq, int sk, bool has_left, int wl, bool has_right, int wr, int BM, int& t_lo) {
    const int shift = sk - sq, end = n0 + kBwdKeyBlock < sk ? n0 + kBwdKeyBlock : sk;
    int lo = 0, hi = sq;
    if (has_right && n0 - shift - wr > 0) lo = n0 - shift - wr;
    if (has_left && end - shift + wl < hi) hi = end - shift + wl;
    t_lo = lo / BM;
    return hi > lo ? (hi + BM - 1) / BM - t_lo : 0;
}
// parts of a key block of n steps
constexpr int kBwdMaxParts = 16;
__host__ __device__ inline int bwd_block_parts(int n, int split_steps) {
    if (n <= split_steps) return 1;
    const int parts = (n + split_steps - 1) / split_steps;
    return parts < kBwdMaxParts ? parts : kBwdMaxParts;
}
// partial sums of one part, fp32; a block of n parts has room for 2n - 2
constexpr __host__ __device__ int64_t bwd_partial_bytes(int D) { return (int64_t)kBwdKeyBlock * D * 2 * 4; }

// The kernel's arguments through a pointer of unknown value: read where they are used.  (Read the ordinary way all of them
// stay in scalar registers across the loops, which spill to lanes of vector registers: two thousand cycles per step of the
// one-pass kernel, which spills 57-67 as it is.)
typedef const __attribute__((address_space(4))) BwdKParams* BwdArgs;
FA_DEV BwdArgs fresh_bwd_args() {
    uint64_t a = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return (BwdArgs)a;
}

struct BwdSeq {
    int sq, sk;
    int64_t q_off, k_off, v_off, o_off, do_off, dq_off, dk_off, dv_off;   // element offsets of (row 0, head 0)
};
FA_DEV BwdSeq bwd_seq(const fa_bwd_params& p, int b) {
    BwdSeq s;
    if (p.cu_seqlens_q) {
        const int64_t r0 = p.cu_seqlens_q[b];
        s.sq = p.cu_seqlens_q[b + 1] - (int)r0;
        s.q_off = r0 * p.q_row_stride; s.o_off = r0 * p.o_row_stride;
        s.do_off = r0 * p.do_row_stride; s.dq_off = r0 * p.dq_row_stride;
    } else {
        s.sq = p.seqlen_q;
        s.q_off = (int64_t)b * p.q_batch_stride; s.o_off = (int64_t)b * p.o_batch_stride;
        s.do_off = (int64_t)b * p.do_batch_stride; s.dq_off = (int64_t)b * p.dq_batch_stride;
    }
    if (p.cu_seqlens_k) {
        const int64_t r0 = p.cu_seqlens_k[b];
        s.sk = p.cu_seqlens_k[b + 1] - (int)r0;
        s.k_off = r0 * p.k_row_stride; s.v_off = r0 * p.v_row_stride;
        s.dk_off = r0 * p.dk_row_stride; s.dv_off = r0 * p.dv_row_stride;
    } else {
        s.sk = p.seqlen_k;
        s.k_off = (int64_t)b * p.k_batch_stride; s.v_off = (int64_t)b * p.v_batch_stride;
        s.dk_off = (int64_t)b * p.dk_batch_stride; s.dv_off = (int64_t)b * p.dv_batch_stride;
    }
    return s;
}

// ------------------------------------------------------------------------------------------------
// D_i = rowsum(dO o O), formed by the dQ pass, whose lanes hold their row of dO anyway (a half of it each: pieces of 8 columns,
// every other one).  A pass of its own read dO and O once more and was a launch that short calls waited for: backward alone, bf16, 33 x 226,
// d 96 99.4 -> 92.9 us, 3 x 1299, 32 heads, d 128 204.5 -> 195.5, 1 x 311, 8 heads, d 64 22.2 -> 20.7.  Long calls take what they took (2 x 8k causal,
// 16 heads, d 128: a launch of 35 us less, the dQ pass 9 longer, no difference in the call beyond that of two runs; 4 x 2039, 16 / 4 heads, d 256: 22 and 14).
// ------------------------------------------------------------------------------------------------
template <typename T, int KS, class V8>
FA_DEV float bwd_row_dot(const fa_bwd_params& p, const BwdSeq& si, int head, int row, bool row_ok, int hh, const V8 (&gf)[KS]) {
    const T* orow = reinterpret_cast<const T*>(p.out) + si.o_off + (int64_t)row * p.o_row_stride + (int64_t)head * p.o_head_stride;
    u32x4 raw[KS];
#pragma unroll
    for (int dk = 0; dk < KS; dk++) {
        const int d0 = dk * 16 + 8 * hh;
        raw[dk] = u32x4{0, 0, 0, 0};
        if (row_ok && d0 < p.d) raw[dk] = ld_global16(orow + d0);
    }
    float acc = 0.f;
#pragma unroll
    for (int dk = 0; dk < KS; dk++) {
        float o8[8], g8[8];
        unpack8<T>(raw[dk], o8);
        unpack8<T>(__builtin_bit_cast(u32x4, gf[dk]), g8);
#pragma unroll
        for (int e = 0; e < 8; e++) acc += o8[e] * g8[e];
    }
    return xhalf_sum(acc);
}
// What the dQ pass does beside dQ ahead of the dK/dV pass: D of the rows of a row block that the sequence does not have (the last
// block's up to the pitch of softmax_d), and the arrival counters of cut key blocks, by all threads of the launch.
FA_DEV void bwd_clear_counters(const BwdKParams& kp) {
    if (kp.split_steps) {
        const int64_t stride = (int64_t)gridDim.x * blockDim.x;
        for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < kp.split_joins; i += stride) kp.split_counters[i] = 0;
    }
}
FA_DEV void bwd_pad_d(const fa_bwd_params& p, int b, int head, int m0, int sq, bool last) {
    float* sd = p.softmax_d + ((int64_t)b * p.h + head) * p.seqlen_q_rounded;
    const int end = last ? p.seqlen_q_rounded : min(m0 + 128, p.seqlen_q_rounded);
    for (int row = max(m0, sq) + (int)threadIdx.x; row < end; row += (int)blockDim.x) sd[row] = 0.f;
}

// ------------------------------------------------------------------------------------------------
// dQ: a workgroup owns 128 query rows of one (batch, head) and streams K / V tiles of BN keys.
// ------------------------------------------------------------------------------------------------
// DV: head dims the products run over (a multiple of 32, d <= DV <= D); tiles keep the LDS layout of the bucket D
template <typename T, int D, int BN, int DV = D>
struct BwdDqCfg {
    static constexpr int kThreads = 256, kWaves = 4, BM = 128;
    static constexpr int NB = BN / 32, KS = DV / 16, DB = DV / 32, PT = BN / 16, CPR = D / 8, ROWB = D * 2;
    static constexpr int TILE_BYTES = BN * ROWB;
    static constexpr int LOADS = BN * CPR / kThreads;
    static constexpr int STAGE_BYTES = stage_tile_bytes<DB>();   // a wave's dQ rows on their way out
    static constexpr int SMEM = 4 * TILE_BYTES > kWaves * STAGE_BYTES ? 4 * TILE_BYTES : kWaves * STAGE_BYTES;   // {K, V} x 2 stages
    static_assert(BN % 32 == 0 && D % 32 == 0 && (BN * CPR) % kThreads == 0, "tile shape");
    static_assert(TILE_BYTES % (kWaves * 1024) == 0 && TILE_BYTES / (kWaves * 1024) == LOADS, "one fill = 1 KB per wave");
};

template <typename T, int D, int BN, int MINW, bool DROPOUT, int DV = D>
__global__ void __launch_bounds__(256, MINW) bwd_dq_kernel(const BwdKParams kp) {
    typedef BwdDqCfg<T, D, BN, DV> C;
    typedef typename Elem<T>::v8 v8;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const fa_bwd_params& p = kp.p;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;

    // logical order: heads of one group adjacent, then query tiles, then kv heads, then batch; whole
    // (batch, kv head) streams go to one XCD so that workgroups streaming the same K / V share an L2
    // (xcd_stream_unit: contiguous eighths for dense batches, every 8th stream for packed ones)
    bwd_clear_counters(kp);
    const int G = p.h / p.h_k;
    const int num_m_blocks = (p.seqlen_q + C::BM - 1) / C::BM;
    int g, mb, hk, b;
    if (!xcd_rows_item(false, p.cu_seqlens_q != nullptr, (uint32_t)p.b, (uint32_t)p.h_k, (uint32_t)G, (uint32_t)num_m_blocks,
                       (kp.has_left || kp.has_right) ? 32u * MINW : 0u, g, mb, hk, b)) return;
    const int head = hk * G + g;

    const BwdSeq si = bwd_seq(p, b);
    const int m0 = mb * C::BM;
    bwd_pad_d(p, b, head, m0, si.sq, mb == num_m_blocks - 1);
    if (m0 >= si.sq) return;
    const int shift = si.sk - si.sq;
    const int wl = p.window_left, wr = p.window_right;
    const bool has_left = kp.has_left, has_right = kp.has_right;
    int n_hi = si.sk;
    if (has_right) n_hi = min(n_hi, min(m0 + C::BM, si.sq) + shift + wr);
    const int n_lo = has_left ? max(0, m0 + shift - wl) : 0;
    const int t_lo = n_lo / BN;
    const int t_hi = n_hi > 0 ? (n_hi + BN - 1) / BN : 0;

    const T* __restrict__ kg = reinterpret_cast<const T*>(p.k) + si.k_off + (int64_t)hk * p.k_head_stride;
    const T* __restrict__ vg = reinterpret_cast<const T*>(p.v) + si.v_off + (int64_t)hk * p.v_head_stride;

    // resident operands: this lane's query row of Q and dO, its log-sum-exp and D
    const int r0w = m0 + wave * 32;
    const int row = r0w + l32;
    const bool row_ok = row < si.sq;
    v8 qf[C::KS], gf[C::KS];
    {
        const T* qrow = reinterpret_cast<const T*>(p.q) + si.q_off + (int64_t)row * p.q_row_stride + (int64_t)head * p.q_head_stride;
        const T* grow = reinterpret_cast<const T*>(p.dout) + si.do_off + (int64_t)row * p.do_row_stride + (int64_t)head * p.do_head_stride;
#pragma unroll
        for (int dk = 0; dk < C::KS; dk++) {
            const int d0 = dk * 16 + 8 * hh;
            u32x4 a = {0, 0, 0, 0}, c = {0, 0, 0, 0};
            if (row_ok && d0 < p.d) { a = ld_global16(qrow + d0); c = ld_global16(grow + d0); }
            qf[dk] = __builtin_bit_cast(v8, a);
            gf[dk] = __builtin_bit_cast(v8, c);
        }
    }
    // a row beyond the sequence, or one that saw no key (lse = +inf), gets P = exp2(-inf) = 0
    const float lse2 = row_ok ? p.softmax_lse[((int64_t)b * p.h + head) * p.seqlen_q + row] * kLog2e : INFINITY;
    const float dsum = bwd_row_dot<T, C::KS>(p, si, head, row, row_ok, hh, gf);
    if (row_ok && hh == 0) p.softmax_d[((int64_t)b * p.h + head) * p.seqlen_q_rounded + row] = dsum;

    wait_resident_loads();
    f32x16 dq_acc[C::DB];
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) dq_acc[db][r] = 0.f;

    // Tile movers: K and V go from global memory straight into LDS (global_load_lds, 1 KB per wave
    // instruction); the swizzle is applied on the global side.  No zero fill: keys past the sequence
    // repeat its last key and are masked, columns past d repeat the last chunk and meet the zero
    // columns of the resident Q / dO rows or land in dQ columns that are never written.
    const int d_last_chunk = p.d / 8 - 1;
    const uint32_t lds0 = (uint32_t)(size_t)((FA_LDS_PTR(char))smem);
    const uint32_t fill0 = __builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)(wave * C::LOADS * 1024)));
    // fill j of this lane: row f_row(j), chunk f_col(j) of the tile (recomputed where the last tile needs them)
    auto f_row = [&](int j) { return ((wave * C::LOADS + j) * 1024 + lane * 16) / C::ROWB; };
    auto f_col = [&](int j) { return min(swz_u<D>((((wave * C::LOADS + j) * 1024 + lane * 16) % C::ROWB) / 16, f_row(j)), d_last_chunk); };
    uint32_t f_koff[C::LOADS], f_voff[C::LOADS];
#pragma unroll
    for (int j = 0; j < C::LOADS; j++) {
        f_koff[j] = (uint32_t)((f_row(j) * (int)p.k_row_stride + f_col(j) * 8) * 2);
        f_voff[j] = (uint32_t)((f_row(j) * (int)p.v_row_stride + f_col(j) * 8) * 2);
    }
    auto load_tile = [&](int buf, int t) {
        const int n0 = t * BN;
        const T* kt = kg + (int64_t)n0 * p.k_row_stride;
        const T* vt = vg + (int64_t)n0 * p.v_row_stride;
        const uint32_t dk_ = fill0 + (uint32_t)(buf * 2 * C::TILE_BYTES);
        const uint32_t dv_ = dk_ + (uint32_t)C::TILE_BYTES;
        if (n0 + BN <= si.sk) {
#pragma unroll
            for (int j = 0; j < C::LOADS; j++) {
                async_fill16(kt, f_koff[j], dk_ + j * 1024);
                async_fill16(vt, f_voff[j], dv_ + j * 1024);
            }
        } else {
#pragma unroll
            for (int j = 0; j < C::LOADS; j++) {
                const int r = min(f_row(j), si.sk - 1 - n0);
                async_fill16(kt, (uint32_t)((r * (int)p.k_row_stride + f_col(j) * 8) * 2), dk_ + j * 1024);
                async_fill16(vt, (uint32_t)((r * (int)p.v_row_stride + f_col(j) * 8) * 2), dv_ + j * 1024);
            }
        }
    };

    const float sl2 = kp.scale_log2;
    Drop drop = {0, 0, 256, 1.f};
    if constexpr (DROPOUT) drop = drop_init(p.rng_state, p.p_dropout, b, head, p.h);
    LdsOffs<D, C::KS, C::DB> lo;
    lo.init(lane);
    if (t_hi > t_lo) { load_tile(0, t_lo); wait_vmcnt<0>(); }
    __syncthreads();
    int buf = 0;
    for (int t = t_lo; t < t_hi; ++t) {
        const bool has_next = t + 1 < t_hi;
        if (has_next) load_tile(buf ^ 1, t + 1);     // the other stage was last read before the previous barrier
        const int n0 = t * BN;
        const char* kb = smem + buf * 2 * C::TILE_BYTES;
        const char* vb = kb + C::TILE_BYTES;
        const bool skip = (has_right && n0 > r0w + 31 + shift + wr) || (has_left && n0 + BN - 1 < r0w + shift - wl) ||
                          (r0w >= si.sq);
        if (!skip) {
            // one 32-key block at a time, so that only one block's S and dP are live
            const bool need_mask = (n0 + BN > si.sk) || (has_right && n0 + BN - 1 > r0w + shift + wr) ||
                                   (has_left && n0 < r0w + 31 + shift - wl);
            int lim_hi = si.sk - 1;
            if (has_right) lim_hi = min(lim_hi, row + shift + wr);
            const int lim_lo = has_left ? row + shift - wl : 0;
            v8 dsf[C::PT];
#pragma unroll
            for (int nb = 0; nb < C::NB; nb++) {
                f32x16 s_acc[1], dp_acc[1];
                product_rows<T, D, 1, C::KS, 4>(s_acc, kb + nb * 32 * C::ROWB, lo.r, qf);
                product_rows<T, D, 1, C::KS, 4>(dp_acc, vb + nb * 32 * C::ROWB, lo.r, gf);
                if (need_mask) mask_acc16(s_acc[0], n0 + nb * 32 + 4 * hh, lim_lo, lim_hi);
                uint32_t keep[8];
                if constexpr (DROPOUT) drop_pairs_row(drop, row, n0 + nb * 32, hh, keep);
#pragma unroll
                for (int r = 0; r < 16; r++) {
                    const float pv = fast_exp2(s_acc[0][r] * sl2 - lse2);
                    float dpv = dp_acc[0][r];
                    if constexpr (DROPOUT) dpv = drop_gate_half(dpv * drop.rp, keep[r >> 1], r & 1);   // gradient through the dropped P
                    s_acc[0][r] = pv * (dpv - dsum);
                }
                dsf[2 * nb] = pack_acc8<T>(s_acc[0], 0);
                dsf[2 * nb + 1] = pack_acc8<T>(s_acc[0], 8);
            }
            // dQ^T += K^T dS^T
            product_cols<T, D, C::PT, C::DB, 4>(dq_acc, kb, lo.c, dsf);
        }
        wait_vmcnt<0>();       // this wave's fills of the next tile have landed; the barrier publishes them
        __syncthreads();
        buf ^= 1;
    }

    // every tile read is behind the loop's last barrier: the ring is free to stage the gradient rows
    T* obase = reinterpret_cast<T*>(p.dq) + si.dq_off + (int64_t)r0w * p.dq_row_stride + (int64_t)head * p.dq_head_stride;
    store_tile_rows<T, C::DB>(dq_acc, p.softmax_scale, smem + wave * C::STAGE_BYTES, lane, obase, p.dq_row_stride, si.sq - r0w, p.d);
}

// ------------------------------------------------------------------------------------------------
// dQ at head dims 161-256, with dropout 129-256: 128 query rows per workgroup as above, two waves to every 32 rows, so that each fits the 256
// registers of two waves per SIMD (one wave alone needs Q, dO and dQ of its rows, 256 registers at head dim 256, and runs
// by itself on its SIMD: nothing overlaps its exponentials).  Wave w < 4 ("P wave") keeps Q and forms S and P; wave w + 4
// ("dS wave") keeps dO, forms dP and dS; each accumulates one half of dQ's columns.  P crosses in fp32, dS in the 16 bits it
// has as an operand anyway, both lane to same lane (the layouts agree), and both one tile later, so that the hand-overs add
// no barrier: in step t the P wave forms P of tile t, the dS wave dS of tile t - 1 and its half of that tile's dQ, and the
// P wave its half of tile t - 2.  The K ring has four stages for that, V two.
// Bound by each wave's serial stream (reads of a tile, products, exponentials), with the matrix cores busy 39 % of the time
// instead of 26 % (4 x 2039, below).  Whole backward, one wave per 32 rows -> two, bf16: 4 x 2039 causal, 16 / 4 heads, d 256 764 -> 680 us; 2 x 8k, 16 heads
// 5.26 -> 4.67 ms; d 192 2 x 8k causal 3.01 -> 2.85 ms, 4 x 2k full 803 -> 748 us; with dropout 2 x 4k, d 256 1.70 -> 1.51 ms,
// d 192 1.61 -> 1.41 ms, d 136 1.56 -> 1.27 ms, d 160 1.57 -> 1.29 ms (products over 256 columns there too).
// ------------------------------------------------------------------------------------------------
template <typename T, int D, int DV>
struct BwdDq2Cfg {
    static constexpr int kThreads = 512, kWaves = 8, BM = 128, BN = 32;
    static constexpr int KS = DV / 16, DBH = DV / 64, ROWB = D * 2;       // DBH: column blocks of dQ per wave
    static constexpr int TILE = BN * ROWB, FILLS = TILE / 4096;           // fills of 1 KB per requesting wave and tensor
    static constexpr int V_OFF = 4 * TILE, X_OFF = V_OFF + 2 * TILE;      // P hand-over: 2 buffers x 4 row blocks, fp32
    static constexpr int Y_OFF = X_OFF + 2 * 4 * 4096;                    // dS hand-over: 2 x 4, 16 bits
    static constexpr int RING_END = Y_OFF + 2 * 4 * 2048;
    static constexpr int STAGE_BYTES = stage_tile_bytes<DBH>();           // a wave's dQ rows on their way out
    static constexpr int SMEM = RING_END > kWaves * STAGE_BYTES ? RING_END : kWaves * STAGE_BYTES;
    static_assert(DV % 64 == 0 && DV <= D && D % 32 == 0, "halves of whole column blocks");
    static_assert(SMEM <= 160 * 1024, "LDS budget");
};

template <typename T, int D, int DV, bool DROPOUT>
__global__ void __launch_bounds__(512, 2) bwd_dq2_kernel(const BwdKParams kp) {
    typedef BwdDq2Cfg<T, D, DV> C;
    typedef typename Elem<T>::v8 v8;
    constexpr int BN = C::BN;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const fa_bwd_params& p = kp.p;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const bool role_ds = wave >= 4;         // wave-uniform
    const int rblk = wave & 3;

    bwd_clear_counters(kp);
    const int G = p.h / p.h_k;
    const int num_m_blocks = (p.seqlen_q + C::BM - 1) / C::BM;
    int g, mb, hk, b;
    if (!xcd_rows_item(false, p.cu_seqlens_q != nullptr, (uint32_t)p.b, (uint32_t)p.h_k, (uint32_t)G, (uint32_t)num_m_blocks,
                       (kp.has_left || kp.has_right) ? 32u : 0u, g, mb, hk, b)) return;
    const int head = hk * G + g;

    const BwdSeq si = bwd_seq(p, b);
    const int m0 = mb * C::BM;
    bwd_pad_d(p, b, head, m0, si.sq, mb == num_m_blocks - 1);
    if (m0 >= si.sq) return;
    const int shift = si.sk - si.sq;
    const int wl = p.window_left, wr = p.window_right;
    const bool has_left = kp.has_left, has_right = kp.has_right;
    int n_hi = si.sk;
    if (has_right) n_hi = min(n_hi, min(m0 + C::BM, si.sq) + shift + wr);
    const int n_lo = has_left ? max(0, m0 + shift - wl) : 0;
    const int t_lo = n_lo / BN;
    const int t_hi = n_hi > 0 ? (n_hi + BN - 1) / BN : 0;
    const int n = max(0, t_hi - t_lo);

    const T* __restrict__ kg = reinterpret_cast<const T*>(p.k) + si.k_off + (int64_t)hk * p.k_head_stride;
    const T* __restrict__ vg = reinterpret_cast<const T*>(p.v) + si.v_off + (int64_t)hk * p.v_head_stride;

    // Tile movers, as in bwd_dq_kernel.  The dS waves request the tiles: their step is the shorter one (the P waves: 0..2 % slower).
    const int d_last_chunk = p.d / 8 - 1;
    const uint32_t lds0 = (uint32_t)(size_t)((FA_LDS_PTR(char))smem);
    const uint32_t fill0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)(rblk * C::FILLS * 1024)));
    auto f_row = [&](int j) { return ((rblk * C::FILLS + j) * 1024 + lane * 16) / C::ROWB; };
    auto f_col = [&](int j) { return min(swz_u<D>((((rblk * C::FILLS + j) * 1024 + lane * 16) % C::ROWB) / 16, f_row(j)), d_last_chunk); };
    uint32_t f_koff[C::FILLS], f_voff[C::FILLS];
#pragma unroll
    for (int j = 0; j < C::FILLS; j++) {
        f_koff[j] = (uint32_t)((f_row(j) * (int)p.k_row_stride + f_col(j) * 8) * 2);
        f_voff[j] = (uint32_t)((f_row(j) * (int)p.v_row_stride + f_col(j) * 8) * 2);
    }
    auto load_tile = [&](int it) {
        if (!role_ds) return;
        const int n0 = (t_lo + it) * BN;
        const T* kt = kg + (int64_t)n0 * p.k_row_stride;
        const T* vt = vg + (int64_t)n0 * p.v_row_stride;
        const uint32_t dk_ = fill0 + (uint32_t)((it & 3) * C::TILE);
        const uint32_t dv_ = fill0 + (uint32_t)(C::V_OFF + (it & 1) * C::TILE);
        if (n0 + BN <= si.sk) {
#pragma unroll
            for (int j = 0; j < C::FILLS; j++) {
                async_fill16(kt, f_koff[j], dk_ + j * 1024);
                async_fill16(vt, f_voff[j], dv_ + j * 1024);
            }
        } else {
#pragma unroll
            for (int j = 0; j < C::FILLS; j++) {
                const int r = min(f_row(j), si.sk - 1 - n0);
                async_fill16(kt, (uint32_t)((r * (int)p.k_row_stride + f_col(j) * 8) * 2), dk_ + j * 1024);
                async_fill16(vt, (uint32_t)((r * (int)p.v_row_stride + f_col(j) * 8) * 2), dv_ + j * 1024);
            }
        }
    };
    if (n > 0) load_tile(0);

    // resident operand: this lane's query row of Q (P wave) or dO (dS wave)
    const int r0w = m0 + rblk * 32;
    const int row = r0w + l32;
    const bool row_ok = row < si.sq;
    v8 rf[C::KS];
    {
        const T* src = role_ds
            ? reinterpret_cast<const T*>(p.dout) + si.do_off + (int64_t)row * p.do_row_stride + (int64_t)head * p.do_head_stride
            : reinterpret_cast<const T*>(p.q) + si.q_off + (int64_t)row * p.q_row_stride + (int64_t)head * p.q_head_stride;
#pragma unroll
        for (int dk = 0; dk < C::KS; dk++) {
            const int d0 = dk * 16 + 8 * hh;
            u32x4 a = {0, 0, 0, 0};
            if (row_ok && d0 < p.d) a = ld_global16(src + d0);
            rf[dk] = __builtin_bit_cast(v8, a);
        }
    }
    // a row beyond the sequence, or one that saw no key (lse = +inf), gets P = exp2(-inf) = 0
    const float lse2 = row_ok ? p.softmax_lse[((int64_t)b * p.h + head) * p.seqlen_q + row] * kLog2e : INFINITY;
    float dsum = 0.f;
    if (role_ds) {
        dsum = bwd_row_dot<T, C::KS>(p, si, head, row, row_ok, hh, rf);
        if (row_ok && hh == 0) p.softmax_d[((int64_t)b * p.h + head) * p.seqlen_q_rounded + row] = dsum;
    }
    wait_resident_loads();

    f32x16 dq_acc[C::DBH];
#pragma unroll
    for (int db = 0; db < C::DBH; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) dq_acc[db][r] = 0.f;
    LdsOffs<D, C::KS, C::DBH> lo;
    lo.init(lane, role_ds ? C::DBH : 0);
    const float sl2 = kp.scale_log2;
    Drop drop = {0, 0, 256, 1.f};
    if constexpr (DROPOUT) drop = drop_init(p.rng_state, p.p_dropout, b, head, p.h);
    // keys of a tile against this wave's rows: something is visible
    auto live = [&](int it) {
        const int n0 = (t_lo + it) * BN;
        return it >= 0 && it < n && r0w < si.sq && !(has_right && n0 > r0w + 31 + shift + wr) && !(has_left && n0 + BN - 1 < r0w + shift - wl);
    };
    __syncthreads();      // the first tile has landed (every wave waited for its requests above)

    // two steps more than tiles: the last ones drain the hand-overs
    auto walk = [&](auto&& body) {
        for (int it = 0; it < n + 2; ++it) {
            // slots free since the previous barrier: K's held tile it - 3, V's tile it - 1
            if (it + 1 < n) load_tile(it + 1);
            body(it);
            wait_vmcnt<0>();
            __syncthreads();
        }
    };
    if (!role_ds) {
        walk([&](int it) {
            if (live(it)) {
                const int n0 = (t_lo + it) * BN;
                f32x16 s_acc[1];
                product_rows<T, D, 1, C::KS, 4>(s_acc, smem + (it & 3) * C::TILE, lo.r, rf);
                const bool need_mask = (n0 + BN > si.sk) || (has_right && n0 + BN - 1 > r0w + shift + wr) || (has_left && n0 < r0w + 31 + shift - wl);
                if (need_mask) {
                    int lim_hi = si.sk - 1;
                    if (has_right) lim_hi = min(lim_hi, row + shift + wr);
                    mask_acc16(s_acc[0], n0 + 4 * hh, has_left ? row + shift - wl : 0, lim_hi);
                }
                f32x4* x = reinterpret_cast<f32x4*>(smem + C::X_OFF + ((it & 1) * 4 + rblk) * 4096) + lane;
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    f32x4 e4;
#pragma unroll
                    for (int e = 0; e < 4; e++) e4[e] = fast_exp2(s_acc[0][4 * q4 + e] * sl2 - lse2);
                    x[q4 * 64] = e4;
                }
            }
            if (live(it - 2)) {
                const u32x4* y = reinterpret_cast<const u32x4*>(smem + C::Y_OFF + ((it & 1) * 4 + rblk) * 2048) + lane;
                const v8 dsf[2] = {__builtin_bit_cast(v8, y[0]), __builtin_bit_cast(v8, y[64])};
                product_cols<T, D, 2, C::DBH, 4>(dq_acc, smem + ((it - 2) & 3) * C::TILE, lo.c, dsf);
            }
        });
    } else {
        f32x16 dp[1];       // dP - D (dropout: dP) of the previous step's tile, carried over the loop
#pragma unroll
        for (int r = 0; r < 16; r++) dp[0][r] = 0.f;
        walk([&](int it) {
            if (live(it - 1)) {
                const f32x4* x = reinterpret_cast<const f32x4*>(smem + C::X_OFF + (((it - 1) & 1) * 4 + rblk) * 4096) + lane;
                uint32_t keep[8];
                if constexpr (DROPOUT) drop_pairs_row(drop, row, (t_lo + it - 1) * BN, hh, keep);
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const f32x4 p4 = x[q4 * 64];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int r = 4 * q4 + e;
                        if constexpr (DROPOUT) dp[0][r] = p4[e] * (drop_gate_half(dp[0][r] * drop.rp, keep[r >> 1], r & 1) - dsum);   // gradient through the dropped P
                        else dp[0][r] *= p4[e];
                    }
                }
                const v8 dsf[2] = {pack_acc8<T>(dp[0], 0), pack_acc8<T>(dp[0], 8)};
                u32x4* y = reinterpret_cast<u32x4*>(smem + C::Y_OFF + (((it - 1) & 1) * 4 + rblk) * 2048) + lane;
                y[0] = __builtin_bit_cast(u32x4, dsf[0]);
                y[64] = __builtin_bit_cast(u32x4, dsf[1]);
                product_cols<T, D, 2, C::DBH, 4>(dq_acc, smem + ((it - 1) & 3) * C::TILE, lo.c, dsf);
            }
            if (live(it)) {
                if constexpr (!DROPOUT) {
                    // dP - D in one go: the accumulators start from -D of the lane's row
#pragma unroll
                    for (int r = 0; r < 16; r++) dp[0][r] = -dsum;
                }
                product_rows<T, D, 1, C::KS, 4, DROPOUT>(dp, smem + C::V_OFF + (it & 1) * C::TILE, lo.r, rf);
            }
        });
    }
    // every tile read is behind the loop's last barrier: the ring is free to stage the gradient rows
    const int col0 = role_ds ? C::DBH * 32 : 0;
    T* obase = reinterpret_cast<T*>(p.dq) + si.dq_off + (int64_t)r0w * p.dq_row_stride + (int64_t)head * p.dq_head_stride + col0;
    store_tile_rows<T, C::DBH>(dq_acc, p.softmax_scale, smem + wave * C::STAGE_BYTES, lane, obase, p.dq_row_stride, si.sq - r0w, p.d - col0);
}

// ------------------------------------------------------------------------------------------------
// dK, dV: a workgroup owns 128 keys of one (batch, kv head) and streams the Q / dO tiles (BM query rows)
// of every query head of the group; no product is repeated.  8 waves; wave w < 4 ("P wave") owns key
// block w for S = Q K^T, P = exp(S - lse) and dV^T += dO^T P; wave w + 4 ("dS wave") owns the same keys
// for dP = dO V^T, dS = P o (dP - D) and dK^T += Q^T dS.  P goes from the first to the second through
// LDS in accumulator layout (both waves map lanes to keys and registers to query rows identically,
// so the hand-over is lane to same lane, 16 bytes at a time, sign bit = dropped by dropout).  P is
// handed over in fp16 whatever the tensor type: it lies in [0, 1], and its rounding (2^-11 relative)
// is no coarser than the rounding dS = P o (dP - D) gets anyway as an operand of the dK product.
// The dS wave runs ONE TILE BEHIND: in step t it forms dP of tile t (matrix pipe) and dS, dK of tile
// t - 1 (P of that tile was published before the barrier that ended step t - 1), so no barrier is
// added and its exp-free vector work overlaps its own products.  The Q ring therefore has three
// stages (tile t + 1 arriving, t read by the P wave, t - 1 read transposed by the dS wave); dO has two.
// With DPARTS = 2 two workgroups share a key block and each accumulates half of the head dimension of dK / dV (both form S
// and dP in full: six products' worth of work for four): the form for launches of too few key blocks to fill the CUs.
// Head dims 193-256 (129-256 with dropout) ran on it altogether until the accumulators of all 256 columns fitted (C::LEAN).
// Whole backward, bf16, d 256: causal 8k, 16 heads 2304 -> 1750 us; 16 x 512 316 -> 252 us; d 224, 8 x 1000, full, 16 / 8 heads
// 630 -> 488 us; forward + backward with dropout, 16 packed sequences of 500-2000 tokens, 16 heads, d 256 3366 -> 3010 us.
// ------------------------------------------------------------------------------------------------
template <typename T, int D, int BM, int DPARTS, int DV = D>
struct BwdDkv3Cfg {
    static constexpr int kThreads = 512, kWaves = 8, BNW = kBwdKeyBlock;
    static constexpr int MBK = BM / 32, KS = DV / 16, DB = DV / 32 / DPARTS, PT = BM / 16, CPR = D / 8, ROWB = D * 2;
    static constexpr int TILE_BYTES = BM * ROWB;
    // Whole accumulators past head dim 192 (128 registers next to the 64 of the resident row): the products take one ring of LA
    // operands and offsets formed at the read, and the tile requests form theirs anew, so that no register is spilled, not 55.
    static constexpr bool LEAN = DPARTS == 1 && DV > 192;
    static constexpr int LA = 4;       // 5: the same time; 6: 9 registers spilled
    static constexpr int LOADS = BM * CPR / kThreads;
    static constexpr int Q_OFF = 0;                                  // 3 stages
    static constexpr int G_OFF = 3 * TILE_BYTES;                     // dO: 2 stages
    static constexpr int AUX_OFF = 5 * TILE_BYTES;                   // 3 stages x {lse (log2 units), D} x BM floats
    static constexpr int X_OFF = AUX_OFF + 3 * 2 * BM * 4;           // P hand-over: 2 buffers x 4 key blocks
    static constexpr int XBLK = BM * 32 * 2;                         // one key block's P tile, fp16
    static constexpr int RING_END = X_OFF + 2 * 4 * XBLK;
    static constexpr int OUT_BYTES = kWaves * stage_tile_bytes<DB>();   // the gradient rows, staged over the ring after the loop
    static constexpr int SMEM = RING_END > OUT_BYTES ? RING_END : OUT_BYTES;
    // Which waves request the tiles (see the tile movers).  With half the accumulators to a workgroup the P waves' exponentials
    // weigh more against their products and the dS waves wait for them: there those request (whole backward, bf16: d 256, 4 x 2039
    // 680 -> 655 us, 2 x 8k 4.67 -> 4.55 ms; without the split d 192 and d 256 +-0, d 128 1-2 % slower).
    static constexpr bool REQ_DS = DPARTS == 2 && D == 256;
    // the resident K / V rows come in through LDS where the idle ring stages and the hand-over hold them
    static constexpr bool STAGED_ROWS = 4 * 32 * ROWB <= 2 * TILE_BYTES && 4 * 32 * ROWB <= 2 * 4 * XBLK;
    static_assert(BM % 32 == 0 && DV % (32 * DPARTS) == 0 && DV <= D && (BM * CPR) % kThreads == 0 && 2 * BM <= kThreads, "tile shape");
    static_assert(SMEM <= 160 * 1024, "LDS budget");
    static_assert(TILE_BYTES % (kWaves * 1024) == 0 && TILE_BYTES / (kWaves * 1024) == LOADS, "one fill = 1 KB per wave");
};

// The parts of a key block's steps meet in a binary tree (node n has the children 2n and 2n + 1, part i of n is leaf n + i): the
// child that gets to a node second adds the other's partial sums, which that one left in its slot, and goes on to the node above;
// the one that leaves the root has the whole sum and returns true.  Nobody waits, and as a + b = b + a the result does not depend
// on who came first.  Only a child that finds its sibling absent writes its sums out.  Sums go past the L2 of the XCD in both
// directions (relaxed agent-scope accesses, completed before the arrival is counted): a release and an acquire fence instead write
// back and empty that L2 for everyone (16 x 512 tokens, 16 heads on 2, cut in 1.9 parts: the pass 131 us against 93).  Costs 5 us a
// piece at head dim 128 (64 KB of dK, 64 KB of dV).
template <int DB>
FA_DEV bool join_parts(f32x16 (&acc)[DB], uint32_t node, int32_t* counters, char* slots, int64_t slot_bytes, int32_t* flag, int tid) {
    for (; node > 1; node >>= 1) {
        int32_t* const arrived = counters + (node >> 1) - 1;
        if (tid == 0) *flag = __hip_atomic_load(arrived, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        bool second = *flag != 0;
        __syncthreads();
        if (!second) {
            uint64_t* mine = reinterpret_cast<uint64_t*>(slots + (int64_t)(node - 2) * slot_bytes) + tid;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int r = 0; r < 16; r += 2)
                    __hip_atomic_store(mine + (db * 8 + r / 2) * 512, __builtin_bit_cast(uint64_t, f32x2{acc[db][r], acc[db][r + 1]}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the stores of every wave have passed the L2 before the arrival shows
            __syncthreads();
            if (tid == 0) *flag = __hip_atomic_fetch_add(arrived, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            second = *flag != 0;
            __syncthreads();
            if (!second) return false;
        }
        const uint64_t* other = reinterpret_cast<const uint64_t*>(slots + (int64_t)((node ^ 1u) - 2) * slot_bytes) + tid;
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const f32x2 v = __builtin_bit_cast(f32x2, __hip_atomic_load(other + (db * 8 + r / 2) * 512, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                acc[db][r] += v[0];
                acc[db][r + 1] += v[1];
            }
    }
    return true;
}

template <typename T, int D, int BM, int DPARTS, bool DROPOUT, int DV = D>
__global__ void __launch_bounds__(512, 1) bwd_dkv3_kernel(const BwdKParams kp) {
    typedef BwdDkv3Cfg<T, D, BM, DPARTS, DV> C;
    typedef typename Elem<T>::v8 v8;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const fa_bwd_params& p = kp.p;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    const bool role_ds = wave >= 4;         // wave-uniform
    const int kblk = wave & 3;

    const int G = p.h / p.h_k;
    const int num_n_blocks = (p.seqlen_k + C::BNW - 1) / C::BNW;
    const bool split = DPARTS == 1 && kp.split_steps != 0;
    const uint32_t per_stream = split ? (uint32_t)kp.split_pieces : (uint32_t)(num_n_blocks * DPARTS);
    uint32_t unit;
    int hk, b;
    if (!xcd_stream_unit(xcd_strided(p.cu_seqlens_q != nullptr, p.b, p.h_k), (uint32_t)p.b, (uint32_t)p.h_k, per_stream,
                         (kp.has_left || kp.has_right) ? 32u : 0u, (uint32_t)DPARTS, unit, hk, b)) return;
    const int dpart = (int)(unit % DPARTS);      // with DPARTS = 2 a workgroup accumulates half of the head dim
    int nblk = (int)(unit / DPARTS), part = 0, parts = 1, first_join = 0;
    if (split) {
        // the key block and part of this unit: every wave counts the parts of all key blocks, 64 at a time
        int before = 0;
        for (int base = 0; base < num_n_blocks; base += 64) {
            int t_lo, mine = 0;
            if (base + lane < num_n_blocks)
                mine = bwd_block_parts(bwd_block_tiles((base + lane) * kBwdKeyBlock, p.seqlen_q, p.seqlen_k, kp.has_left, p.window_left, kp.has_right,
                                                       p.window_right, BM, t_lo) * G, kp.split_steps);
            int sum = mine;
#pragma unroll
            for (int m = 1; m < 64; m *= 2) {
                const int other = __shfl_up(sum, m);
                if (lane >= m) sum += other;
            }
            const uint64_t past = __ballot(before + sum > (int)unit);
            if (past) {
                const int at = __builtin_ctzll(past), first = before + __builtin_amdgcn_readlane(sum - mine, at);
                nblk = base + at;
                part = (int)unit - first;
                parts = __builtin_amdgcn_readlane(mine, at);
                first_join = first - nblk;
                break;
            }
            before += __builtin_amdgcn_readlane(sum, 63);
        }
    }

    const BwdSeq si = bwd_seq(p, b);
    const int n0 = nblk * C::BNW;
    if (n0 >= si.sk) return;
    const int shift = si.sk - si.sq;
    const int wl = p.window_left, wr = p.window_right;
    const bool has_left = kp.has_left, has_right = kp.has_right;
    int t_lo;
    const int nt = bwd_block_tiles(n0, si.sq, si.sk, has_left, wl, has_right, wr, BM, t_lo);
    const int t_hi = t_lo + nt;
    // this workgroup's part of the key block's nt * G steps
    const int it0 = split ? (int)((int64_t)(nt * G) * part / parts) : 0;
    const int iters = split ? (int)((int64_t)(nt * G) * (part + 1) / parts) - it0 : nt * G;
    const int g0 = it0 ? it0 / nt : 0, t0 = t_lo + it0 - g0 * nt;

    const int j0w = n0 + kblk * 32;
    const int key = j0w + l32;
    const bool key_ok = key < si.sk;

    f32x16 acc[C::DB];      // dV^T (P wave) or dK^T (dS wave) of this wave's keys
#pragma unroll
    for (int db = 0; db < C::DB; db++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[db][r] = 0.f;

    // Tile movers.  Q and dO go from global memory straight into their ring slots (global_load_lds,
    // 1 KB per wave instruction, no staging registers and no LDS store pass): LDS bytes are laid down
    // in lane order, so the swizzle is applied on the global side -- the lane that fills physical chunk
    // pc of row r fetches logical chunk swz_u(pc, r).  There is no zero fill on this path: rows past
    // the sequence repeat its last row and are neutralised by lse = +inf (P = 0), columns past d repeat
    // the last chunk and meet the zero columns of the resident K / V rows, or land in gradient
    // columns that are never written.  lse and D take the register path (one float per lane).
    float aux = 0.f;
    const int d_last_chunk = p.d / 8 - 1;
    const uint32_t lds0 = (uint32_t)(size_t)((FA_LDS_PTR(char))smem);
    // Only the waves of one kind request tiles (FL fills each per tensor), the P waves unless C::REQ_DS: a CU accepts
    // 64 bytes of vector loads per cycle, so a tile keeps the requesting waves at the top of the step for several
    // hundred cycles; meanwhile the others have the matrix pipe to themselves.
    constexpr bool REQ_DS = C::REQ_DS;
    constexpr int FL = 2 * C::LOADS;
    const uint32_t fill0 = __builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)(kblk * FL * 1024)));
    int f_row[FL], f_col[FL];
    uint32_t f_qoff[FL], f_goff[FL];
    if constexpr (!C::LEAN)
#pragma unroll
    for (int j = 0; j < FL; j++) {
        const int pos = (kblk * FL + j) * 1024 + lane * 16;
        f_row[j] = pos / C::ROWB;
        f_col[j] = min(swz_u<D>((pos % C::ROWB) / 16, f_row[j]), d_last_chunk);
        f_qoff[j] = (uint32_t)((f_row[j] * (int)p.q_row_stride + f_col[j] * 8) * 2);
        f_goff[j] = (uint32_t)((f_row[j] * (int)p.do_row_stride + f_col[j] * 8) * 2);
    }
    const int aux_row = tid < BM ? tid : tid - BM;
    auto load_tile = [&](int g, int t, int q3, int g2) {
        const int head = hk * G + g;
        const int i0 = t * BM;
        const T* qt = reinterpret_cast<const T*>(p.q) + si.q_off + (int64_t)head * p.q_head_stride + (int64_t)i0 * p.q_row_stride;
        const T* gt = reinterpret_cast<const T*>(p.dout) + si.do_off + (int64_t)head * p.do_head_stride + (int64_t)i0 * p.do_row_stride;
        const uint32_t dq_ = fill0 + (uint32_t)(C::Q_OFF + q3 * C::TILE_BYTES);
        const uint32_t dg_ = fill0 + (uint32_t)(C::G_OFF + g2 * C::TILE_BYTES);
        if (role_ds != REQ_DS) {
            // nothing to request
        } else if constexpr (C::LEAN) {
            // (offsets formed anew: their tables do not fit)
            const int ln = opaque(lane);
            const int left = si.sq - 1 - i0;
#pragma unroll
            for (int j = 0; j < FL; j++) {
                const int pos = (kblk * FL + j) * 1024 + ln * 16, row = pos / C::ROWB, r = min(row, left);
                const int col = min(swz_u<D>((pos % C::ROWB) / 16, row), d_last_chunk);
                async_fill16(qt, (uint32_t)((r * (int)p.q_row_stride + col * 8) * 2), dq_ + j * 1024);
                async_fill16(gt, (uint32_t)((r * (int)p.do_row_stride + col * 8) * 2), dg_ + j * 1024);
            }
        } else if (i0 + BM <= si.sq) {
#pragma unroll
            for (int j = 0; j < FL; j++) {
                async_fill16(qt, f_qoff[j], dq_ + j * 1024);
                async_fill16(gt, f_goff[j], dg_ + j * 1024);
            }
        } else {
#pragma unroll
            for (int j = 0; j < FL; j++) {
                const int r = min(f_row[j], si.sq - 1 - i0);
                async_fill16(qt, (uint32_t)((r * (int)p.q_row_stride + f_col[j] * 8) * 2), dq_ + j * 1024);
                async_fill16(gt, (uint32_t)((r * (int)p.do_row_stride + f_col[j] * 8) * 2), dg_ + j * 1024);
            }
        }
        if (tid < 2 * BM) {
            // raw value only: anything computed from it here would make the wave wait for the load
            const float* src = tid < BM ? p.softmax_lse + ((int64_t)b * p.h + head) * p.seqlen_q
                                        : p.softmax_d + ((int64_t)b * p.h + head) * p.seqlen_q_rounded;
            aux = src[min(i0 + aux_row, si.sq - 1)];
        }
    };
    // end of a step: the wave's own fills have landed (the barrier that follows publishes them), lse / D go to LDS
    auto finish_tile = [&](int q3, int t) {
        wait_vmcnt<0>();
        if (tid < 2 * BM) {
            const bool in_range = t * BM + aux_row < si.sq;   // rows past the end: lse = +inf => P = 0
            // D goes in negated where the dS wave starts dP from it (dS = P o (dP - D) without a subtraction)
            const float dval = DROPOUT ? aux : -aux;
            reinterpret_cast<float*>(smem + C::AUX_OFF + q3 * 2 * BM * 4)[tid] = tid < BM ? (in_range ? aux * kLog2e : INFINITY) : (in_range ? dval : 0.f);
        }
    };
    auto skip_tile = [&](int i0) {   // keys of this wave against the rows of a tile: nothing visible
        return (has_right && j0w > i0 + BM - 1 + shift + wr) || (has_left && j0w + 31 < i0 + shift - wl) || (j0w >= si.sk);
    };

    // Prologue: the first tile's requests go out first, then the resident operand -- this lane's key
    // row of K (P wave) or of V (dS wave) -- so that the two latencies overlap.
    if (iters > 0) load_tile(g0, t0, 0, 0);
    v8 rf[C::KS];
    {
        const T* blk = role_ds
            ? reinterpret_cast<const T*>(p.v) + si.v_off + (int64_t)n0 * p.v_row_stride + (int64_t)hk * p.v_head_stride
            : reinterpret_cast<const T*>(p.k) + si.k_off + (int64_t)n0 * p.k_row_stride + (int64_t)hk * p.k_head_stride;
        const int rs = (int)(role_ds ? p.v_row_stride : p.k_row_stride);
        if constexpr (C::STAGED_ROWS) {
            // through a wave-private piece of LDS that the ring does not use before the first barrier
            // (K rows: Q stages 1 and 2, V rows: the P hand-over); keys past the sequence repeat its
            // last key: whatever a lane computes for such a key stays in that lane and is never written
            const int region = (role_ds ? C::X_OFF : C::Q_OFF + C::TILE_BYTES) + kblk * 32 * C::ROWB;
            const int last = si.sk - 1 - n0;
            stage_rows_issue<T, D>(blk, [&](int r) { return min(kblk * 32 + r, last) * rs; }, p.d,
                                   (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)region)), lane);
            wait_vmcnt<0>();
            stage_rows_read<T, D, C::KS>(rf, smem + region, p.d, lane);
        } else {
            const T* row = blk + (int64_t)(kblk * 32 + l32) * rs;
#pragma unroll
            for (int dk = 0; dk < C::KS; dk++) {
                const int d0 = dk * 16 + 8 * hh;
                u32x4 a = {0, 0, 0, 0};
                if (key_ok && d0 < p.d) a = ld_global16(row + d0);
                rf[dk] = __builtin_bit_cast(v8, a);
            }
        }
    }
    wait_resident_loads();
    if (iters > 0) finish_tile(0, t0);
    __syncthreads();

    const float sl2 = kp.scale_log2;
    const int rel_hi = has_right ? shift + wr : 0x3fffffff;
    const int rel_lo = has_left ? shift - wl : -0x3fffffff;
    std::conditional_t<C::LEAN, LdsBase<D>, LdsOffs<D, C::KS, C::DB>> lo;
    if constexpr (C::LEAN) lo.init(lane); else lo.init(lane, dpart * C::DB);

    // The tile walk shared by both kinds of wave; `body(it, i0, g, live, prev_live, q3, q3_prev)` is the
    // wave's own work of one step.  iters + 1 steps: the last one drains the dS wave's final tile.
    auto walk = [&](auto&& body) {
        int q3 = 0, q3_prev = 0;                     // Q / aux ring slots of the current and the previous tile
        int cur_t = t0, cur_g = g0, nxt_g = g0, nxt_t = t0;
        bool prev_live = false;                      // the previous tile was not skipped (its P is in the hand-over)
        for (int it = 0; it <= iters; ++it) {
            const bool has_next = it + 1 < iters;
            const int q3_next = q3 == 2 ? 0 : q3 + 1;
            if (has_next) {
                if (++nxt_t == t_hi) { nxt_t = t_lo; ++nxt_g; }
                // slots free since the barrier that ended the previous step: Q[q3_next] held tile it - 2
                // (last read transposed by the dS wave in step it - 1), dO[(it + 1) & 1] held tile it - 1
                load_tile(nxt_g, nxt_t, q3_next, (it + 1) & 1);
            }
            const int i0 = cur_t * BM;
            const bool live = it < iters && !skip_tile(i0);
            body(it, i0, cur_g, live, prev_live, q3, q3_prev);
            prev_live = live;
            if (has_next) finish_tile(q3_next, nxt_t);
            __syncthreads();
            q3_prev = q3;
            q3 = q3_next;
            cur_t = nxt_t;
            cur_g = nxt_g;
        }
    };

    if (!role_ds) {
        walk([&](int it, int i0, int g, bool live, bool, int q3, int) {
            if (live) {
            const char* qb = smem + C::Q_OFF + q3 * C::TILE_BYTES;
            const char* gb = smem + C::G_OFF + (it & 1) * C::TILE_BYTES;
            const float* lse_s = reinterpret_cast<const float*>(smem + C::AUX_OFF + q3 * 2 * BM * 4);
            char* xw = smem + C::X_OFF + ((it & 1) * 4 + kblk) * C::XBLK;
            Drop drop = {0, 0, 256, 1.f};
            if constexpr (DROPOUT) drop = drop_init(p.rng_state, p.p_dropout, b, hk * G + g, p.h);
            f32x16 s_acc[C::MBK];
            if constexpr (C::LEAN) product_rows_ring<T, D, C::KS, C::LA>(s_acc[0], lds0 + (uint32_t)(C::Q_OFF + q3 * C::TILE_BYTES), lo, rf);
            else product_rows<T, D, C::MBK, C::KS, 4>(s_acc, qb, lo.r, rf);
            v8 pf[C::PT];
#pragma unroll
            for (int mb = 0; mb < C::MBK; mb++) {
                const int ib = i0 + mb * 32;
                const bool need_mask = (has_right && j0w + 31 > ib + shift + wr) || (has_left && j0w < ib + 31 + shift - wl);
                if (need_mask) {
                    // entry r is query row ib + 4 hh + c_r, visible iff rel_lo + c_r <= key - ib - 4 hh <= rel_hi + c_r
                    const int rel = key - ib - 4 * hh;
                    mask_acc16(s_acc[mb], 0, rel - rel_hi, rel - rel_lo);
                }
                uint32_t keep[8];
                if constexpr (DROPOUT) drop_pairs_key(drop, key, ib, hh, keep);
#pragma unroll
                for (int q4 = 0; q4 < 4; q4++) {
                    const f32x4 l4 = *reinterpret_cast<const f32x4*>(lse_s + mb * 32 + 8 * q4 + 4 * hh);
#pragma unroll
                    for (int e = 0; e < 4; e++) s_acc[mb][4 * q4 + e] = fast_exp2(s_acc[mb][4 * q4 + e] * sl2 - l4[e]);
                }
                // hand-over copy in fp16 with the sign bit set where dropped (P >= 0), own copy with zeros there:
                // both masked as packed pairs
#pragma unroll
                for (int h8 = 0; h8 < 2; h8++) {
                    u32x4 xo = __builtin_bit_cast(u32x4, pack_acc8<_Float16>(s_acc[mb], 8 * h8));
                    u32x4 pk = __builtin_bit_cast(u32x4, pack_acc8<T>(s_acc[mb], 8 * h8));
                    if constexpr (DROPOUT) {
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            xo[e] |= ~keep[4 * h8 + e] & 0x80008000u;
                            pk[e] &= keep[4 * h8 + e];
                        }
                    }
                    *reinterpret_cast<u32x4*>(xw + ((mb * 2 + h8) * 64 + lane) * 16) = xo;
                    pf[2 * mb + h8] = __builtin_bit_cast(v8, pk);
                }
            }
            if constexpr (C::LEAN) product_cols_ring<T, D, C::PT, C::DB, C::LA>(acc, lds0 + (uint32_t)(C::G_OFF + (it & 1) * C::TILE_BYTES), lo, pf);
            else product_cols<T, D, C::PT, C::DB, 4>(acc, gb, lo.c, pf);
            }
        });
    } else {
        f32x16 dp[C::MBK];      // dP of the tile of the previous step, carried over the loop
#pragma unroll
        for (int mb = 0; mb < C::MBK; mb++)
#pragma unroll
            for (int r = 0; r < 16; r++) dp[mb][r] = 0.f;
        walk([&](int it, int, int, bool live, bool prev_live, int q3, int q3_prev) {
            // first the previous tile (consumes dp), then dP of this tile into the same registers
            if (prev_live) {
                const char* qp = smem + C::Q_OFF + q3_prev * C::TILE_BYTES;
                const float* dsum_s = reinterpret_cast<const float*>(smem + C::AUX_OFF + q3_prev * 2 * BM * 4) + BM;
                const char* xr = smem + C::X_OFF + (((it - 1) & 1) * 4 + kblk) * C::XBLK;
                const float rp = DROPOUT ? 1.f / (1.f - p.p_dropout) : 1.f;
                v8 dsf[C::PT];
#pragma unroll
                for (int mb = 0; mb < C::MBK; mb++) {
                    const f16x8 ph[2] = {*reinterpret_cast<const f16x8*>(xr + ((mb * 2) * 64 + lane) * 16),
                                         *reinterpret_cast<const f16x8*>(xr + ((mb * 2 + 1) * 64 + lane) * 16)};
                    if constexpr (DROPOUT) {
#pragma unroll
                        for (int q4 = 0; q4 < 4; q4++) {
                            const f32x4 d4 = *reinterpret_cast<const f32x4*>(dsum_s + mb * 32 + 8 * q4 + 4 * hh);
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const int r = 4 * q4 + e;
                                const float pv = (float)ph[r >> 3][r & 7];
                                const float dpv = __builtin_signbit(pv) ? 0.f : dp[mb][r] * rp;
                                dp[mb][r] = fabsf(pv) * (dpv - d4[e]);
                            }
                        }
                    } else {
                        // dp already holds dP - D: the product below started from -D
#pragma unroll
                        for (int r = 0; r < 16; r++) dp[mb][r] *= (float)ph[r >> 3][r & 7];
                    }
                    dsf[2 * mb] = pack_acc8<T>(dp[mb], 0);
                    dsf[2 * mb + 1] = pack_acc8<T>(dp[mb], 8);
                }
                if constexpr (C::LEAN) product_cols_ring<T, D, C::PT, C::DB, C::LA>(acc, lds0 + (uint32_t)(C::Q_OFF + q3_prev * C::TILE_BYTES), lo, dsf);
                else product_cols<T, D, C::PT, C::DB, 4>(acc, qp, lo.c, dsf);
            }
            if (live) {
                const char* gb = smem + C::G_OFF + (it & 1) * C::TILE_BYTES;
                if constexpr (DROPOUT) {
                    if constexpr (C::LEAN) product_rows_ring<T, D, C::KS, C::LA>(dp[0], lds0 + (uint32_t)(C::G_OFF + (it & 1) * C::TILE_BYTES), lo, rf);
                    else product_rows<T, D, C::MBK, C::KS, 4>(dp, gb, lo.r, rf);
                } else {
                    // dP - D in one go: the accumulators start from -D of their rows (entry r of a lane
                    // is row 8 (r >> 2) + 4 hh + (r & 3) of its block)
                    const float* nd = reinterpret_cast<const float*>(smem + C::AUX_OFF + q3 * 2 * BM * 4) + BM;
#pragma unroll
                    for (int mb = 0; mb < C::MBK; mb++)
#pragma unroll
                        for (int q4 = 0; q4 < 4; q4++) {
                            const f32x4 d4 = *reinterpret_cast<const f32x4*>(nd + mb * 32 + 8 * q4 + 4 * hh);
                            dp[mb][4 * q4] = d4[0]; dp[mb][4 * q4 + 1] = d4[1]; dp[mb][4 * q4 + 2] = d4[2]; dp[mb][4 * q4 + 3] = d4[3];
                        }
                    if constexpr (C::LEAN) product_rows_ring<T, D, C::KS, C::LA, false>(dp[0], lds0 + (uint32_t)(C::G_OFF + (it & 1) * C::TILE_BYTES), lo, rf);
                    else product_rows<T, D, C::MBK, C::KS, 4, false>(dp, gb, lo.r, rf);
                }
            }
        });
    }
    // every tile read is behind the loop's last barrier: the ring is free
    const BwdArgs ka = fresh_bwd_args();
    if (DPARTS == 1 && parts > 1) {
        const int64_t join = first_join + ((int64_t)b * ka->p.h_k + hk) * (ka->split_pieces - (ka->p.seqlen_k + C::BNW - 1) / C::BNW);
        if (!join_parts<C::DB>(acc, (uint32_t)(parts + part), ka->split_counters + join, ka->scratch + 2 * join * bwd_partial_bytes(D), bwd_partial_bytes(D),
                               reinterpret_cast<int32_t*>(smem), tid)) return;
    }
    const int64_t row_stride = role_ds ? ka->p.dk_row_stride : ka->p.dv_row_stride;
    T* obase = (role_ds ? reinterpret_cast<T*>(ka->p.dk) + si.dk_off : reinterpret_cast<T*>(ka->p.dv) + si.dv_off) + (int64_t)j0w * row_stride
        + (int64_t)hk * (role_ds ? ka->p.dk_head_stride : ka->p.dv_head_stride);
    const float sc = role_ds ? ka->p.softmax_scale : (DROPOUT ? 1.f / (1.f - ka->p.p_dropout) : 1.f);
    const int col0 = dpart * C::DB * 32;
    store_tile_rows<T, C::DB>(acc, sc, smem + wave * stage_tile_bytes<C::DB>(), lane, obase + col0,
                              row_stride, si.sk - j0w, ka->p.d - col0);
}

// ------------------------------------------------------------------------------------------------
// launchers
// ------------------------------------------------------------------------------------------------
template <typename T, int D, int BN, int MINW, bool DROPOUT, int DV = D>
int launch_bwd_dq(const BwdKParams& kp, hipStream_t stream) {
    typedef BwdDqCfg<T, D, BN, DV> C;
    const int64_t nmb = (kp.p.seqlen_q + C::BM - 1) / C::BM;
    if (nmb * kp.p.h * kp.p.b <= 0) return 0;
    const int64_t nblocks = xcd_rows_grid(false, kp.p.cu_seqlens_q != nullptr, kp.p.b, kp.p.h_k, kp.p.h / kp.p.h_k, nmb);
    if (nblocks == 0) return -2;
    auto kern = bwd_dq_kernel<T, D, BN, MINW, DROPOUT, DV>;
    if (int e = (int)FA_ALLOW_DYNAMIC_LDS(kern, C::SMEM)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::kThreads), C::SMEM, stream, kp);
    return (int)hipGetLastError();
}

template <typename T, int D, int DV, bool DROPOUT>
int launch_bwd_dq2(const BwdKParams& kp, hipStream_t stream) {
    typedef BwdDq2Cfg<T, D, DV> C;
    const int64_t nmb = (kp.p.seqlen_q + C::BM - 1) / C::BM;
    if (nmb * kp.p.h * kp.p.b <= 0) return 0;
    const int64_t nblocks = xcd_rows_grid(false, kp.p.cu_seqlens_q != nullptr, kp.p.b, kp.p.h_k, kp.p.h / kp.p.h_k, nmb);
    if (nblocks == 0) return -2;
    auto kern = bwd_dq2_kernel<T, D, DV, DROPOUT>;
    if (int e = (int)FA_ALLOW_DYNAMIC_LDS(kern, C::SMEM)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::kThreads), C::SMEM, stream, kp);
    return (int)hipGetLastError();
}

template <typename T, int D, int BM, int DPARTS, bool DROPOUT, int DV = D>
int launch_bwd_dkv3(const BwdKParams& kp, hipStream_t stream) {
    typedef BwdDkv3Cfg<T, D, BM, DPARTS, DV> C;
    const int64_t per_stream = DPARTS == 1 && kp.split_steps ? kp.split_pieces : (int64_t)((kp.p.seqlen_k + C::BNW - 1) / C::BNW) * DPARTS;
    if (per_stream * kp.p.h_k * kp.p.b <= 0) return 0;
    const int64_t nblocks = xcd_grid(xcd_strided(kp.p.cu_seqlens_q != nullptr, kp.p.b, kp.p.h_k), kp.p.b, kp.p.h_k, per_stream);
    if (nblocks == 0) return -2;
    auto kern = bwd_dkv3_kernel<T, D, BM, DPARTS, DROPOUT, DV>;
    if (int e = (int)FA_ALLOW_DYNAMIC_LDS(kern, C::SMEM)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)nblocks), dim3(C::kThreads), C::SMEM, stream, kp);
    return (int)hipGetLastError();
}

}  // namespace fa
