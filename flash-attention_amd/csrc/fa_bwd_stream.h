// Backward in one pass for head dims up to 64: one workgroup computes dQ, dK and dV of a whole (batch, kv head).
//
// The two-pass form (fa_bwd.h) forms S and dP twice and reads q, k, v and dout twice, and on short sequences its
// workgroups are all start-up: a dK/dV workgroup of a 512-token causal sequence runs one to four steps behind an
// exposed fetch of its rows.  Here every product is formed once (5 tile products instead of 7, one exponential instead
// of two), D = rowsum(dO o O) is formed on the way in, and the start-up of one key block overlaps the write-out of the
// one before it.
//
//   * grid: persistent workgroups of 4 waves, two per CU (75 KB of LDS each), so that one's fetches and write-outs run under
//     the other's products; a workgroup takes whole (batch, kv head) streams, packed sequences by falling cost in a snake
//     order, so that workgroups get equal sums.
//   * a stream's keys are taken 128 at a time (32 per wave, K and V rows resident in registers as B operands); the query
//     tiles (64 rows of every grouped q head) stream through LDS.  S = Q K^T and dP = dO V^T give each lane one key and
//     16 query rows per 32-row block, the layout in which P and dS are the B operands of dV^T += dO^T P and dK^T += Q^T dS
//     as they stand: neither leaves the registers for those two products.
//   * dQ sums over the keys of all waves, so dS also goes to LDS, [key][query row] in 16 bits, and behind a barrier every
//     wave forms a 32 x 32 piece of the tile's dQ^T = K^T dS^T.
//   * a dQ tile that several key blocks contribute to is kept in fp32 in a scratch slot of the workgroup between them
//     (written and read by the same lanes, in the same order every time: deterministic); with up to 128 keys, or where
//     the mask leaves a tile to one key block, it goes straight out.
//
// What bounds it: no unit alone.  fp16, 32 x 512 tokens, 32 heads, causal: 351 us (rowsum 31, dQ pass 119, dK/dV pass 201) ->
// 207-215 us.  1.14 GB go past the L2 (0.73 read, 0.41 written, counted): 0.54 of inputs and results, 0.40 of dQ tiles that go
// out and come back (in 64 MB of slots, which the 256 MB memory-side cache can hold), 0.20 of query tiles read again by later
// key blocks: 5.4 TB/s, where a copy from and to HBM reaches 4.9.  The matrix pipe is busy 21 % of the time; waves spend 36 % of
// theirs in s_waitcnt, 31 % waiting to issue and 33 % issuing.  64 packed sequences of 64..512 tokens, 16 heads, dropout: 371 ->
// 192-202 us, 0.82 GB, matrix pipe 16 %, waves 43 / 21 / 36 %.  A form with 8 waves and 256 keys per block moves 0.78 GB in the
// first case, but its one workgroup per CU leaves the memory idle while it computes and the other way round: 229 us.
#pragma once
#include "fa_bwd.h"

namespace fa {

constexpr int kBwdStreamOrdered = 2048;

template <typename T, int D>
struct BwdStreamCfg {
    static constexpr int kThreads = 256, kWaves = 4, kPerCU = 2, BN = 128, BM = 64;
    static constexpr int KS = D / 16, DB = D / 32, ROWB = D * 2;
    static constexpr int TILE = BM * ROWB;
    static constexpr int SLOT = 2 * TILE, AUX = 2 * BM * 4;   // ring slot: Q tile, dO tile; its {lse, -D} row pair apart
    // LDS: two ring slots, dS, the K tile, one O tile, {lse, -D} x 2, the order of the sequences
    static constexpr int DS_OFF = 2 * SLOT, KT_OFF = DS_OFF + BN * BM * 2;
    static constexpr int O_OFF = KT_OFF + BN * ROWB, AUX_OFF = O_OFF + TILE;
    static constexpr int ORD_OFF = AUX_OFF + 2 * AUX;
    static constexpr int kMaxBatch = kBwdStreamOrdered;     // packed sequences that are ordered by cost
    static constexpr int SMEM = ORD_OFF + kMaxBatch * 2;
    // Between two key blocks V rows arrive in the dS buffer (wave 3's first), and gradient rows leave through the second
    // ring slot, whose end wave 3 exceeds into its own V rows once it has read them
    static FA_DEV int v_off(int wave) { return DS_OFF + (kWaves - 1 - wave) * 32 * ROWB; }
    static constexpr int OUT_OFF = SLOT;
    static_assert(D == 64, "tile geometry");
    static_assert(TILE == 2 * kWaves * 1024, "two fills per wave, tensor and tile");
    static_assert(OUT_OFF + kWaves * stage_tile_bytes<DB>() <= DS_OFF + 32 * ROWB, "staged gradient rows");
    static_assert(SMEM * kPerCU <= 160 * 1024, "LDS budget");
};

// Scratch of one workgroup slot: when several key blocks contribute to dQ, a stream's dQ tiles in fp32.
inline int64_t bwd_stream_slot_bytes(const fa_bwd_params& p) {
    typedef BwdStreamCfg<_Float16, 64> C;
    return p.seqlen_k > C::BN ? (int64_t)(p.h / p.h_k) * ((p.seqlen_q + C::BM - 1) / C::BM) * (C::BM * 64 * 4) : 0;
}
constexpr int64_t kBwdStreamSlots = 512;      // two workgroups per CU
inline int64_t bwd_stream_slots(const fa_bwd_params& p) { return std::min(kBwdStreamSlots, (int64_t)p.b * p.h_k); }

// Indices 0 .. n - 1 (n <= N) by falling cost, ties by index, in a workgroup of 4 waves: a counting sort over 256 costs (larger
// ones, 1024 x 1024 tokens have 153, count as 255).  A wave ranks 64 indices at a time among themselves by ballots over the bits of
// the cost; the counts by (cost, chunk of 64) are then summed up.  Every workgroup of the launch does this for itself and gets the
// same order.  It must not take long: comparing all pairs took 80 us with 900 sequences (28 us of work).
template <int N, class Cost>
FA_DEV void order_by_cost(uint16_t* order, int n, char* smem, Cost cost) {
    constexpr int CH = N / 64;                  // chunks; counts[key][chunk], 2 bytes each, then the sums of the four waves
    uint16_t* const counts = reinterpret_cast<uint16_t*>(smem);
    int* const sums = reinterpret_cast<int*>(smem + 256 * CH * 2);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    static_assert(N % 512 == 0, "a thread owns the counts of one cost, 16 bytes at a time");
    u32x4* const mine = reinterpret_cast<u32x4*>(counts + tid * CH);
#pragma unroll
    for (int j = 0; j < CH / 8; j++) mine[j] = u32x4{0, 0, 0, 0};
    __syncthreads();
    int slot[CH / 4];                           // (key << 8 | rank among its chunk's equals) of this lane's index of each chunk
#pragma unroll
    for (int c = 0; c < CH / 4; c++) {
        const int chunk = 4 * c + wave, i = chunk * 64 + lane;
        if (chunk * 64 >= n) break;
        const bool in = i < n;
        const int key = in ? 255 - min(max(cost(i), 0), 255) : 0;
        uint64_t same = __ballot(in);
#pragma unroll
        for (int bit = 0; bit < 8; bit++) {
            const uint64_t set = __ballot((key >> bit) & 1);
            same &= ((key >> bit) & 1) ? set : ~set;
        }
        const int before = __popcll(same & ((1ull << lane) - 1ull));
        if (in && before == 0) counts[key * CH + chunk] = (uint16_t)__popcll(same);
        slot[c] = key << 8 | before;
    }
    __syncthreads();
    int total = 0;
    for (int j = 0; j < CH; j++) total += counts[tid * CH + j];
    int upto = total;                           // sum over the keys of this wave's threads up to this one
#pragma unroll
    for (int s = 1; s < 64; s *= 2) {
        const int v = __shfl_up(upto, s, 64);
        if (lane >= s) upto += v;
    }
    if (lane == 63) sums[wave] = upto;
    __syncthreads();
    int at = upto - total;
    for (int w = 0; w < wave; w++) at += sums[w];
    for (int j = 0; j < CH; j++) {
        const int v = counts[tid * CH + j];
        counts[tid * CH + j] = (uint16_t)at;
        at += v;
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < CH / 4; c++) {
        const int chunk = 4 * c + wave, i = chunk * 64 + lane;
        if (i < n) order[counts[(slot[c] >> 8) * CH + chunk] + (slot[c] & 255)] = (uint16_t)i;
    }
    __syncthreads();
}

// dq = K^T dS^T for 32 head dims (block dblk) x 32 query rows (block qblk) of a tile over NK x 16 keys: A = columns of the K
// tile, B = columns of the dS tile ([key][64 query rows], the same layout)
template <typename T, int D, int NK, class Offs>
FA_DEV void dq_product_32(f32x16& dq, const char* kt, const char* ds, const Offs& lo, int dblk, int qblk) {
    typedef typename Elem<T>::v8 v8;
    // (selected by arithmetic: an array index that depends on the wave would put the table into scratch memory)
    const int a0 = dblk ? lo.c[1][0] : lo.c[0][0], a1 = dblk ? lo.c[1][1] : lo.c[0][1];
    const int b0 = qblk ? lo.c[1][0] : lo.c[0][0], b1 = qblk ? lo.c[1][1] : lo.c[0][1];
    constexpr int GRP = 2, NG = NK / GRP;
    v8 fa_[2][GRP], fb_[2][GRP];
    auto rd = [&](int g, int set) {
#pragma unroll
        for (int j = 0; j < GRP; j++) {
            fa_[set][j] = lds_cols_at<T, D>(kt, a0, a1, g * GRP + j);
            fb_[set][j] = lds_cols_at<T, D>(ds, b0, b1, g * GRP + j);
        }
    };
    rd(0, 0);
#pragma unroll
    for (int g = 0; g < NG; g++) {
        if (g + 1 < NG) rd(g + 1, (g + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < GRP; j++) mfma_step<T>(dq, fa_[g & 1][j], fb_[g & 1][j], g * GRP + j);
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <typename T, int D, bool DROPOUT>
__global__ void __launch_bounds__(256, 2) bwd_stream_kernel(const BwdKParams) {
    typedef BwdStreamCfg<T, D> C;
    typedef typename Elem<T>::v8 v8;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, l32 = lane & 31, hh = lane >> 5;
    int n_items, G, d;
    float sl2, scale;
    char* dq_slot;            // this workgroup's scratch: dQ tiles by (grouped head, query tile)
    int max_tiles;
    bool ordered;
    uint16_t* const order = reinterpret_cast<uint16_t*>(smem + C::ORD_OFF);
    {
        const BwdArgs a = fresh_bwd_args();
        G = a->p.h / a->p.h_k;
        d = a->p.d;
        n_items = a->p.b * a->p.h_k;
        sl2 = a->scale_log2;
        scale = a->p.softmax_scale;
        max_tiles = (a->p.seqlen_q + C::BM - 1) / C::BM;
        dq_slot = a->scratch + (int64_t)blockIdx.x * a->slot_bytes;
        // packed sequences: indices by falling (query tiles x key blocks), ties by index
        const int nb = a->p.b;
        ordered = a->p.cu_seqlens_q != nullptr && nb <= C::kMaxBatch;
        if (ordered) {
            const int32_t* cq = a->p.cu_seqlens_q;
            const int32_t* ck = a->p.cu_seqlens_k;
            order_by_cost<C::kMaxBatch>(order, nb, smem, [&](int i) { return ((cq[i + 1] - cq[i]) / C::BM + 1) * ((ck[i + 1] - ck[i]) / C::BN + 1); });
        }
    }

    const uint32_t lds0 = (uint32_t)(size_t)((FA_LDS_PTR(char))smem);
    const uint32_t fill0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)(wave * 2048)));
    LdsOffs<D, C::KS, C::DB> lo;
    lo.init(lane);
    // dS writes: this lane's key row of the [key][64] tile; chunk c of it sits at ((c ^ x) * 16)
    const int ds_row = C::DS_OFF + (wave * 32 + l32) * 128 + hh * 8;
    const int ds_x = swz_u<64>(0, l32) * 16;
    // dQ product: query rows 32 (wave & 1) .. + 31, head dims 32 (wave >> 1) .. + 31 of a tile; both operands are read
    // transposed, so the permutation of the keys within 16 is the same for both
    const int qblk = wave & 1, dblk = wave >> 1;

    f32x16 dk_acc[C::DB], dv_acc[C::DB];
    // where the accumulators of the previous key block go, once the next one's rows have come in
    T* out_dk = nullptr;
    T* out_dv = nullptr;
    int out_rows = 0;
    bool pending = false;
    auto write_out = [&]() {
        const BwdArgs a = fresh_bwd_args();
        const int ln = opaque(lane);
        char* st = smem + C::OUT_OFF + wave * stage_tile_bytes<C::DB>();
        store_tile_rows<T, C::DB>(dk_acc, a->p.softmax_scale, st, ln, out_dk, a->p.dk_row_stride, out_rows, a->p.d);
        store_tile_rows<T, C::DB>(dv_acc, DROPOUT ? 1.f / (1.f - a->p.p_dropout) : 1.f, st, ln, out_dv, a->p.dv_row_stride, out_rows, a->p.d);
        pending = false;
    };

    for (int round = 0; round * (int)gridDim.x < n_items; ++round) {
        const int rank = round * (int)gridDim.x + ((round & 1) ? (int)gridDim.x - 1 - (int)blockIdx.x : (int)blockIdx.x);
        if (rank >= n_items) continue;
        int hk, b, sq, sk, shift, ntiles, nkb;
        int64_t bh0;                                  // (b, first grouped head) of lse and softmax_d
        const T *q0, *g0, *o0, *kg, *vg;                 // row 0 of the stream: first grouped head, this kv head
        T *dq0, *dk0, *dv0;
        bool has_left, has_right;
        int wl, wr;
        {
            const BwdArgs a = fresh_bwd_args();
            hk = rank % a->p.h_k;
            b = rank / a->p.h_k;
            if (ordered) b = __builtin_amdgcn_readfirstlane((int)order[b]);
            sq = a->p.seqlen_q;
            sk = a->p.seqlen_k;
            int64_t rq = 0, rk = 0, bb = b;           // first packed row / batch index
            if (a->p.cu_seqlens_q) { rq = a->p.cu_seqlens_q[b]; sq = a->p.cu_seqlens_q[b + 1] - (int)rq; rk = a->p.cu_seqlens_k[b]; sk = a->p.cu_seqlens_k[b + 1] - (int)rk; bb = 0; }
            const int head = hk * G;
            bh0 = (int64_t)b * a->p.h + head;
            q0 = reinterpret_cast<const T*>(a->p.q) + bb * a->p.q_batch_stride + rq * a->p.q_row_stride + (int64_t)head * a->p.q_head_stride;
            g0 = reinterpret_cast<const T*>(a->p.dout) + bb * a->p.do_batch_stride + rq * a->p.do_row_stride + (int64_t)head * a->p.do_head_stride;
            o0 = reinterpret_cast<const T*>(a->p.out) + bb * a->p.o_batch_stride + rq * a->p.o_row_stride + (int64_t)head * a->p.o_head_stride;
            kg = reinterpret_cast<const T*>(a->p.k) + bb * a->p.k_batch_stride + rk * a->p.k_row_stride + (int64_t)hk * a->p.k_head_stride;
            vg = reinterpret_cast<const T*>(a->p.v) + bb * a->p.v_batch_stride + rk * a->p.v_row_stride + (int64_t)hk * a->p.v_head_stride;
            dq0 = reinterpret_cast<T*>(a->p.dq) + bb * a->p.dq_batch_stride + rq * a->p.dq_row_stride + (int64_t)head * a->p.dq_head_stride;
            dk0 = reinterpret_cast<T*>(a->p.dk) + bb * a->p.dk_batch_stride + rk * a->p.dk_row_stride + (int64_t)hk * a->p.dk_head_stride;
            dv0 = reinterpret_cast<T*>(a->p.dv) + bb * a->p.dv_batch_stride + rk * a->p.dv_row_stride + (int64_t)hk * a->p.dv_head_stride;
            has_left = a->has_left; has_right = a->has_right;
            wl = a->p.window_left; wr = a->p.window_right;
            shift = sk - sq;
            // scratch, lse and softmax_d hold max_seqlen rows of a sequence (the two-pass grids end there too)
            sq = min(sq, a->p.seqlen_q);
            sk = min(sk, a->p.seqlen_k);
            ntiles = (sq + C::BM - 1) / C::BM;
            nkb = (sk + C::BN - 1) / C::BN;
        }
        // Bounds with the mask folded in: query row i sees keys i + rel_lo .. i + rel_hi.  Key block kb visits query tile t iff
        // first_kb(t) <= kb <= last_kb(t)
        const int rel_hi = has_right ? shift + wr : 0x3fffffff;
        const int rel_lo = has_left ? shift - wl : -0x3fffffff;
        auto first_kb = [&](int t) { return max(0, (t * C::BM + rel_lo) >> 7); };
        auto last_kb = [&](int t) { return min(nkb - 1, (t * C::BM + C::BM - 1 + rel_hi) >> 7); };

        for (int kb = 0; kb < max(nkb, 1); ++kb) {
            const int n0 = kb * C::BN;
            const int j0w = n0 + wave * 32, key = j0w + l32;
            // tiles t with 64 t + 63 >= n0 - rel_hi and 64 t < n0 + 128 - rel_lo
            const int t_lo = min(ntiles, max(0, n0 - rel_hi) / C::BM);
            const int t_hi = min(ntiles, (max(0, n0 + C::BN - rel_lo) + C::BM - 1) / C::BM);
            const int nt = nkb > 0 ? max(0, t_hi - t_lo) : 0;
            const int iters = nt * G;

            // Tile mover, one tile ahead: Q and dO straight into their ring slot, O next to them the first time a tile is
            // visited, two fills of 1 KB per wave and tensor.  Rows past the end repeat the last one.
            int ld_t = t_lo, ld_g = 0, ld_s = 0;
            const T *ld_q, *ld_do, *ld_o;
            uint32_t f_qoff[2], f_goff[2], f_ooff[2], q_step, g_step, o_step;
            {
                const BwdArgs a = fresh_bwd_args();
                const int ln = opaque(lane);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int f_row = wave * 16 + j * 8 + (ln >> 3), f_col = min(swz_u<D>(ln & 7, f_row), d / 8 - 1);
                    f_qoff[j] = (uint32_t)((f_row * (int)a->p.q_row_stride + f_col * 8) * 2);
                    f_goff[j] = (uint32_t)((f_row * (int)a->p.do_row_stride + f_col * 8) * 2);
                    f_ooff[j] = (uint32_t)((f_row * (int)a->p.o_row_stride + f_col * 8) * 2);
                }
                q_step = (uint32_t)(C::BM * (int)a->p.q_row_stride);
                g_step = (uint32_t)(C::BM * (int)a->p.do_row_stride);
                o_step = (uint32_t)(C::BM * (int)a->p.o_row_stride);
            }
            auto load_head = [&]() {
                const BwdArgs a = fresh_bwd_args();
                ld_q = scalar_ptr(q0 + (int64_t)ld_g * a->p.q_head_stride + (int64_t)t_lo * q_step);
                ld_do = scalar_ptr(g0 + (int64_t)ld_g * a->p.do_head_stride + (int64_t)t_lo * g_step);
                ld_o = scalar_ptr(o0 + (int64_t)ld_g * a->p.o_head_stride + (int64_t)t_lo * o_step);
            };
            load_head();
            auto load_tile = [&]() {
                const BwdArgs a = fresh_bwd_args();
                const bool fresh = first_kb(ld_t) == kb;
                const uint32_t dst = fill0 + (uint32_t)(ld_s * C::SLOT);
                if ((ld_t + 1) * C::BM <= sq) {
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        async_fill16(ld_q, f_qoff[j], dst + j * 1024);
                        async_fill16(ld_do, f_goff[j], dst + C::TILE + j * 1024);
                        if (fresh) async_fill16(ld_o, f_ooff[j], fill0 + C::O_OFF + j * 1024);
                    }
                } else {
                    const int ln = opaque(lane);
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const int f_row = wave * 16 + j * 8 + (ln >> 3), r = min(f_row, sq - 1 - ld_t * C::BM), f_col = min(swz_u<D>(ln & 7, f_row), d / 8 - 1);
                        async_fill16(ld_q, (uint32_t)((r * (int)a->p.q_row_stride + f_col * 8) * 2), dst + j * 1024);
                        async_fill16(ld_do, (uint32_t)((r * (int)a->p.do_row_stride + f_col * 8) * 2), dst + C::TILE + j * 1024);
                        if (fresh) async_fill16(ld_o, (uint32_t)((r * (int)a->p.o_row_stride + f_col * 8) * 2), fill0 + C::O_OFF + j * 1024);
                    }
                }
                // lse by wave 0, D of a tile visited before by wave 1
                if (wave == 0 || (wave == 1 && !fresh)) {
                    const float* src = wave == 0 ? a->p.softmax_lse + (bh0 + ld_g) * a->p.seqlen_q : a->p.softmax_d + (bh0 + ld_g) * a->p.seqlen_q_rounded;
                    async_fill4(scalar_ptr(src + ld_t * C::BM), (uint32_t)(min(lane, sq - 1 - ld_t * C::BM) * 4),
                                (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + C::AUX_OFF + ld_s * C::AUX + wave * C::BM * 4)));
                }
            };
            // The wave's own fills of the loader's tile have landed; what it fetched of lse, dO and O becomes {lse in log2 units,
            // -D} (rows past the end: lse = +inf, so P = 0), and the loader steps over to the following tile.
            auto finish_tile = [&]() {
                wait_vmcnt<0>();
                asm volatile("" ::: "memory");
                const bool fresh = first_kb(ld_t) == kb;
                float* aux = reinterpret_cast<float*>(smem + C::AUX_OFF + ld_s * C::AUX);
                const int left = sq - ld_t * C::BM;
                if (wave == 0) aux[lane] = lane < left ? aux[lane] * kLog2e : INFINITY;
                if (fresh) {
                    const int ln = opaque(lane);
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        // this lane's own 16 bytes of a row of dO and O (8 lanes hold a row; columns past d repeat others)
                        const int row = wave * 16 + j * 8 + (ln >> 3);
                        const char* at = smem + wave * 2048 + j * 1024 + ln * 16;
                        float o8[8], g8[8], dot = 0.f;
                        unpack8<T>(*reinterpret_cast<const u32x4*>(at + C::O_OFF), o8);
                        unpack8<T>(*reinterpret_cast<const u32x4*>(at + ld_s * C::SLOT + C::TILE), g8);
#pragma unroll
                        for (int e = 0; e < 8; e++) dot += o8[e] * g8[e];
                        if (swz_u<D>(ln & 7, row) * 8 >= d) dot = 0.f;
                        dot += __shfl_xor(dot, 4, 8);
                        dot += __shfl_xor(dot, 2, 8);
                        dot += __shfl_xor(dot, 1, 8);
                        if ((ln & 7) == 0) {
                            aux[C::BM + row] = row < left ? -dot : 0.f;
                            if (row < left) {
                                const BwdArgs a = fresh_bwd_args();
                                a->p.softmax_d[(bh0 + ld_g) * a->p.seqlen_q_rounded + ld_t * C::BM + row] = dot;
                            }
                        }
                    }
                } else if (wave == 1) {
                    aux[C::BM + lane] = lane < left ? -aux[C::BM + lane] : 0.f;
                }
                ld_s ^= 1;
                ld_q += q_step;
                ld_do += g_step;
                ld_o += o_step;
                if (++ld_t == t_hi) {
                    ld_t = t_lo;
                    if (++ld_g < G) load_head();
                }
            };

            // This key block's rows and its first tiles (every LDS read of the block before is behind a barrier).
            const int ln = opaque(lane);
            if (nkb > 0) {
                const BwdArgs a = fresh_bwd_args();
                const int last_key = sk - 1 - n0;
                const uint32_t rows = (uint32_t)(wave * 32 * C::ROWB);
                const int krs = (int)a->p.k_row_stride, vrs = (int)a->p.v_row_stride;
                stage_rows_issue<T, D>(scalar_ptr(kg + (int64_t)n0 * krs), [&](int r) { return min(wave * 32 + r, last_key) * krs; }, d,
                                       (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + C::KT_OFF + rows)), ln);
                stage_rows_issue<T, D>(scalar_ptr(vg + (int64_t)n0 * vrs), [&](int r) { return min(wave * 32 + r, last_key) * vrs; }, d,
                                       (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds0 + (uint32_t)C::v_off(wave))), ln);
            }
            if (iters > 0) load_tile();
            if (kb == 0) {
                // D of the padding rows; dQ and D of rows that no key block visits
                const BwdArgs a = fresh_bwd_args();
                const int pitch = a->p.seqlen_q_rounded;
                for (int g = 0; g < G; ++g) {
                    float* sd = a->p.softmax_d + (bh0 + g) * pitch;
                    for (int row = sq + tid; row < pitch; row += C::kThreads) sd[row] = 0.f;
                    if (!has_left && !has_right && nkb > 0) continue;
                    for (int row = tid >> 3; row < sq; row += C::kThreads / 8) {
                        if (first_kb(row / C::BM) <= last_kb(row / C::BM)) continue;
                        const int c8 = (tid & 7) * 8;
                        if (c8 == 0) sd[row] = 0.f;
                        if (c8 < d) st_global16(dq0 + (int64_t)g * a->p.dq_head_stride + (int64_t)row * a->p.dq_row_stride + c8, u32x4{0, 0, 0, 0});
                    }
                }
                if (nkb == 0) break;
            }
            if (iters > 0) finish_tile(); else wait_vmcnt<0>();
            v8 kf[C::KS], vf[C::KS];
            stage_rows_read<T, D, C::KS>(kf, smem + C::KT_OFF + wave * 32 * C::ROWB, d, ln);
            stage_rows_read<T, D, C::KS>(vf, smem + C::v_off(wave), d, ln);
            if (pending) write_out();      // (its stores drain under the first steps)
#pragma unroll
            for (int db = 0; db < C::DB; db++)
#pragma unroll
                for (int r = 0; r < 16; r++) { dk_acc[db][r] = 0.f; dv_acc[db][r] = 0.f; }
            __syncthreads();

            int cur_g = 0, cur_t = t_lo;
            for (int it = 0; it < iters; ++it) {
                const int s = it & 1;
                if (it + 1 < iters) load_tile();      // its slot was last read before the previous barrier
                // dQ of this tile: the sum so far, then this key block's share
                const bool dq_first = first_kb(cur_t) == kb, dq_last = last_kb(cur_t) == kb;
                f32x16 dq;
                f32x4* const sp = reinterpret_cast<f32x4*>(dq_slot + (int64_t)(cur_g * max_tiles + cur_t) * (C::BM * 64 * 4)) + wave * 256;
                f32x4 prior[4];
                if (!dq_first) {
#pragma unroll
                    for (int j = 0; j < 4; j++) prior[j] = sp[j * 64 + lane];
                }
                const int i0 = cur_t * C::BM;
                const bool live = j0w < sk && j0w <= i0 + C::BM - 1 + rel_hi && j0w + 31 >= i0 + rel_lo;
                {
                    const char* qb = smem + s * C::SLOT;
                    const char* gb = qb + C::TILE;
                    const float* aux = reinterpret_cast<const float*>(smem + C::AUX_OFF + s * C::AUX);
                    char* dsw = smem + ds_row;
                    if (!live) {
#pragma unroll
                        for (int c = 0; c < 8; c++) *reinterpret_cast<u32x2*>(dsw + ((c * 16) ^ ds_x)) = u32x2{0, 0};
                    } else {
                        Drop drop = {0, 0, 256, 1.f};
                        if constexpr (DROPOUT) {
                            const BwdArgs a = fresh_bwd_args();
                            drop = drop_init(a->p.rng_state, a->p.p_dropout, b, hk * G + cur_g, a->p.h);
                        }
                        // one block of 32 rows at a time: only its S and dP are live
#pragma unroll
                        for (int mb = 0; mb < 2; mb++) {
                            const int ib = i0 + mb * 32;
                            f32x16 sa[1], dp[1];
                            product_rows<T, D, 1, C::KS, 4>(sa, qb + mb * 32 * C::ROWB, lo.r, kf);
                            if constexpr (!DROPOUT) {
                                // dP - D in one go: the accumulators start from -D of their rows
#pragma unroll
                                for (int q4 = 0; q4 < 4; q4++) {
                                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(aux + C::BM + mb * 32 + 8 * q4 + 4 * hh);
                                    dp[0][4 * q4] = d4[0]; dp[0][4 * q4 + 1] = d4[1]; dp[0][4 * q4 + 2] = d4[2]; dp[0][4 * q4 + 3] = d4[3];
                                }
                            }
                            product_rows<T, D, 1, C::KS, 4, DROPOUT>(dp, gb + mb * 32 * C::ROWB, lo.r, vf);
                            const bool need_mask = j0w + 31 >= sk || j0w + 31 > ib + rel_hi || j0w < ib + 31 + rel_lo;
                            if (need_mask) {
                                // entry r is query row ib + 4 hh + c_r, visible iff rel_lo + c_r <= key - ib - 4 hh <= rel_hi + c_r
                                const int rel = key - ib - 4 * hh;
                                const bool ok = key < sk;
                                mask_acc16(sa[0], 0, ok ? rel - rel_hi : 1, ok ? rel - rel_lo : 0);
                            }
                            uint32_t keep[8];
                            if constexpr (DROPOUT) drop_pairs_key(drop, key, ib, hh, keep);
#pragma unroll
                            for (int q4 = 0; q4 < 4; q4++) {
                                const f32x4 l4 = *reinterpret_cast<const f32x4*>(aux + mb * 32 + 8 * q4 + 4 * hh);
#pragma unroll
                                for (int e = 0; e < 4; e++) {
                                    const int r = 4 * q4 + e;
                                    sa[0][r] = fast_exp2(sa[0][r] * sl2 - l4[e]);
                                    if constexpr (!DROPOUT) dp[0][r] *= sa[0][r];
                                }
                                if constexpr (DROPOUT) {
                                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(aux + C::BM + mb * 32 + 8 * q4 + 4 * hh);
#pragma unroll
                                    for (int e = 0; e < 4; e++) {
                                        const int r = 4 * q4 + e;
                                        dp[0][r] = sa[0][r] * (drop_gate_half(dp[0][r] * drop.rp, keep[r >> 1], r & 1) + d4[e]);
                                    }
                                }
                            }
                            v8 pf[2], dsf[2];
#pragma unroll
                            for (int h8 = 0; h8 < 2; h8++) {
                                u32x4 pk = __builtin_bit_cast(u32x4, pack_acc8<T>(sa[0], 8 * h8));
                                if constexpr (DROPOUT) {
#pragma unroll
                                    for (int e = 0; e < 4; e++) pk[e] &= keep[4 * h8 + e];
                                }
                                pf[h8] = __builtin_bit_cast(v8, pk);
                                dsf[h8] = pack_acc8<T>(dp[0], 8 * h8);
                                const u32x4 d_ = __builtin_bit_cast(u32x4, dsf[h8]);
                                const int c = 4 * mb + 2 * h8;
                                *reinterpret_cast<u32x2*>(dsw + ((c * 16) ^ ds_x)) = u32x2{d_[0], d_[1]};
                                *reinterpret_cast<u32x2*>(dsw + (((c + 1) * 16) ^ ds_x)) = u32x2{d_[2], d_[3]};
                            }
                            product_cols<T, D, 2, C::DB, 4>(dv_acc, gb + mb * 32 * C::ROWB, lo.c, pf);
                            product_cols<T, D, 2, C::DB, 4>(dk_acc, qb + mb * 32 * C::ROWB, lo.c, dsf);
                        }
                    }
                }
                __syncthreads();
                dq_product_32<T, D, C::BN / 16>(dq, smem + C::KT_OFF, smem + C::DS_OFF, lo, dblk, qblk);
                // the next tile has landed; the barrier publishes it
                if (it + 1 < iters) finish_tile(); else wait_vmcnt<0>();
                if (!dq_first) {
#pragma unroll
                    for (int r_ = 0; r_ < 16; r_++) dq[r_] += prior[r_ >> 2][r_ & 3];
                }
                if (dq_last) {
                    const BwdArgs a = fresh_bwd_args();
                    const int row = i0 + 32 * qblk + l32;
                    T* dst = dq0 + (int64_t)cur_g * a->p.dq_head_stride + (int64_t)row * a->p.dq_row_stride;
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const int col = 32 * dblk + 8 * j + 4 * hh;
                        const u32x2 v = {pack2<T>(dq[4 * j] * scale, dq[4 * j + 1] * scale), pack2<T>(dq[4 * j + 2] * scale, dq[4 * j + 3] * scale)};
                        if (row < sq && col < d) st_global8(dst + col, v);
                    }
                } else {
#pragma unroll
                    for (int j = 0; j < 4; j++) sp[j * 64 + lane] = f32x4{dq[4 * j], dq[4 * j + 1], dq[4 * j + 2], dq[4 * j + 3]};
                }
                __syncthreads();
                if (++cur_t == t_hi) { cur_t = t_lo; ++cur_g; }
            }
            {
                const BwdArgs a = fresh_bwd_args();
                out_dk = dk0 + (int64_t)j0w * a->p.dk_row_stride;
                out_dv = dv0 + (int64_t)j0w * a->p.dv_row_stride;
                out_rows = sk - j0w;
                pending = true;
            }
        }
    }
    if (pending) write_out();
}

template <typename T, int D, bool DROPOUT>
int launch_bwd_stream(const BwdKParams& kp, hipStream_t stream) {
    typedef BwdStreamCfg<T, D> C;
    auto kern = bwd_stream_kernel<T, D, DROPOUT>;
    if (int e = (int)FA_ALLOW_DYNAMIC_LDS(kern, C::SMEM)) return e;
    hipLaunchKernelGGL(kern, dim3((unsigned)bwd_stream_slots(kp.p)), dim3(C::kThreads), C::SMEM, stream, kp);
    return (int)hipGetLastError();
}

}  // namespace fa
