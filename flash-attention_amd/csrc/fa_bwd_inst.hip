// Backward kernels, one translation unit per (dtype, head-dim bucket): compiled with
// -DFA_T_BF16=0/1 -DFA_D=64/128/256.
#include "fa_bwd.h"
#include "fa_bwd_stream.h"
#include "fa_launch.h"

namespace fa {
#if FA_T_BF16
typedef __bf16 InstT;
#define FA_INST_NAME2(d) launch_bwd_bf16_##d
#else
typedef _Float16 InstT;
#define FA_INST_NAME2(d) launch_bwd_fp16_##d
#endif
#define FA_INST_NAME(d) FA_INST_NAME2(d)

// dQ pass, which leaves softmax_d and clears the counters of cut key blocks, then dK/dV pass, which reads both, on the same stream.
#ifndef FA_DQ_BN
#define FA_DQ_BN (FA_D > 64 ? 32 : 64)
#endif
// DV: head dims the products run over (head dims up to 96 on the 128 bucket, up to 160 and up to 192 on the 256 bucket)
template <bool DROPOUT, int DV = FA_D>
static int run(const BwdKParams& kp, hipStream_t stream) {
#if FA_D <= 128
    // two workgroups (8 waves) per CU: the key tile is sized so that the kernel stays within 256 registers;
    // three at head dim 64 (168 registers), where the vector work per matrix instruction doubles -- without
    // dropout: the mask words do not fit in 168 registers (19 spilled, 7-15 % slower than two workgroups)
    if (int e = launch_bwd_dq<InstT, FA_D, FA_DQ_BN, (FA_D == 64 && !DROPOUT ? 3 : 2), DROPOUT, DV>(kp, stream)) return e;
    // Fewer key blocks than CUs (one long sequence on one or two kv heads, say): two workgroups per
    // key block, each accumulating half of the head dimension, fill the CUs at 3/4 of the work each.
    if (kp.halves) return launch_bwd_dkv3<InstT, FA_D, bwd_dkv_rows(FA_D), 2, DROPOUT>(kp, stream);
    return launch_bwd_dkv3<InstT, FA_D, bwd_dkv_rows(FA_D), 1, DROPOUT, DV>(kp, stream);
#else
    // Up to head dim 160 the dQ pass fits 256 registers with 32-key steps: two workgroups per CU, as at head dim 128
    // (d 160, bf16 causal 8k, 16 heads: backward 5.79 -> 5.07 ms against one workgroup with 64-key steps).  Beyond
    // that one wave cannot hold a row block's Q, dO and dQ next to another on its SIMD (76 registers spilled at 192), and
    // two waves share it (bwd_dq2_kernel; figures there).  With dropout the whole bucket takes it, head dims 129-160 too.
    if constexpr (DV <= 160) {
        if (int e = launch_bwd_dq<InstT, FA_D, 32, 2, DROPOUT, DV>(kp, stream)) return e;
    } else {
        if (int e = launch_bwd_dq2<InstT, FA_D, DV, DROPOUT>(kp, stream)) return e;
    }
    // A wave holds its whole dK / dV accumulator next to its resident key row, except where that leaves too many CUs without a key
    // block (bwd_halves, fa_api.hip)
    if constexpr (DV > 192) {
        if (kp.halves) return launch_bwd_dkv3<InstT, FA_D, bwd_dkv_rows(FA_D), 2, DROPOUT, DV>(kp, stream);
    }
    return launch_bwd_dkv3<InstT, FA_D, bwd_dkv_rows(FA_D), 1, DROPOUT, DV>(kp, stream);
#endif
}

int FA_INST_NAME(FA_D)(const BwdKParams& kp, hipStream_t stream) {
#if FA_D == 64
    if (kp.one_pass)
        return kp.p.p_dropout > 0.f ? launch_bwd_stream<InstT, FA_D, true>(kp, stream) : launch_bwd_stream<InstT, FA_D, false>(kp, stream);
#endif
    if (kp.p.p_dropout > 0.f) return run<true>(kp, stream);
#if FA_D == 128
    if (kp.p.d <= 96) return run<false, 96>(kp, stream);
#elif FA_D == 256
    if (kp.p.d <= 160) return run<false, 160>(kp, stream);
    if (kp.p.d <= 192) return run<false, 192>(kp, stream);
#endif
    return run<false>(kp, stream);
}

}  // namespace fa
