// The streaming single-launch kernel of Op::MoeFfn instantiated for the benchmark shapes with hidden size, intermediate
// size and token rows as compile-time constants: the lane placement, the item counts and every index division of the
// kernel then fold, which is worth a tenth of the launch (measured on one box, same bits: hidden 2048 / 768, one row
// 19.4 -> 17.5 us per layer; hidden 4096 / 1536 with the always-on expert 39.9 -> 35.0 us).  Translation units of their own,
// so that the sets of instantiations compile side by side; and two of these, the K-quant banks here, the others in
// k_layer_stream_shapes_other.hip: a unit is one code object, and in one of 3.3 MB the same instructions took longer than in two (three
// layers of 256 experts of 4096 x 1536 with norm and residual 105.9 us a pass, and 105.0; other shapes as before).
#include "layer_stream.h"

namespace infr {

bool launch_stream_fixed(hipStream_t s, const MoeLayerParams& q, const StreamShape& sh, bool launch, bool* taken) {
    const MoeGemvParams& p = q.g;
    const int norm = q.norm_w ? 1 : 0;
    *taken = true;
    if (p.gate_dt == INFR_Q4K && p.down_dt == INFR_Q6K) {
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 2, 1, 2, 2048, 768, 1)    // 128 experts, one token row
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 1, 2, 2048, 768, 2)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 1, 2, 2048, 768, 4)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 2, 2, 2048, 768, 8)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 1, 4, 4096, 1536, 1)   // 256 experts, with or without the always-on expert
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 2, 4, 4096, 1536, 2)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 4, 4, 4096, 1536, 4)
    }
    return launch_stream_fixed_other(s, q, sh, launch, taken);
}

}  // namespace infr
