// The fixed shapes of k_layer_stream_shapes.hip that are not K-quant banks of hidden size 2048 or 4096.
#include "layer_stream.h"

namespace infr {

bool launch_stream_fixed_other(hipStream_t s, const MoeLayerParams& q, const StreamShape& sh, bool launch, bool* taken) {
    const MoeGemvParams& p = q.g;
    *taken = true;
    const int norm = q.norm_w ? 1 : 0;
    if (p.n_used == 4) {   // MXFP4 (stream_four)
        if (p.ne == 2880 && p.nff == 2880 && p.route.n_expert == 128) {
            if (!launch) return true;
            return norm ? launch_stream<Mxfp4Fmt, Mxfp4Fmt, 3, 4, 1, 2, 2880, 2880, 1, 1, 4>(s, q, sh.lds)
                        : launch_stream<Mxfp4Fmt, Mxfp4Fmt, 3, 4, 1, 2, 2880, 2880, 1, 0, 4>(s, q, sh.lds);
        }
        *taken = false;
        return false;
    }
    if (p.gate_dt == INFR_Q4K && p.down_dt == INFR_Q6K) {
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 2, 1, 0, 1024, 512, 1)    // 32 experts (the only instantiations of this width)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 2, 1, 0, 1024, 512, 2)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 2, 1, 0, 1024, 512, 4)
        INFR_STREAM_AT(Q4KFmt, Q6KFmt, 2, 4, 1, 0, 1024, 512, 8)
    } else if (p.gate_dt == INFR_Q8_0 && p.down_dt == INFR_Q8_0) {
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 4, 5, 1, 2, 2048, 768, 1)
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 2, 4, 1, 2, 2048, 768, 2)
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 2, 4, 1, 2, 2048, 768, 4)
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 2, 2, 1, 0, 1024, 512, 1)    // 32 experts
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 4, 2, 1, 0, 1024, 512, 2)
        INFR_STREAM_AT(Q80Fmt, Q80Fmt, 2, 5, 1, 0, 1024, 512, 4)
    }
    *taken = false;
    return false;
}

}  // namespace infr
