// Op::MoeFfn of one, two, four or eight token rows as ONE launch in which the expert weights are requested before the routing is known.
//
// What the reference fixes for this op is the routing (ids in rank order, routing weights, bit for bit:
// crates/infr-cpu/src/lib.rs:3684-3716 for the logits' summation order, :3746-3861 for gating, selection and
// renormalisation) and the rank order of the final sum (:4290-4302).  The expert stages need much less: the SET of
// selected experts.  This kernel therefore computes every router logit twice.  A fast estimate (each thread multiplies
// the eight elements it loaded, a tree adds them up) gives a guess of the selected set a few hundred nanoseconds
// after the operands have arrived, and the expert rows of the guessed set are requested at once.  The exact logits
// (eight 256- or 512-step chains of dependent multiply-adds per logit), the exact routing routine and the check of the
// guess run on one wavefront beside the stream of weights.  Only the exact results are published, decide the ranks and
// weigh the sum.  When the guess misses an expert of the exact set (logits that differ by less than the estimate's
// rounding), the workgroups that hold an expert outside the set compute the missing one late; a record's tag carries
// the expert it belongs to, so a consumer can never take the product of a wrong guess for the one it waits for.
//
// Work split.  256 workgroups of 8 wavefronts; of R token rows each has 256 / R of them, whole XCDs (consecutive workgroups go to
// consecutive XCDs).  A row's workgroups form 8 groups of 32 / R that each share an XCD's L2, or, with four experts per token (one
// row), 4 groups of 64 on two XCDs.  Group g computes one expert of the set: workgroup m of its M the features
// [m * nff / M, +nff / M) of gate and up, then the output rows [m * ne / M, +ne / M) of down.  An
// always-on expert folded into the op is spread over all workgroups of the row (256 for one row: features [b * nff / 256, ..), rows
// [b * ne / 256, ..)); it needs no routing, so its rows are the first bytes requested.  Wavefront 0 is the router
// (exact chains, exact routing, check of the guess), wavefronts 1..7 stream weights: each keeps a ring of items
// (a gate row and an up row, or a group of down rows) in flight, finishes the oldest and requests the one D places
// ahead.  The first down rows are requested before the group's activations have been handed over.
//
// Hand-over between workgroups: 64-bit records {value bits, tag} written and polled with agent-scope relaxed atomics,
// no fence anywhere; the tag is the launch's sequence number (kept in device memory, advanced by the workgroup that
// leaves last) and, for the activations, the expert id.  Every wait is bounded: after `spin_limit` polls a workgroup
// raises the host-visible fault word and skips to the end; its peers run into their own limits, so the grid drains.
// Inside a workgroup the wavefronts hand over through LDS flags; a flag is always set, also on the failure path.
//
// The inner products, the activation, the routing routine and the order of the final sum are those of the
// three-launch kernels (k_gemv.hip): same bits.
#include "layer_stream.h"

namespace infr {

size_t moe_layer_stream_workspace_bytes(int ne, int nff, int n_expert, int rows) {
    // [launch count of each workgroup: 1 KB], then for each of the regions one part per token row:
    // [estimates 8 * n_expert][logits 8 * n_expert][h 8 * nff][h always-on nff][partials 8 * ne]
    return 1024 + (size_t)rows * ((size_t)2 * kGroups * n_expert + (size_t)kGroups * nff + (size_t)nff + (size_t)kGroups * ne) * 8;
}

namespace {

template <class FG, class FD>
bool stream_shape(const MoeLayerParams& q, StreamShape* out) {
    const MoeGemvParams& p = q.g;
    const int ne = p.ne, nff = p.nff, n_expert = p.route.n_expert;
    const bool shared = p.sh_gate != nullptr;
    if (ne != 1024 && ne != 2048 && ne != 4096) return false;        // 128, 256 or 512 octets on 512 threads
    if (ne % FG::kBlockElems || nff % FD::kBlockElems || nff % 256 || nff > 1536) return false;
    // (1024 / 512, 32 experts, 12 layers with norm and residual, three launches and this one, us: one row in Q8_0 242 and 146, in Q4_K /
    // Q6_K 233 and 132; two rows 315 and 220, 290 and 166; four 351 and 282, 316 and 204; eight in Q4_K / Q6_K 351 and 268)
    if (ne == 1024 ? nff != 512 || n_expert != 32 : nff % 384 || n_expert == 32) return false;   // whole shares of the gathering wavefronts
    const int lpr_g = ne / FG::kBlockElems * FG::kLPB, lpr_d = nff / FD::kBlockElems * FD::kLPB;
    if (lpr_g > 64 || lpr_d > 64) return false;
    if (n_expert != 32 && (n_expert % 64 || n_expert > 256 || n_expert < 64)) return false;
    const int rwc_g = 64 / lpr_g, rwc_d = 64 / lpr_d;
    const int rows = p.rows;
    if (rows != 1 && rows != 2 && rows != 4 && rows != 8) return false;   // whole XCDs per token row
    // eight rows (one XCD per row, four workgroups per group): faster than the per-token kernels for the K-quant shape
    // (48.4 against 51.4 us at 2048 / 768), slower for Q8_0 banks (86.3 against 79 us)
    if (rows == 8 && std::is_same<FG, Q80Fmt>::value) return false;
    const int mpg = kPerGroup / rows, bpr = kBlocks / rows;
    if (nff % mpg || ne % bpr) return false;
    const int fpb = nff / mpg, R = ne / mpg;
    const int n_gi = (fpb + rwc_g - 1) / rwc_g, n_di = (R + rwc_d - 1) / rwc_d;
    const int my_gi = (n_gi + kSW - 1) / kSW, my_di = (n_di - router_wave_down_items(n_di) + kSW - 1) / kSW;
    if (my_gi * rwc_g > 64) return false;                            // a wavefront's results wait in one 64-float row
    if (shared) {
        if (nff % bpr) return false;
    }
    // every logit once for the grid when a group's copy of the router would be a large share of the layer's bytes
    out->once = q.logits_once;
    if (ne / bpr > 64) return false;                                  // a workgroup's output rows: one per lane of the summing wavefront
    out->epb = out->once ? (n_expert + bpr - 1) / bpr : n_expert / mpg;
    const int H = kThreads / (ne / 8);
    out->ept = (out->epb + H - 1) / H;
    out->nsp = n_expert / 64;   // 0: half a wavefront's
    // everything in flight at once when a wavefront has few items, rings otherwise
    out->dg = my_gi <= 2 ? 2 : my_gi <= 4 && std::is_same<FG, Q80Fmt>::value ? 4 : 2;
    out->early_down = my_gi <= out->dg ? 1 : 0;
    // down rows requested behind the last gate/up rows ride out the hand-over of the activations: a deep ring
    out->dd = my_di <= 2 ? 2 : my_di <= 5 && std::is_same<FD, Q80Fmt>::value ? 5 : out->early_down ? 3 : 4;
    const int jstride = ne / 8 + 4;
    const size_t floats = (size_t)(out->epb + 1) * 8 * jstride + 2 * (size_t)n_expert +
                          ((route_scratch_floats(n_expert, p.route.n_groups) + 3) & ~(size_t)3) + 2 * (size_t)nff;
    out->lds = cells_bytes(ne) + floats * 4 + 2 * cells_bytes(nff);
    return out->lds <= 150 * 1024;
}

template <class FG, class FD>
bool dispatch_stream(hipStream_t s, MoeLayerParams q, bool launch) {
    StreamShape sh;
    if (!stream_shape<FG, FD>(q, &sh)) return false;
    q.epb = sh.epb;
    q.early_down = sh.early_down;
#define INFR_STREAM(DGv, DDv, EPTv, NSPv)                                                        \
    if (sh.dg == DGv && sh.dd == DDv && sh.ept == EPTv && sh.nsp == NSPv)                           \
        return launch ? launch_stream<FG, FD, DGv, DDv, EPTv, NSPv>(s, q, sh.lds) : true;
    {   // the benchmark shapes with their sizes as constants, ahead of the instantiations for any shape
        bool taken = false;
        const bool done = launch_stream_fixed(s, q, sh, launch, &taken);
        if (taken) return done;
    }
    if (q.norm_w || q.g.ne == 1024) return false;   // the fold of the token row's RmsNorm and this width exist for the fixed shapes only
    if constexpr (std::is_same<FG, Q4KFmt>::value) {
        INFR_STREAM(2, 2, 2, 2)   // ne 2048, nff 768, 128 experts, a copy of the router per group
        INFR_STREAM(2, 2, 1, 2)   // ... every logit once
        INFR_STREAM(2, 2, 1, 4)   // ... 256 experts
        INFR_STREAM(2, 4, 1, 2)   // ne 2048, nff 768, 128 experts, two or four token rows
        INFR_STREAM(2, 4, 1, 4)   // ne 4096, nff 1536, 256 experts, every logit once
    } else {
        INFR_STREAM(4, 5, 2, 2)   // Q8_0: ne 2048, nff 768, 128 experts
        INFR_STREAM(4, 5, 1, 2)
        INFR_STREAM(4, 5, 1, 4)
        INFR_STREAM(2, 4, 1, 2)   // two or four token rows
    }
#undef INFR_STREAM
    return false;
}

template <int NSP, int NORM>
bool launch_stream4(hipStream_t s, const MoeLayerParams& q, size_t lds) {
    return launch_stream<Mxfp4Fmt, Mxfp4Fmt, 3, 4, 1, NSP, 0, 0, 1, NORM, 4>(s, q, lds);
}

// Four experts per token, MXFP4 banks (one token row, no always-on expert).  us per layer of 2880 / 2880, 128 experts, with norm and
// residual: three launches 32 to 37 over boxes, this one 30.  The stream bounds it (10 us of 1530-byte rows for gate/up, 5 for down: a
// row is 45 lanes' 34 unaligned bytes, whose loads keep the CU's address path busy as long as their 96 instructions a row keep
// the vector ALUs), then the hand-over of h between 64 workgroups on two XCDs (3 us).
// Where three launches are as fast they stay: with narrow rows and many of them the hand-overs cost more than the launches.  us a layer that
// one launch saves, with norm and residual | the op alone, at 64 experts: nff 512 1024 / 1280 / 2048 / 2880 / 4096 wide 0.7 0.3 0.9 1.5 3.3 |
// -0.2 0.1 0.4 1.1 2.4; 1536 -0.5 -0.7 -0.9 0.7 2.0 | -2.0 -0.9 0.3 0.4 1.9; 2880 -1.8 -1.8 -0.2 0.6 1.7 | -1.5 -1.1 -0.1 0.6 2.1; 3456 -1.2 -0.9 -0.8
// -1.1 0.6 | -1.9 -1.7 -0.4 -1.1 1.0.  At 128: 512 0.9 1.1 1.3 2.3 5.2 | 0.4 0.5 1.4 1.6 2.2; 1024 0.6 1.2 0.7 0.0 2.4 | -0.5 0.0 0.2 0.6 0.2; 2048 0.3 -0.4 0.3
// 0.2 3.5 | -0.9 -0.7 -0.5 0.2 0.6.  (2304 to 3328 wide at 64 experts and nff 768 to 3072 lies within 1.3 us of either side and stays here.)
bool four_pays(int ne, int nff, int n_expert) {
    if (nff <= 640 || ne >= 4096) return true;
    return n_expert == 128 ? ne >= 2048 || nff <= 1024 : ne >= 2304 && nff <= 3072;
}
bool stream_four(hipStream_t s, MoeLayerParams q, bool launch) {
    const MoeGemvParams& p = q.g;
    const int ne = p.ne, nff = p.nff, n_expert = p.route.n_expert, rwc = ne <= 1024 ? 4 : ne <= 2048 ? 2 : 1;
    if (p.rows != 1 || p.sh_gate || !q.logits_once || (n_expert != 64 && n_expert != 128)) return false;
    if (ne % 64 || ne < 1024 || ne > 4096 || nff % 64 || nff < 512 || nff > 4096) return false;   // 64 elements per lane, 8 to 64 lanes per row
    if (!four_pays(ne, nff, n_expert)) return false;
    const int share = nff / gather_waves(nff);
    if (nff % gather_waves(nff) || share % 64 || share > 9 * 64) return false;
    const int n_gi = (nff / 64 + rwc - 1) / rwc;
    q.epb = 1;   // one logit on each of the first n_expert workgroups
    q.early_down = (n_gi + kSW - 1) / kSW <= 3;
    const int jstride = ne / 8 + 4;
    const size_t floats = (size_t)2 * 8 * jstride + 2 * (size_t)n_expert + ((route_scratch_floats(n_expert, p.route.n_groups) + 3) & ~(size_t)3) +
                          2 * (size_t)nff;
    const size_t lds = cells_bytes<Mxfp4Fmt>(ne) + floats * 4 + 2 * cells_bytes<Mxfp4Fmt>(nff);
    if (lds > 150 * 1024) return false;
    if (!launch) return true;
    if (n_expert == 64) return q.norm_w ? launch_stream4<1, 1>(s, q, lds) : launch_stream4<1, 0>(s, q, lds);
    {   // the benchmark shape with its sizes as constants, ahead of the instantiation for any (4 layers 120 us, 126)
        bool taken = false;
        const bool done = launch_stream_fixed(s, q, StreamShape{3, 4, 1, 2, 1, 1, 0, lds}, launch, &taken);
        if (taken) return done;
    }
    return q.norm_w ? launch_stream4<2, 1>(s, q, lds) : launch_stream4<2, 0>(s, q, lds);
}

bool stream_any(hipStream_t s, const MoeLayerParams& q, bool launch) {
    const MoeGemvParams& p = q.g;
    const RouteParams& r = p.route;
    const bool four = p.n_used == 4 && p.gate_dt == INFR_MXFP4 && p.down_dt == INFR_MXFP4;
    if ((p.n_used != kGroups && !four) || p.n_cu < kBlocks || p.gate_dt != p.up_dt) return false;
    if ((p.sh_gate != nullptr) != (p.sh_down != nullptr) || (p.sh_gate != nullptr) != (p.sh_up != nullptr)) return false;
    // the guess ranks the experts by their logits: gatings that are monotone in the logit, no bias, no groups, no given
    // ids; options that need the routing weights before the gate/up stage or remap ids stay on the in-order kernels
    if ((r.gating != INFR_GATING_SOFTMAX && r.gating != INFR_GATING_SIGMOID) || r.exp_probs_b || r.expert_ids ||
        (r.n_groups > 1 && r.n_groups_used > 0) || r.ep_n > 0 || p.weight_before || p.skip_zero_w)
        return false;
    if (launch && ((((uintptr_t)q.router | (uintptr_t)q.router_x | (uintptr_t)p.x) & 15) != 0 || (q.router_row_floats & 3) != 0))
        return false;
    if (four) return stream_four(s, q, launch);
    if (p.gate_dt == INFR_Q4K && p.down_dt == INFR_Q6K) return dispatch_stream<Q4KFmt, Q6KFmt>(s, q, launch);
    if (p.gate_dt == INFR_Q8_0 && p.down_dt == INFR_Q8_0) return dispatch_stream<Q80Fmt, Q80Fmt>(s, q, launch);
    return false;
}

}  // namespace

bool moe_layer_stream_supported(const MoeLayerParams& q) { return stream_any(nullptr, q, false); }
bool launch_moe_layer_stream(hipStream_t s, const MoeLayerParams& q) { return stream_any(s, q, true); }

}  // namespace infr
