// Batched Op::MoeFfn and large Linear ops on block-quantised weights: the per-expert GEMMs.
//
// An item is (expert, tile of up to 64 tokens of its bucket, column tile); a workgroup of four waves takes one, three
// workgroups share a CU and drift apart, so that one's barriers, loads and stores hide behind the others' arithmetic.
//   * A wave owns 32 weight rows (gate/up: 16 gate rows and the 16 up rows of the same features; down: 32 rows) over the
//     whole of K, against all tokens of the tile.  It loads a step of its rows (kStep k) with consecutive lanes on
//     consecutive 16-byte chunks of a row (a lane reading its own row would touch a cache line per lane) and turns it to
//     a row per lane through a small LDS region of its own, the next step being in flight in registers meanwhile.
//   * v_mfma_f32_16x16x32_f16: lane = weight row (lane & 15) and a quarter of 32 k (lane / 16).  Tiles of up to 16, 32
//     and 64 tokens have code of their own (T = 1, 2, 4): nothing is contracted for more than 15 absent tokens.
//   * The tile's activations go from memory straight into LDS, in pieces of 16 T tokens x 512 / T k, two pieces in
//     turn: one barrier per piece.
//   * The weight operand holds small integers, not values: a code masked into the low mantissa bits of a half IS the
//     subnormal number code * 2^-24, which the matrix instruction takes at full rate, so unpacking is an AND (no bias to
//     subtract) and one packed multiply by the sub-block's integer scale.  Integer scale times code fits the 11 bits of
//     a half (Q4_K always; Q6_K rounds products beyond 2048 once).  The super-block's float scale d is applied to the
//     sums: before a block is contracted the sums so far are multiplied by d_before / d (one instruction per sum and
//     256 k), so the sums of a row are always in units of its current d.  Q4_K's minimums are one more matrix
//     instruction per 256 k, the integer mins against the activations' group sums (f16 pairs high + low).
// What bounds it: tiles of few tokens the stream of weight rows (64 token rows of a 128-expert layer, 226 MB of Q4_K gate/up
// and 165 MB of Q6_K down rows: 50 and 41 us; the same launches without unpacking and matrix instructions 46 and 37, a bare
// read in the same pattern 42 and 34; the kernel before, 128-token tiles on one workgroup per CU, 75 and 69); full tiles
// the vector instructions (about 1.4 cycles of them per cycle of matrix instructions: 2048 token rows of 128 experts of
// 2048 x 768, Q4_K / Q6_K, 171 and 114 us, the kernel before 187 and 141 in turn on one box; Q8_0 206 and 111, 226 and 138;
// times of one build differ by some 5 % between boxes).  Two workgroups of twice the rows per wave (64 rows, 250 registers) came to 196 and 153 us there, column
// tiles in sequence in one workgroup (no start-up between them) to nothing: the stream is continuous anyway.
// The order of the additions depends on k alone, not on T or on which tile a token is in: a token's result has the same
// bits wherever it lands.
#include "grouped_fmt.h"

namespace infr {

namespace {

constexpr int kGW = 4;                      // waves per workgroup
__device__ __forceinline__ float4v mfma16(half8 a, half8 b, float4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

template <class F>
constexpr int kWStage = 256 * F::kChunks;              // LDS bytes of 16 rows' step
constexpr int kAPiece = 16 * 1024;                     // an activation piece: 16 groups of 1 KB
constexpr int kXSums = 2048;                           // group sums: two buffers of 16 or 32 tokens, one of 64
template <class F>
constexpr size_t gemm_lds() { return (size_t)kGW * kWStage<F> + 2 * kAPiece + (F::kMin ? kXSums : 0) + kGemmTok * sizeof(float); }

// T: 16-token tiles of the item.  LO: measurement variant, loads, LDS reads and barriers only.
template <class F, bool DOWN, int T, bool LO>
__device__ __forceinline__ void gemm_tile(const GroupedParams& p, const Tile& t, int n0, uint8_t* lds) {
    constexpr int NB = 2;                                              // 16-row weight operands of a wave
    constexpr int KC = 512 / T;                                        // k of an activation piece
    constexpr int SPP = KC > F::kStep ? KC / F::kStep : 1, PPS = F::kStep > KC ? F::kStep / KC : 1;   // steps per piece, pieces per step
    constexpr int G = T;                                               // tokens per 1 KB group of a piece
    constexpr int NC = 16 * NB * F::kChunks, NL = (NC + 63) / 64;      // 16-byte chunks of a wave's step, loads of a lane
    constexpr bool kPartial = F::kBlock < F::kStep;                    // rows need not be whole steps
    constexpr int GPP = F::kStep / 32 / PPS;                           // groups of a step in one piece
    static_assert(PPS <= 2 && NL < 64, "");
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const wl = lds + wave * kWStage<F>;
    uint8_t* const al = lds + kGW * kWStage<F>;
    uint8_t* const xl = al + 2 * kAPiece;
    float* const s_scale = reinterpret_cast<float*>(xl + (F::kMin ? kXSums : 0));   // the tokens' row scales
    const uint32_t al0 = lds_address(al), xl0 = lds_address(xl);

    // the token rows behind the lane's activation loads: requested ahead of the weights, which would hold them up
    constexpr int XB = T == 1 ? 2 : 1;                                 // blocks per load of the group sums
    constexpr int XCH = 2 * XB;                                        // 16-byte chunks per token
    uint32_t asrc[4], xsrc = 0, srow = 0;
    auto row_of = [&](int tok) -> uint32_t {
        const int pr = t.p0 + min(tok, t.cnt - 1);
        return (uint32_t)(DOWN ? pr : p.pair_row[pr]);
    };
#pragma unroll
    for (int q = 0; q < 4; q++) asrc[q] = row_of((wave + 4 * q) * G + lane / (64 / G));
    if (F::kMin) xsrc = row_of(tid / XCH);
    if (!DOWN || !p.out_f16) srow = row_of(tid % (16 * T));
    asm volatile("" ::: "memory");

    // ---- weights: the lane's chunks 64 i + lane of the wave's 32 rows x kChunks
    constexpr int kStepBytes = F::kStep / F::kBlock * F::kBlockBytes;
    const uint32_t row_bytes = (uint32_t)(p.K / F::kBlock) * F::kBlockBytes;
    const uint8_t* const b0 = p.w0 + (size_t)t.e * p.w0_stride;
    const uint8_t* const b1 = DOWN ? b0 : p.w1 + (size_t)t.e * p.w1_stride;
    uint32_t woff[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {          // rows beyond the matrix's last one repeat it
        const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, c = idx - r * F::kChunks;
        const int f = n0 + (DOWN ? 16 * NB * wave + r : 8 * NB * wave + r % (8 * NB));
        woff[i] = (uint32_t)min(f, p.N - 1) * row_bytes + F::src(c, r & 15);
    }
    uint4v w[NL];
    const int n_steps = (p.K + F::kStep - 1) / F::kStep;
    auto request = [&](int s) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            constexpr int kHalf = NC / 2;   // first chunk of the up rows
            const bool pure0 = DOWN || 64 * i + 63 < kHalf, pure1 = 64 * i >= kHalf;
            const uint8_t* const b = (pure0 ? b0 : pure1 ? b1 : (64 * i + lane < kHalf ? b0 : b1)) + (uint32_t)(kStepBytes * s);
            uint32_t off = woff[i];
            if (kPartial && (s + 1) * F::kStep > p.K) {   // chunks behind the row's end are not read (the step's first one instead)
                const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, at = F::src(idx - r * F::kChunks, r & 15);
                if (kStepBytes * s + at >= (int)row_bytes) off -= (uint32_t)at;
            }
            w[i] = ldu<uint4v>(b + off);
        }
    };
    request(0);
    asm volatile("" ::: "memory");

    // ---- activations: a wave's groups of a piece are wave, wave + 4, ..; a group is G whole token pieces of 1024 / G
    // bytes; 16-byte chunk c of token t lies at place c ^ (t & 15), so that sixteen tokens reading the same chunk hit
    // distinct banks
#pragma unroll
    for (int q = 0; q < 4; q++) asrc[q] *= (uint32_t)(p.K / 8);
    const int n_pieces = (p.K + KC - 1) / KC;
    xsrc *= (uint32_t)(p.K / 128);   // group sums: 32 bytes per token and 256 k
    auto fetch = [&](int pc) {   // piece pc into its buffer; nothing is fetched past the last one
        if (pc >= n_pieces) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int grp = wave + 4 * q, a_ch = lane % (64 / G) ^ ((grp * G + lane / (64 / G)) & 15);
            const uint32_t k8 = (uint32_t)min(pc * (KC / 8) + a_ch, p.K / 8 - 1);
            if (grp * G < t.cnt) dma16(reinterpret_cast<const uint4*>(p.a) + (asrc[q] + k8), al0 + (pc & 1) * kAPiece + grp * 1024);
        }
        if constexpr (F::kMin) {
            // two buffers in turn; 64 tokens fill both, but a block's sums then come with its second piece and are read
            // behind it, a barrier before the next block's are fetched
            constexpr int kEvery = KC >= 256 ? 1 : 256 / KC;           // pieces per load of the sums
            if (pc % kEvery == kEvery - 1 && wave * 64 < 16 * T * XCH) {
                const uint32_t c = (uint32_t)min(pc / kEvery * XCH + tid % XCH, p.K / 128 - 1);
                dma16(reinterpret_cast<const uint4*>(p.a_sum) + (xsrc + c), xl0 + (T == 4 ? 0 : (pc & 1) * (kXSums / 2)) + wave * 1024);
            }
        }
    };
    fetch(0);
    if ((!DOWN || !p.out_f16) && tid < 16 * T) s_scale[tid] = p.a_scale[srow];   // read behind barriers
    asm volatile("" ::: "memory");

    float4v acc[NB][T];
    float dcur[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) {
        dcur[n] = 1.0f;
#pragma unroll
        for (int m = 0; m < T; m++) acc[n][m] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    const uint8_t* abase[4];   // groups g & 3; 16 chunks = 256 bytes further for every four groups
#pragma unroll
    for (int g = 0; g < 4; g++) abase[g] = al + col * (1024 / G) + 16 * ((F::a_lane(kq) | F::a_group(g)) ^ col);
    for (int s = 0; s < n_steps; s++) {
        // the wave's 16 rows of one operand at a time through its LDS region, out again as every lane's share of its row
        // (the LDS serves a wave in order: no waiting between the two)
        typename F::Raw raw[NB];
#pragma unroll
        for (int n = 0; n < NB; n++) {
#pragma unroll
            for (int i = 0; i < NL; i++) {
                constexpr int kHalf = NC / NB;
                const int at = 64 * i - n * kHalf;   // first chunk of the load inside the operand
                if (at + 63 < 0 || at >= kHalf) continue;
                if (at >= 0 && at + 63 < kHalf) *reinterpret_cast<uint4v*>(wl + 16 * (at + lane)) = w[i];
                else if (at + lane >= 0 && at + lane < kHalf) *reinterpret_cast<uint4v*>(wl + 16 * (at + lane)) = w[i];
            }
            asm volatile("" ::: "memory");
            F::load(wl, col, kq, raw[n]);
            asm volatile("" ::: "memory");
        }
        // The freed registers are requested again at once; the activation pieces go by barriers.  The piece needed now was
        // fetched ahead of the NL weight loads that may stay in flight.  (A step of two pieces needs the second one before
        // the next step's weights: fetched ahead of them.)
        const bool more = s + 1 < n_steps;
        if (PPS == 1 && more) request(s + 1);
        asm volatile("" ::: "memory");
        if (s % SPP == 0) {
            if (PPS == 1 && more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(NL) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            fetch(s / SPP * PPS + 1);
        }
        if (PPS > 1 && more) request(s + 1);
        asm volatile("" ::: "memory");
        const int groups = kPartial ? (p.K - s * F::kStep) / 32 : F::kStep / 32;   // groups of 32 k from here to the row's end
        if constexpr (kPartial && F::kUnits) {
            if (groups < F::kStep / 32) {
#pragma unroll
                for (int n = 0; n < NB; n++) F::cut(raw[n], kq, groups);
            }
        }
        typename F::St st[NB];
#pragma unroll
        for (int n = 0; n < NB; n++) st[n] = F::prep(raw[n], kq);
        if constexpr (F::kScale && !LO) {
#pragma unroll
            for (int n = 0; n < NB; n++) {
                // a block of d = 0 contributes nothing (its codes count for nothing): the unit stays
                const bool zero = st[n].d == 0.0f;
                const float r = zero ? 1.0f : dcur[n] * __builtin_amdgcn_rcpf(st[n].d);
                dcur[n] = zero ? dcur[n] : st[n].d;
#pragma unroll
                for (int m = 0; m < T; m++)
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[n][m][q] *= r;
            }
        }
#pragma unroll
        for (int sub = 0; sub < PPS; sub++) {
            if (sub) {
                if (more) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(NL) : "memory");
                else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
                fetch(s * PPS + sub + 1);
            }
            const int off = (PPS > 1 ? sub : (s / SPP) & 1) * kAPiece + (SPP > 1 ? (s % SPP) * (F::kStep * 2) : 0);
#pragma unroll
            for (int gp = 0; gp < GPP; gp++) {
                const int g = sub * GPP + gp;
                if (kPartial && (F::kUnits ? g & ~3 : g) >= groups) break;
                half8 b[NB];
                if constexpr (!LO) {
#pragma unroll
                    for (int n = 0; n < NB; n++) b[n] = F::frag(raw[n], st[n], g);
                } else {
#pragma unroll
                    for (int n = 0; n < NB; n++) asm volatile("" : : "v"(*reinterpret_cast<const uint32_t*>(&raw[n])));
                }
#pragma unroll
                for (int m = 0; m < T; m++) {
                    const half8 a = *reinterpret_cast<const half8*>(abase[gp & 3] + off + m * (16 * 1024 / G) + (gp >> 2) * 256);
                    if constexpr (LO) {
                        asm volatile("" : : "v"(a));
                    } else {
#pragma unroll
                        for (int n = 0; n < NB; n++) acc[n][m] = mfma16(a, b[n], acc[n][m]);
                    }
                }
            }
        }
        if constexpr (F::kMin && !LO) {
            const int xo = T == 4 ? 0 : ((s / SPP) & 1) * (kXSums / 2) + (T == 1 ? (s & 1) * 32 : 0);
            float mn[NB];
#pragma unroll
            for (int n = 0; n < NB; n++) mn[n] = -st[n].dmin * __builtin_amdgcn_rcpf(dcur[n]) * (1.0f / kTwo24);
#pragma unroll
            for (int m = 0; m < T; m++) {
                const half8 x = *reinterpret_cast<const half8*>(xl + xo + (16 * m + col) * (16 * XCH) + 16 * (kq & 1));
#pragma unroll
                for (int n = 0; n < NB; n++) {
                    const float4v y = mfma16(x, st[n].mins, float4v{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int q = 0; q < 4; q++) acc[n][m][q] = fmaf(mn[n], y[q], acc[n][m][q]);
                }
            }
        }
    }

    // ---- results through the wave's LDS region, as rows of 64 bytes that leave in 16-byte stores.  Accumulator register q of
    // tile m: token 16 m + 4 kq + q, weight row col of operand n; token 16 m + 4 a + b lies in row 4 b + a, so that a
    // wave's write covers all banks.
    float fin[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) fin[n] = F::kScale ? dcur[n] * kTwo24 : 1.0f;
    const bool half_out = DOWN && p.out_f16;
    const float ds = DOWN && p.down_scale ? p.down_scale[t.e] : 1.0f;
    const int es = half_out ? 2 : 4, vals = 16 / es, fw = n0 + 8 * (DOWN ? 2 : 1) * NB * wave + (lane & 3) * vals;
#pragma unroll
    for (int m = 0; m < T; m++) {
        for (int part = 0; part < (DOWN && !half_out ? 2 : 1); part++) {   // f32 rows of 32 columns leave in halves
            asm volatile("" ::: "memory");
#pragma unroll
            for (int q = 0; q < 4; q++) {
                uint8_t* const o = wl + (4 * q + kq) * 64;
                const int tok = 16 * m + 4 * kq + q;
                if (half_out) {   // without the row's power-of-two scale: the combine multiplies it back in
#pragma unroll
                    for (int n = 0; n < NB; n++) reinterpret_cast<_Float16*>(o)[16 * n + col] = (_Float16)(acc[n][m][q] * fin[n] * ds);
                } else if (DOWN) {
                    const float sc = s_scale[tok] * ds;
                    reinterpret_cast<float*>(o)[col] = (part ? acc[1][m][q] * fin[1] : acc[0][m][q] * fin[0]) * sc;
                } else {
                    const float sc = s_scale[tok];
                    float g = acc[0][m][q] * fin[0] * sc, u = acc[1][m][q] * fin[1] * sc;
                    if (p.act == INFR_ACT_SILU && !p.has_clamp && !p.weight_before) {
                        // silu(g) * u with the hardware exp2 and reciprocal (1 ulp each; the operands were f16)
                        g = g * u * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
                    } else {
                        if (p.weight_before) {
                            const float wp = p.route_w[p.pair_src[t.p0 + min(tok, t.cnt - 1)]];
                            g *= wp;
                            u *= wp;
                        }
                        g = gated_act_fast(p.act, p.has_clamp, p.clamp, g, u);
                    }
                    reinterpret_cast<float*>(o)[col] = g;
                }
            }
            asm volatile("" ::: "memory");
            const int tok = 16 * m + 4 * ((lane >> 2) & 3) + (lane >> 4), f = fw + 16 * part;
            const uint4v v = *reinterpret_cast<const uint4v*>(wl + 16 * lane);
            uint8_t* const dst = reinterpret_cast<uint8_t*>(p.out) + ((size_t)(t.p0 + tok) * p.N + f) * es;
            if (tok >= t.cnt) continue;
            if (f + vals <= p.N && p.N % 8 == 0) {
                *reinterpret_cast<uint4v*>(dst) = v;
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    if (half_out && f + i < p.N) reinterpret_cast<uint16_t*>(dst)[i] = (uint16_t)(v[i >> 1] >> (16 * (i & 1)));
                    if (!half_out && i < 4 && f + i < p.N) reinterpret_cast<uint32_t*>(dst)[i] = v[i & 3];
                }
            }
        }
    }
}

template <class F, bool DOWN, bool LO>
__global__ __launch_bounds__(kGW * 64, 3) void grouped_gemm(GroupedParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_gemm[];
    Tile t;
    int n0;
    if (!tile_item(p.tiles, p.n_tiles_n, p.n_tiles_rcp, kGemmTok, t, n0)) return;
    n0 *= (DOWN ? 32 : 16) * kGW;
    if (t.cnt <= 16) gemm_tile<F, DOWN, 1, LO>(p, t, n0, lds_gemm);
    else if (t.cnt <= 32) gemm_tile<F, DOWN, 2, LO>(p, t, n0, lds_gemm);
    else gemm_tile<F, DOWN, 4, LO>(p, t, n0, lds_gemm);
}

template <class F, bool DOWN>
void gemm(hipStream_t s, const GroupedParams& p) {
    const int width = DOWN ? 32 * kGW : 16 * kGW;
    GroupedParams q = p;
    q.n_tiles_n = (p.N + width - 1) / width;
    q.n_tiles_rcp = (uint32_t)((0x100000000ull + q.n_tiles_n - 1) / q.n_tiles_n);
    const dim3 grid((unsigned)((gemm_max_tiles(p.n_pairs, p.n_expert) * q.n_tiles_n + 7) & ~7));   // whole rounds of the 8 XCDs
    INFR_LDS_LIMIT((grouped_gemm<F, DOWN, false>), (int)gemm_lds<F>());
    if constexpr (std::is_same_v<F, G4K> || std::is_same_v<F, G6K> || std::is_same_v<F, G80>) {
        INFR_LDS_LIMIT((grouped_gemm<F, DOWN, true>), (int)gemm_lds<F>());
        if (p.loads_only) {
            INFR_LAUNCH((grouped_gemm<F, DOWN, true>), grid, dim3(kGW * 64), gemm_lds<F>(), s, q);
            return;
        }
    }
    INFR_LAUNCH((grouped_gemm<F, DOWN, false>), grid, dim3(kGW * 64), gemm_lds<F>(), s, q);
}

}  // namespace

// A row is a whole number of blocks and of 64-k slices.
bool grouped_supported(int dt, int k) {
    if (k <= 0 || k % 64 != 0) return false;
    if (dt == INFR_F16 || dt == INFR_BF16 || dt == INFR_F32) return true;   // rounded to f16 (weights beyond 65504 would not fit)
    const int block = unit_format_block(dt);
    return block != 0 && k % block == 0;
}
bool grouped_k256_supported(int dt, int k) { return k > 0 && k % 256 == 0 && (dt == INFR_Q4K || dt == INFR_Q6K || dt == INFR_Q8_0); }

bool grouped_reads_units(int dt) {
    switch (dt) {
        case INFR_Q4K: case INFR_Q5K: case INFR_Q6K: case INFR_Q8_0: case INFR_Q4_0: case INFR_MXFP4: case INFR_IQ4_XS: return false;
        default: return unit_format_block(dt) != 0;
    }
}

template <bool DOWN>
static void gemm_any(hipStream_t s, int dt, const GroupedParams& p) {
    switch (dt) {
        case INFR_Q4K: gemm<G4K, DOWN>(s, p); break;
        case INFR_Q5K: gemm<G5K, DOWN>(s, p); break;
        case INFR_Q6K: gemm<G6K, DOWN>(s, p); break;
        case INFR_Q8_0: gemm<G80, DOWN>(s, p); break;
        case INFR_Q4_0: gemm<G40, DOWN>(s, p); break;
        case INFR_MXFP4: gemm<GMX, DOWN>(s, p); break;
        case INFR_IQ4_XS: gemm<GIX, DOWN>(s, p); break;
#define INFR_GU(D) case D: gemm<GU<D>, DOWN>(s, p); break;
        INFR_GU(INFR_Q4_1) INFR_GU(INFR_Q5_0) INFR_GU(INFR_Q5_1) INFR_GU(INFR_Q2K) INFR_GU(INFR_Q3K) INFR_GU(INFR_IQ4_NL)
        INFR_GU(INFR_TQ1_0) INFR_GU(INFR_TQ2_0) INFR_GU(INFR_Q2_0) INFR_GU(INFR_NVFP4) INFR_GU(INFR_IQ2_XXS) INFR_GU(INFR_IQ2_XS)
        INFR_GU(INFR_IQ2_S) INFR_GU(INFR_IQ3_XXS) INFR_GU(INFR_IQ3_S) INFR_GU(INFR_IQ1_S) INFR_GU(INFR_IQ1_M)
#undef INFR_GU
        default: break;
    }
}

void launch_grouped_gate_up(hipStream_t s, int dt, const GroupedParams& p) {
    if (dt == INFR_F16 || dt == INFR_BF16 || dt == INFR_F32) launch_grouped_float_gate_up(s, dt, p);
    else gemm_any<false>(s, dt, p);
}

void launch_grouped_down(hipStream_t s, int dt, const GroupedParams& p) {
    if (dt == INFR_F16 || dt == INFR_BF16 || dt == INFR_F32) launch_grouped_float_down(s, dt, p);
    else gemm_any<true>(s, dt, p);
}

}  // namespace infr
