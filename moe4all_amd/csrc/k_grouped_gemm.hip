// Batched Op::MoeFfn and large Linear ops on block-quantised weights: the per-expert GEMMs.
//
// An item is (expert, tile of up to 64 or 128 tokens of its bucket, column tile); a workgroup of four waves takes one.  Two
// kernels: tiles of up to 128 tokens on two workgroups per CU, of up to 64 on three (gemm_tile_log2 says which batch
// takes which); the workgroups of a CU drift apart, so that one's barriers and loads hide behind the other's arithmetic.
//   * A wave owns 32 weight rows (gate/up: 16 gate rows and the 16 up rows of the same features; down: 32 rows) over the
//     whole of K, against all tokens of the tile.  A step of its rows (kStep k) goes from memory straight into an LDS region
//     of its own, consecutive lanes on consecutive 16-byte chunks of a row (a lane reading its own row would touch a cache
//     line per lane), and from there to registers as a row per lane, while the next step (small tiles on two workgroups: the next
//     two) is on its way.
//   * v_mfma_f32_16x16x32_f16: lane = weight row (lane & 15) and a quarter of 32 k (lane / 16).  Tiles of up to 8, 16, 32,
//     64, 96 and 128 tokens have code of their own (Geo).
//   * The tile's activations go from memory straight into LDS too, in pieces of 64 to 256 k, three in turn: two pieces are on
//     their way while one is worked on, with one barrier per piece.
//   * The weight operand holds small integers, not values: a code masked into the low mantissa bits of a half IS the
//     subnormal number code * 2^-24, which the matrix instruction takes at full rate, so unpacking is an AND (no bias to
//     subtract) and one packed multiply by the sub-block's integer scale.  Integer scale times code fits the 11 bits of
//     a half (Q4_K always; Q6_K rounds products beyond 2048 once).  The super-block's float scale d is applied to the
//     sums: before a block is contracted the sums so far are multiplied by d_before / d (one instruction per sum and
//     256 k), so the sums of a row are always in units of its current d.  Q4_K's minimums are one more matrix
//     instruction per 256 k, the integer mins against the activations' group sums (f16 pairs high + low).
// What bounds it.  Tiles of few tokens: the stream of weight rows (64 token rows of a 128-expert layer, 226 MB of Q4_K gate/up and
// 165 MB of Q6_K down rows: 50 and 40 us; a bare read in the same pattern 42 and 34).  Full tiles: a matrix instruction keeps a SIMD's issue
// of vector instructions busy for 8 of its 16 cycles and each vector instruction for 4 (measured: two are free beside
// a matrix instruction, every further one costs its own time), so what counts is vector instructions per matrix instruction:
// 6.2 on 64 tokens per unpacked weight, 2.6 on 128 (4 x 2.6 + 8 = 18.4 cycles for 16).  128 tokens of each of 128 experts
// of 2048 x 768, gate/up and down, us: Q4_K / Q6_K 130 and 88 against 158 and 107 for tiles of 64 with weights through registers,
// Q8_0 154 and 93 (198 and 110).  Half of the rest goes to the barriers and transfers of a step (8900 cycles per step of 256 k
// for two waves per SIMD before the transfers were spread over the matrix instructions, 4600 of them in matrix instructions).
// Tried and left: 256 rows x 128 tokens per workgroup of eight waves (half the activations' traffic, no gain: 150 and 106 us), 64 rows
// per wave (205 and 135: one wave per SIMD hides nothing), four pieces ahead instead of two (the same).
// The order of the additions depends on k alone, not on the tile a token is in: a token's result has the same bits wherever it lands.
#include "grouped_fmt.h"

namespace infr {

namespace {

constexpr int kGW = 4;                      // waves per workgroup
__device__ __forceinline__ float4v mfma16(half8 a, half8 b, float4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// How a tile of 16 M tokens is worked on (M: 1, 2, 4, 6, 8) by a kernel of W workgroups per CU (3: tiles of up to 64 tokens).
template <class F, int M, int W>
struct Geo {
    static constexpr bool kWide = M > 4;
    // k of an activation piece
    static constexpr int KC = M == 4 && W == 2 ? F::kStep / 2 : kWide ? 64 : 256 / M < F::kStep ? 256 / M : F::kStep;
    static constexpr int L = 512 / KC;                                  // tokens per 1 KB group of a piece
    static constexpr int PPS = F::kStep / KC;                           // pieces per step of the weights
    static constexpr int WB = kWide || W == 3 || (M == 4 && KC == 128) ? 1 : 2;   // steps of weights in LDS
    static constexpr int kPiece = kWide || KC * M >= 512 ? 16 * 1024 : 8 * 1024;
    static constexpr int kSums = !F::kMin ? 0 : PPS == 4 ? 512 * (kWide ? 8 : 4) : 2 * (M > 2 ? 512 * M : 1024);   // LDS bytes of the group sums (whole transfers of 1 KB)
};
constexpr int kABufs = 3;                              // pieces in LDS
template <class F>
constexpr int kWLoads = (32 * F::kChunks + 63) / 64;   // 16-byte loads of a lane per step of the wave's 32 rows
template <class F, int M, int W>
constexpr size_t tile_lds() { return (size_t)kGW * 1024 * kWLoads<F> * Geo<F, M, W>::WB + kABufs * Geo<F, M, W>::kPiece + Geo<F, M, W>::kSums; }
template <class F, int W>
constexpr size_t gemm_lds() {
    const size_t a = tile_lds<F, 2, W>(), b = tile_lds<F, 4, W>(), c = tile_lds<F, W == 3 ? 4 : 8, W>();
    return a > b ? (a > c ? a : c) : b > c ? b : c;
}

// Waits until at most N of the wave's loads are in flight; wait_lds for its LDS reads; wait_barrier for both and the other waves.
template <int N>
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory"); }
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <int N>
__device__ __forceinline__ void wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" : : "n"(N) : "memory"); }

// Results of a tile through the wave's LDS region `wl`, as rows of 64 bytes that leave in 16-byte stores.  The gate/up rows of an
// always-on expert are activated as Op::GatedAct does it, exponential and division rounded correctly, so that its results have the
// bits of the separate ops: on the way out, where one copy of the code serves all registers (1500 rows of 256 experts of
// 4096 x 1536 beside one: 1053 us a layer with it, 1054 with the routed experts' exponential).
// SILU: gate/up rows of a routed expert under a plain silu, in code of their own (all forms in one loop: 1.2 to 1.9 % slower batches).
// s_scale: the tokens' row scales in LDS (unit formats; row_scale is then not read).
template <class F, bool DOWN, int NB, int M, bool SILU>
__device__ __forceinline__ void store_rows(const GroupedParams& p, const Tile& t, int n0, int wave, int lane, uint8_t* wl,
                                           const float (&row_scale)[2], const float4v (&acc)[NB][M], const float (&dcur)[NB], const float* s_scale) {
    // Accumulator register q of
    // tile m: token 16 m + 4 kq + q, weight row col of operand n; token 16 m + 4 a + b lies in row 4 b + a, so that a
    // wave's write covers all banks.
    const int col = lane & 15, kq = lane >> 4;
    float fin[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) fin[n] = F::kScale ? dcur[n] * kTwo24 : 1.0f;
    const bool always = !F::kUnits && !SILU && t.e == p.sh_e, half_out = DOWN && p.out_f16 && !always;
    const float ds = DOWN && p.down_scale && !always ? p.down_scale[t.e] : 1.0f;
    uint8_t* const out = reinterpret_cast<uint8_t*>(DOWN && always ? p.sh_out : p.out);
    const int out0 = DOWN && always ? t.p0 - p.sh_p0 : t.p0;
    const int es = half_out ? 2 : 4, vals = 16 / es, fw = n0 + 8 * (DOWN ? 2 : 1) * NB * wave + (lane & 3) * vals;
#pragma unroll
    for (int m = 0; m < M; m++) {
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
                    const float sc = (F::kUnits ? s_scale[tok] : __shfl(row_scale[m >> 2], tok & 63, 64)) * ds;
                    reinterpret_cast<float*>(o)[col] = (part ? acc[1][m][q] * fin[1] : acc[0][m][q] * fin[0]) * sc;
                } else {
                    const float sc = F::kUnits ? s_scale[tok] : __shfl(row_scale[m >> 2], tok & 63, 64);
                    float g = acc[0][m][q] * fin[0] * sc, u = acc[1][m][q] * fin[1] * sc;
                    if (SILU) {
                        g = silu_fast(g) * u;
                    } else if (always) {
                        reinterpret_cast<float*>(o + 1024)[col] = u;
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
            if (!DOWN && !SILU && always) {
                float* const h = reinterpret_cast<float*>(wl) + 4 * lane;
#pragma unroll 1
                for (int i = 0; i < 4; i++) h[i] = gated_act_fn(p.act, p.has_clamp, p.clamp, h[i], h[256 + i]);
                asm volatile("" ::: "memory");
            }
            const int tok = 16 * m + 4 * ((lane >> 2) & 3) + (lane >> 4), f = fw + 16 * part;
            const uint4v v = *reinterpret_cast<const uint4v*>(wl + 16 * lane);
            uint8_t* const dst = out + ((size_t)(out0 + tok) * p.N + f) * es;
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

template <class F, bool DOWN, int NB, int M>
__device__ __forceinline__ void store_tile(const GroupedParams& p, const Tile& t, int n0, int wave, int lane, uint8_t* wl,
                                           const float (&row_scale)[2], const float4v (&acc)[NB][M], const float (&dcur)[NB], const float* s_scale) {
    if (!DOWN && p.act == INFR_ACT_SILU && !p.has_clamp && !p.weight_before && (F::kUnits || t.e != p.sh_e))
        store_rows<F, DOWN, NB, M, true>(p, t, n0, wave, lane, wl, row_scale, acc, dcur, s_scale);
    else
        store_rows<F, DOWN, NB, M, false>(p, t, n0, wave, lane, wl, row_scale, acc, dcur, s_scale);
}

// An item: M 16-token tiles; FEW: one of up to 8 tokens (the rows of the others hold what was there: a token's sums depend on
// its own row alone).  LO: measurement variant, loads, LDS reads and barriers only.
template <class F, bool DOWN, int M, int W, bool LO, bool FEW = false>
__device__ __forceinline__ void gemm_tile(const GroupedParams& p, const Tile& t, int n0, uint8_t* lds) {
    typedef Geo<F, M, W> S;
    constexpr int NB = 2;                                              // 16-row weight operands of a wave
    constexpr int KC = S::KC, PPS = S::PPS, WB = S::WB, G = S::L;
    constexpr int CH = 64 / G;                                         // 16-byte chunks of a token's piece
    constexpr int NC = 16 * NB * F::kChunks, NL = kWLoads<F>;          // 16-byte chunks of a wave's step, loads of a lane
    constexpr int NA = (FEW ? 2 : 4) * M / G;                          // loads of a lane per piece
    constexpr bool kPartial = F::kBlock < F::kStep;                    // rows need not be whole steps
    // One step of weights in LDS and a tile bound by their stream: a wave's weights of the next step are requested as soon as this step's
    // are in registers, ahead of the barrier, not between the matrix instructions.  us per layer, without and with: 34 rows of 256
    // experts of 4096 x 1536 beside one in Q4_K / Q6_K 532 and 524, in Q8_0 783 and 767; 90 rows of 128 experts of 2048 x 768 in
    // Q4_K / Q6_K 122.6 and 121.7, in MXFP4 107.1 and 105.3.  (Not where workgroups have a CU each: 64 rows of 32 experts of
    // 1024 x 512 in Q5_K 46.4 and 47.2; those take the other kernel.)
    constexpr bool kEarly = WB == 1 && M <= 2;
    constexpr int GPP = KC / 32;                                       // groups of 32 k in a piece
    constexpr int N = GPP * M, R = N < 8 ? N : 8;                                  // activation operands of a piece; those read ahead
    static_assert(NA > 0 && 4 * M % G == 0 && (PPS == 1 || PPS == 2 || (PPS == 4 && WB == 1)) && (2 * PPS - 1) * NA + NL < 63, "");
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const wl = lds + wave * (1024 * NL * WB);
    uint8_t* const al = lds + kGW * (1024 * NL * WB);
    uint8_t* const xl = al + kABufs * S::kPiece;
    const uint32_t wl0 = lds_address(wl), al0 = lds_address(al), xl0 = lds_address(xl);

    // ---- weights: the lane's chunks 64 i + lane of the wave's 32 rows x kChunks
    constexpr int kStepBytes = F::kStep / F::kBlock * F::kBlockBytes;
    const uint32_t row_bytes = (uint32_t)(p.K / F::kBlock) * F::kBlockBytes;
    const bool always = t.e == p.sh_e;
    const uint8_t* const b0 = always ? p.sh0 : p.w0 + (size_t)t.e * p.w0_stride;
    const uint8_t* const b1 = DOWN ? b0 : always ? p.sh1 : p.w1 + (size_t)t.e * p.w1_stride;
    uint32_t woff[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {          // rows beyond the matrix's last one repeat it
        const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, c = idx - r * F::kChunks;
        const int f = n0 + (DOWN ? 16 * NB * wave + r : 8 * NB * wave + r % (8 * NB));
        woff[i] = (uint32_t)min(f, p.N - 1) * row_bytes + F::src(c, r & 15);
    }
    const int n_steps = (p.K + F::kStep - 1) / F::kStep, n_pieces = (p.K + KC - 1) / KC;
    auto request1 = [&](int s, int i) {
        constexpr int kHalf = NC / 2;   // first chunk of the up rows
        const bool pure0 = DOWN || 64 * i + 63 < kHalf, pure1 = 64 * i >= kHalf;
        uint32_t off = woff[i];
        if (kPartial && (s + 1) * F::kStep > p.K) {   // chunks behind the row's end are not read (the step's first one instead)
            const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, at = F::src(idx - r * F::kChunks, r & 15);
            if (kStepBytes * s + at >= (int)row_bytes) off -= (uint32_t)at;
        }
        const uint32_t into = wl0 + (WB == 2 ? (s & 1) * (1024 * NL) : 0) + 1024 * i;
        if (pure0 || pure1) dma16((pure0 ? b0 : b1) + (uint32_t)(kStepBytes * s), off, into);
        else dma16((64 * i + lane < kHalf ? b0 : b1) + (uint32_t)(kStepBytes * s) + off, into);
    };
    auto request = [&](int s) {
#pragma unroll
        for (int i = 0; i < NL; i++) request1(s, i);
    };
    typename F::Raw raw[NB];
    typename F::St st[NB];
    auto read_weights = [&](int s, int n, typename F::Raw& r) {
        F::load(wl + (WB == 2 ? (s & 1) * (1024 * NL) : 0) + n * 256 * F::kChunks, col, kq, r);
    };

    // ---- The token rows behind the lane's activation loads.  Gate/up looks them up: the table comes through LDS (the place of the
    // third piece, unused until step 0 is past its first barrier) ahead of the first weights, so that neither waits for the other; a
    // load to registers would have to be waited for first, as the compiler's wait covers whatever is requested behind it.
    constexpr int NR = DOWN ? 0 : S::kWide ? 2 : 1;   // loads of the table
    const uint32_t* const rows = reinterpret_cast<const uint32_t*>(al + 2 * S::kPiece + wave * 512);
#pragma unroll
    for (int j = 0; j < NR; j++) dma4(p.pair_row, 4u * (uint32_t)(t.p0 + min(64 * j + lane, t.cnt - 1)), al0 + 2 * S::kPiece + wave * 512 + 256 * j);
    request(0);
    if (!DOWN) wait_loads<NL>();
    auto row_of = [&](int tok) -> uint32_t {
        const int i = min(tok, t.cnt - 1);
        return DOWN ? (uint32_t)(t.p0 + i) : rows[i];
    };
    uint32_t asrc[NA], xsrc = 0;
#pragma unroll
    for (int q = 0; q < NA; q++) asrc[q] = row_of((wave + 4 * q) * G + lane / CH);
    if (F::kMin) xsrc = row_of(tid / 2);
    float row_scale[2] = {1.0f, 1.0f};   // scales of tokens `lane` and 64 + lane
    if (!DOWN || !p.out_f16 || always) {
#pragma unroll
        for (int j = 0; j < (S::kWide ? 2 : 1); j++) row_scale[j] = p.a_scale[row_of(64 * j + lane)];
    }
    asm volatile("" ::: "memory");

    // ---- activations: a wave's groups of a piece are wave, wave + 4, ..; a group is G whole token pieces of 1024 / G bytes;
    // 16-byte chunk c of token t lies at place c ^ turn(t), so that sixteen tokens reading the same chunk hit distinct banks
    auto turn = [](int tok) { return CH >= 16 ? tok & 15 : rot7(tok) & (CH - 1); };
#pragma unroll
    for (int q = 0; q < NA; q++) asrc[q] *= (uint32_t)(p.K / 8);
    xsrc *= (uint32_t)(p.K / 128);   // group sums: 32 bytes per token and 256 k
    // behind the last piece the row's end is fetched again, into a place that nothing reads any more
    auto fetch1 = [&](int pc, int buf, int q) {
        const int grp = wave + 4 * q, a_ch = (lane % CH) ^ turn(grp * G + lane / CH);
        const uint32_t k8 = KC == 64 ? (uint32_t)(min(pc, n_pieces - 1) * (KC / 8) + a_ch) : (uint32_t)min(pc * (KC / 8) + a_ch, p.K / 8 - 1);
        dma16(reinterpret_cast<const uint4*>(p.a) + (asrc[q] + k8), al0 + buf * S::kPiece + grp * 1024);
    };
    auto fetch = [&](int pc, int buf) {
#pragma unroll
        for (int q = 0; q < NA; q++) fetch1(pc, buf, q);
    };
    // a step's group sums: fetched behind its first barrier into one buffer where it has three more, else a step ahead into two in turn
    auto fetch_sums = [&](int s) {
        if constexpr (F::kMin) {
            if (s < n_steps && wave * 64 < 32 * M)
                dma16(reinterpret_cast<const uint4*>(p.a_sum) + (xsrc + (uint32_t)(2 * s + (tid & 1))),
                      xl0 + (PPS == 4 ? 0 : (s & 1) * (S::kSums / 2)) + wave * 1024);
        }
    };

    // ---- Transfers land in the order they were requested in; what may be in flight where something is waited for is what was
    // requested behind it.  The order of a step: behind its first barrier group sums, the piece after next, the weights of
    // the next step (WB = 1) or of the one after it (WB = 2); behind each further barrier the piece after next; kEarly: at its end
    // the weights of the step after next.  Here the same order as if two steps had come before.
    const bool two = WB == 2 && n_steps > 1;
    if (PPS != 4) fetch_sums(0);
    fetch(0, 0);
    if (PPS == 1) fetch(1, 1);
    if (two) request(1);
    if (PPS != 1) fetch(1, 1);
    if (two) wait_loads<(PPS == 1 ? 1 : 2) * NA + NL>();
    else wait_loads<(PPS == 1 ? 1 : 2) * NA>();
#pragma unroll
    for (int n = 0; n < NB; n++) read_weights(0, n, raw[n]);
    if (kEarly && n_steps > 1) {
        wait_lds();
        request(1);
    }
#pragma unroll
    for (int n = 0; n < NB; n++) st[n] = F::prep(raw[n], kq);

    float4v acc[NB][M];
    float dcur[NB];
#pragma unroll
    for (int n = 0; n < NB; n++) {
        dcur[n] = 1.0f;
#pragma unroll
        for (int m = 0; m < M; m++) acc[n][m] = float4v{0.f, 0.f, 0.f, 0.f};
    }
    const uint8_t* abase[4];   // groups g & 3; 16 chunks = 256 bytes further for every four groups
#pragma unroll
    for (int g = 0; g < 4; g++) abase[g] = al + col * (1024 / G) + 16 * (((F::a_lane(kq) | F::a_group(g)) & (CH - 1)) ^ turn(col));
    int cur = 0;               // buffer of the piece at hand

    // What a step needs beyond its matrix instructions is spread between them: the transfers one by one (in a burst behind
    // the barrier they held all waves up), the next group's unpacking, the next step's weights from LDS, the minimums.
    // more: steps behind this one (2: or more)
    auto step = [&](int s, auto more_c) {
        constexpr int kMore = decltype(more_c)::value;
        const bool more = kMore < 0 ? s + 1 < n_steps : kMore > 0, req = kMore < 0 ? more : kMore >= WB;   // req: this step requests weights
        const int p0 = s * PPS;
        const int groups = kPartial && !more ? (p.K - s * F::kStep) / 32 : F::kStep / 32;   // groups of 32 k from here to the row's end
        float ratio[NB];   // of the block's unit to the one before: the sums so far are multiplied by it
#pragma unroll
        for (int n = 0; n < NB; n++) {
            ratio[n] = 1.0f;
            if constexpr (F::kScale && !LO) {
                // a block of d = 0 contributes nothing (its codes count for nothing): the unit stays
                const bool zero = st[n].d == 0.0f;
                ratio[n] = zero ? 1.0f : dcur[n] * __builtin_amdgcn_rcpf(st[n].d);
                dcur[n] = zero ? dcur[n] : st[n].d;
            }
        }
        typename F::Raw next[NB];
        typename F::St next_st[NB];
#pragma unroll
        for (int sub = 0; sub < PPS; sub++) {
            if (kPartial && !more && sub && p0 + sub >= n_pieces) break;
            if (PPS == 4) {
                if (sub == 3) {
                    if (more) wait_barrier<NA>();
                    else wait_barrier<0>();
                } else if (sub > 0 && req) {
                    wait_barrier<NL + NA>();
                } else {
                    wait_barrier<NA>();
                }
            } else if (PPS == 2) {
                if (sub == 0) {
                    if ((WB == 2 || kEarly) && more) wait_barrier<NL + NA>();
                    else wait_barrier<NA>();
                } else if (kEarly ? more : req) {
                    wait_barrier<NL + NA>();
                } else if (more) {
                    wait_barrier<NA>();
                } else {
                    wait_barrier<0>();
                }
            } else {
                wait_barrier<63>();   // (in order ahead of this step's weights, which have been read)
            }
            const uint32_t off = cur * S::kPiece;
            const int into = cur == 0 ? 2 : cur - 1;   // the buffer of the piece before
            cur = cur == 2 ? 0 : cur + 1;
            if (sub == 0) fetch_sums(PPS == 4 ? s : s + 1);
            // (no pieces follow those of the last step; where that is not known here, the row's end is fetched again)
            const int na = kMore == 0 && sub + 2 >= PPS ? 0 : NA, nd = na + (sub == 0 && !kEarly && (kMore < 0 || req) ? NL : 0);
            const bool mins = F::kMin && !LO && sub == PPS - 1;
            const int ns = mins ? N + M : N;
            auto operand = [&](int i) {
                if (i < N) return *reinterpret_cast<const half8*>(abase[(i / M) & 3] + off + (i % M) * (16 * 1024 / G) + (i / M >> 2) * 256);
                return *reinterpret_cast<const half8*>(xl + (PPS == 4 ? 0 : (s & 1) * (S::kSums / 2)) + (16 * (i - N) + col) * 32 + 16 * (kq & 1));
            };
            auto unpack = [&](int gp, int n) -> half8 {
                if constexpr (LO) {
                    asm volatile("" : : "v"(*reinterpret_cast<const uint32_t*>(&raw[n])));
                    return half8{};
                } else {
                    return F::frag(raw[n], st[n], sub * GPP + gp);
                }
            };
            half8 a[R], b[2][NB];
            float mn[NB];
            float4v y[NB];
#pragma unroll
            for (int i = 0; i < R; i++) a[i] = operand(i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int n = 0; n < NB; n++) b[0][n] = unpack(0, n);
#pragma unroll
            for (int i = 0; i < N + M; i++) {
                if (i >= ns) break;
                const int gp = i / M, m = i % M;
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (LO) {
                    asm volatile("" : : "v"(a[i % R]));
                } else if (i < N) {
                    if (!kPartial || kMore > 0 || sub * GPP + gp < groups) {
#pragma unroll
                        for (int n = 0; n < NB; n++) {
                            if (F::kScale && sub == 0 && gp == 0) {
#pragma unroll
                                for (int q = 0; q < 4; q++) acc[n][m][q] *= ratio[n];
                            }
                            acc[n][m] = mfma16(a[i % R], b[gp & 1][n], acc[n][m]);
                        }
                    }
                } else if constexpr (F::kMin) {
                    const int before = m ? m - 1 : 0;
                    float4v z[NB];
#pragma unroll
                    for (int n = 0; n < NB; n++) z[n] = mfma16(a[i % R], st[n].mins, float4v{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                    for (int n = 0; n < NB; n++) {
                        if (m) {
#pragma unroll
                            for (int q = 0; q < 4; q++) acc[n][before][q] = fmaf(mn[n], y[n][q], acc[n][before][q]);
                        } else {
                            mn[n] = -st[n].dmin * __builtin_amdgcn_rcpf(dcur[n]) * (1.0f / kTwo24);
                        }
                        y[n] = z[n];
                    }
                }
                if (i + R < ns) a[i % R] = operand(i + R);
#pragma unroll
                for (int j = 0; j < NA + NL; j++) {
                    if (j >= nd || j * N / nd != i) continue;
                    if (j < na) fetch1(p0 + sub + 2, into, j);
                    else if (kMore >= 0 || req) request1(s + WB, j - na);
                }
#pragma unroll
                for (int n = 0; n < NB; n++)
                    if (i < N && gp + 1 < GPP && m == M * (2 * n + 1) / 4) b[(gp + 1) & 1][n] = unpack(gp + 1, n);
                if (kMore > 0 && PPS == 4 && sub == 3) {
                    // the next step's weights, which landed by the last barrier
#pragma unroll
                    for (int n = 0; n < NB; n++) {
                        if (i == 1 + n) read_weights(s + 1, n, next[n]);
                        if (i == (N > 8 ? M + 2 : 4) + n) next_st[n] = F::prep(next[n], kq);
                    }
                }
            }
            if constexpr (F::kMin && !LO) {
                if (mins) {
#pragma unroll
                    for (int n = 0; n < NB; n++)
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[n][M - 1][q] = fmaf(mn[n], y[n][q], acc[n][M - 1][q]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (more) {
            if (PPS != 4) {
                wait_loads<kEarly ? PPS * NA : WB == 1 ? (PPS - 1) * NA : (2 * PPS - 1) * NA + (kMore >= WB ? NL : 0)>();
#pragma unroll
                for (int n = 0; n < NB; n++) read_weights(s + 1, n, next[n]);
                if (kEarly && s + 2 < n_steps) {
                    wait_lds();
                    request(s + 2);
                }
#pragma unroll
                for (int n = 0; n < NB; n++) next_st[n] = F::prep(next[n], kq);
            }
#pragma unroll
            for (int n = 0; n < NB; n++) raw[n] = next[n], st[n] = next_st[n];
        }
    };
    int s = 0;
    if constexpr (M <= 2 && WB == 1 && !kPartial) {   // one copy of the code: it is fetched anew by every launch
        for (; s < n_steps; s++) step(s, std::integral_constant<int, -1>{});
    } else {
        for (; s + WB < n_steps; s++) step(s, std::integral_constant<int, 2>{});
        if (WB == 2 && s + 1 < n_steps) step(s++, std::integral_constant<int, 1>{});
        step(s, std::integral_constant<int, 0>{});
    }
    wait_loads<0>();   // no transfer outlives the item
    store_tile<F, DOWN, NB, M>(p, t, n0, wave, lane, wl, row_scale, acc, dcur, nullptr);
}

// The formats that go through the 32-element unit decoder (units.h), bound by the decoding: tiles of 16 T tokens, T = 1, 2, 4, three
// workgroups per CU.  Weights come to registers a step ahead (a step of three tiles in LDS would leave room for two workgroups:
// 60 token rows of 128 experts of 2048 x 768 in Q5_1 79 + 45 us, 71 + 39 this way) and go row by row through 16 rows of LDS;
// activations in two pieces of 512 / T k in turn, with one barrier per piece.
template <class F>
constexpr size_t unit_lds() { return (size_t)kGW * 256 * F::kChunks + 2 * 16 * 1024 + 64 * sizeof(float); }
template <class F, bool DOWN, int T>
__device__ __forceinline__ void unit_tile(const GroupedParams& p, const Tile& t, int n0, uint8_t* lds) {
    constexpr int NB = 2;                                              // 16-row weight operands of a wave
    constexpr bool kPartial = F::kBlock < F::kStep;                    // rows need not be whole steps
    constexpr int KC = 512 / T;                                        // k of an activation piece
    constexpr int SPP = KC > F::kStep ? KC / F::kStep : 1, PPS = F::kStep > KC ? F::kStep / KC : 1;   // steps per piece, pieces per step
    constexpr int G = T;                                               // tokens per 1 KB group of a piece
    constexpr int kPiece = 16 * 1024;
    constexpr int NC = 16 * NB * F::kChunks, NL = (NC + 63) / 64;      // 16-byte chunks of a wave's step, loads of a lane
    constexpr int GPP = F::kStep / 32 / PPS;                           // groups of a step in one piece
    static_assert(PPS <= 2 && NL < 64, "");
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const wl = lds + wave * (256 * F::kChunks);
    uint8_t* const al = lds + kGW * (256 * F::kChunks);
    float* const s_scale = reinterpret_cast<float*>(al + 2 * kPiece);   // the tokens' row scales
    const uint32_t al0 = lds_address(al);

    // the token rows behind the lane's activation loads: requested ahead of the weights, which would hold them up
    uint32_t asrc[4], srow = 0;
    auto row_of = [&](int tok) -> uint32_t {
        const int pr = t.p0 + min(tok, t.cnt - 1);
        return (uint32_t)(DOWN ? pr : p.pair_row[pr]);
    };
#pragma unroll
    for (int q = 0; q < 4; q++) asrc[q] = row_of((wave + 4 * q) * G + lane / (64 / G));
    if (!DOWN || !p.out_f16) srow = row_of(lane);
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

    // ---- activations: as in gemm_tile
#pragma unroll
    for (int q = 0; q < 4; q++) asrc[q] *= (uint32_t)(p.K / 8);
    const int n_pieces = (p.K + KC - 1) / KC;
    auto fetch = [&](int pc) {   // piece pc into its buffer; nothing is fetched past the last one
        if (pc >= n_pieces) return;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int grp = wave + 4 * q, a_ch = lane % (64 / G) ^ ((grp * G + lane / (64 / G)) & 15);
            const uint32_t k8 = (uint32_t)min(pc * (KC / 8) + a_ch, p.K / 8 - 1);
            if (grp * G < t.cnt) dma16(reinterpret_cast<const uint4*>(p.a) + (asrc[q] + k8), al0 + (pc & 1) * kPiece + grp * 1024);
        }
    };
    fetch(0);
    // (behind the last step, where they are needed, a memory latency per item; in a register until then, more spills)
    if ((!DOWN || !p.out_f16) && wave == 0) s_scale[lane] = p.a_scale[srow];   // read behind barriers
    asm volatile("" ::: "memory");

    float4v acc[NB][T];
#pragma unroll
    for (int n = 0; n < NB; n++)
#pragma unroll
        for (int m = 0; m < T; m++) acc[n][m] = float4v{0.f, 0.f, 0.f, 0.f};
    const uint8_t* abase[4];   // groups g & 3; 16 chunks = 256 bytes further for every four groups
#pragma unroll
    for (int g = 0; g < 4; g++) abase[g] = al + col * (1024 / G) + 16 * ((F::a_lane(kq) | F::a_group(g)) ^ col);
    for (int s = 0; s < n_steps; s++) {
        // the wave's 16 rows of one operand at a time through its LDS region, out again as every lane's units
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
            if (PPS == 1 && more) wait_barrier<NL>();
            else wait_barrier<0>();
            fetch(s / SPP * PPS + 1);
        }
        if (PPS > 1 && more) request(s + 1);
        asm volatile("" ::: "memory");
        // groups of 32 k from here to the row's end: known where rows are whole steps (tests and cuts left in for those too: Q3_K 2 to 8 %)
        const int groups = kPartial ? (p.K - s * F::kStep) / 32 : F::kStep / 32;
        if (kPartial && groups < F::kStep / 32) {
#pragma unroll
            for (int n = 0; n < NB; n++) F::cut(raw[n], kq, groups);
        }
        typename F::St st[NB];
#pragma unroll
        for (int sub = 0; sub < PPS; sub++) {
            if (sub) {
                if (more) wait_barrier<NL>();
                else wait_barrier<0>();
                fetch(s * PPS + sub + 1);
            }
            const int off = (PPS > 1 ? sub : (s / SPP) & 1) * kPiece + (SPP > 1 ? (s % SPP) * (F::kStep * 2) : 0);
#pragma unroll
            for (int gp = 0; gp < GPP; gp++) {
                const int g = sub * GPP + gp;
                if ((g & ~3) >= groups) break;
                half8 b[NB];
#pragma unroll
                for (int n = 0; n < NB; n++) b[n] = F::frag(raw[n], st[n], g);
#pragma unroll
                for (int m = 0; m < T; m++) {
                    const half8 a = *reinterpret_cast<const half8*>(abase[gp & 3] + off + m * (16 * 1024 / G) + (gp >> 2) * 256);
#pragma unroll
                    for (int n = 0; n < NB; n++) acc[n][m] = mfma16(a, b[n], acc[n][m]);
                }
            }
        }
    }
    const float row_scale[2] = {1.0f, 1.0f};
    const float unit[NB] = {1.0f, 1.0f};
    store_tile<F, DOWN, NB, T>(p, t, n0, wave, lane, wl, row_scale, acc, unit, s_scale);
}

// The workgroup's item: the tiles in the table's order, a tile's columns side by side.  Workgroups go to the 8 XCDs round-robin, so
// the columns of a tile spread over all of them and every XCD has the same mix of work at any time; large tiles come first,
// so that none is left running alone at the end.  (A contiguous eighth of the items per XCD, experts ascending, has an expert's
// tile read from one L2 only, but left the CUs idle for 8 to 39 % of a launch with skewed experts: 1500 token rows of 256
// experts of 4096 x 1536 1331 us a layer, so 1184, 512 rows of 128 experts of 2048 x 768 in Q8_0 210 and 198; classes without order
// inside: neighbouring experts' weights read one after the other, 1 to 2 % of a batch of small tiles.)  deal_log2 = 3, launches with
// about one item per CU, where there is nothing to balance: tile 8 i + j on XCD j, whose L2 alone reads the tile's rows.  Uniform;
// false when there is nothing to do (the grid is an upper bound).
__device__ __forceinline__ bool gemm_item(const GroupedParams& p, Tile& t, int& col) {
    const int item = (int)blockIdx.x >> p.deal_log2, group = p.n_tiles_n == 1 ? item : (int)__umulhi((uint32_t)item, p.n_tiles_rcp);   // item / n_tiles_n: exact below 2^32 / n_tiles_n
    const int tile = (group << p.deal_log2) + ((int)blockIdx.x & ((1 << p.deal_log2) - 1));
    // expert, first pair, pairs: read beside the number of tiles, not behind it (the grid is within the table)
    const int n_tiles = p.tiles[0].x;
    const int4 b = p.tiles[1 + tile];
    asm volatile("" : : "s"(n_tiles), "s"(b.x), "s"(b.y), "s"(b.z));
    if (tile >= n_tiles) return false;
    t = Tile{b.x, b.y, b.z};
    col = item - group * p.n_tiles_n;
    return true;
}

template <class F, bool DOWN, int W, bool LO>
__global__ __launch_bounds__(kGW * 64, W) void grouped_gemm(GroupedParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_gemm[];
    Tile t;
    int n0;
    if (!gemm_item(p, t, n0)) return;
    n0 *= (DOWN ? 32 : 16) * kGW;
    constexpr bool kFew = Geo<F, 1, W>::L <= 2;
    if (kFew && t.cnt <= 8) gemm_tile<F, DOWN, 1, W, LO, kFew>(p, t, n0, lds_gemm);
    else if (t.cnt <= 16) gemm_tile<F, DOWN, 1, W, LO>(p, t, n0, lds_gemm);
    else if (t.cnt <= 32) gemm_tile<F, DOWN, 2, W, LO>(p, t, n0, lds_gemm);
    else if (W == 3 || t.cnt <= 64) gemm_tile<F, DOWN, 4, W, LO>(p, t, n0, lds_gemm);
    else if constexpr (W == 2) {
        if (t.cnt <= 96) gemm_tile<F, DOWN, 6, W, LO>(p, t, n0, lds_gemm);
        else gemm_tile<F, DOWN, 8, W, LO>(p, t, n0, lds_gemm);
    }
}

template <class F, bool DOWN, int W>
void gemm_launch(hipStream_t s, const GroupedParams& q, dim3 grid) {
    INFR_LDS_LIMIT((grouped_gemm<F, DOWN, W, false>), (int)(gemm_lds<F, W>()));
    if constexpr (std::is_same_v<F, G4K> || std::is_same_v<F, G6K> || std::is_same_v<F, G80>) {
        INFR_LDS_LIMIT((grouped_gemm<F, DOWN, W, true>), (int)(gemm_lds<F, W>()));
        if (q.loads_only) {
            INFR_LAUNCH((grouped_gemm<F, DOWN, W, true>), grid, dim3(kGW * 64), (gemm_lds<F, W>()), s, q);
            return;
        }
    }
    INFR_LAUNCH((grouped_gemm<F, DOWN, W, false>), grid, dim3(kGW * 64), (gemm_lds<F, W>()), s, q);
}

// The same for a dense matrix in a format of the unit decoder: a contiguous eighth of the items per XCD, in groups of up to kGroupTiles
// tiles, columns outside.  Every item of such a launch costs about the same, and its weights, decoded by every workgroup that reads them,
// are the smaller part: the XCDs share out the tiles' rows.  us per Linear, this order and the other: 512 rows of 2048 x 2048 in Q3_K
// 29.1 and 30.0, IQ3_S 38.8 and 39.7, 2048 rows of 4096 x 4096 in Q5_1 the same.
// The tiles are the rows in turn, so no table is read (two memory latencies per workgroup less: 512 rows of 2048 x 2048 in IQ3_S 39.1 and
// 38.7, 2048 rows of 4096 x 1024 in Q4_1 56.4 and 55.5).
__device__ __forceinline__ bool dense_item(const GroupedParams& p, Tile& t, int& col) {
    const int tile = 1 << p.tile_log2, n_tiles = (p.n_pairs + tile - 1) >> p.tile_log2, n_items = n_tiles * p.n_tiles_n, per = (n_items + 7) >> 3;
    const int k = (int)(blockIdx.x >> 3), item = (int)(blockIdx.x & 7) * per + k;
    if (k >= per || item >= n_items) return false;
    const int some = p.n_tiles_n == 1 ? item : (int)__umulhi((uint32_t)item, p.n_tiles_rcp), first = some & ~(kGroupTiles - 1);
    const int in_group = min(kGroupTiles, n_tiles - first), r = item - first * p.n_tiles_n;
    col = group_column((uint32_t)r, in_group);
    const int p0 = (first + r - col * in_group) << p.tile_log2;
    t = Tile{0, p0, min(tile, p.n_pairs - p0)};
    return true;
}

template <class F, bool DOWN>
__global__ __launch_bounds__(kGW * 64, 3) void grouped_gemm_units(GroupedParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_gemm[];
    Tile t;
    int n0;
    if constexpr (DOWN) {
        asm volatile("" : : "s"(p.dense), "s"(p.n_tiles_n), "s"(p.n_tiles_rcp), "s"(p.n_pairs), "s"(p.tiles));   // in one round trip
        if (!(p.dense ? dense_item(p, t, n0) : gemm_item(p, t, n0))) return;
    } else {
        if (!gemm_item(p, t, n0)) return;
    }
    n0 *= (DOWN ? 32 : 16) * kGW;
    if (t.cnt <= 16) unit_tile<F, DOWN, 1>(p, t, n0, lds_gemm);
    else if (t.cnt <= 32) unit_tile<F, DOWN, 2>(p, t, n0, lds_gemm);
    else unit_tile<F, DOWN, 4>(p, t, n0, lds_gemm);
}

// Where a tile's columns go to one XCD (gemm_item): up to one and a half items per CU by the launch's bound, and four tiles per XCD
// (of fewer the XCDs' shares would differ).  us, columns side by side and so: 12 layers of 32 experts of 1024 x 512, 48 rows in Q4_K / Q6_K
// 527 and 519, Q5_K / Q6_K 550 and 537, MXFP4 473 and 462, 90 rows 553 and 543, 561 and 554, 521 and 516; 2048 rows of a dense 4096 x 1024 in Q8_0
// 52.7 and 48.4.  Larger launches of skewed buckets lose by it (200 rows of the same experts, Zipf(1.1): 621 and 642).
constexpr int kDealTiles = 32, kDealItems = 384;
template <class F, bool DOWN>
void gemm(hipStream_t s, const GroupedParams& p) {
    GroupedParams q = p;
    const int width = DOWN ? 32 * kGW : 16 * kGW;
    q.n_tiles_n = (p.N + width - 1) / width;
    q.n_tiles_rcp = (uint32_t)((0x100000000ull + q.n_tiles_n - 1) / q.n_tiles_n);
    const int tiles = gemm_max_tiles(p.n_pairs, p.n_expert, 1 << p.tile_log2);
    q.deal_log2 = !F::kUnits && tiles >= kDealTiles && tiles * q.n_tiles_n <= kDealItems ? 3 : 0;
    const int items = (q.deal_log2 ? (tiles + 7) & ~7 : tiles) * q.n_tiles_n;
    const dim3 grid((unsigned)(F::kUnits && DOWN && p.dense ? (items + 7) & ~7 : items));   // (dense_item: whole rounds of the 8 XCDs)
    if constexpr (F::kUnits) {
        INFR_LDS_LIMIT((grouped_gemm_units<F, DOWN>), (int)unit_lds<F>());
        INFR_LAUNCH((grouped_gemm_units<F, DOWN>), grid, dim3(kGW * 64), unit_lds<F>(), s, q);
    } else if (p.tile_log2 == 7) {
        gemm_launch<F, DOWN, 2>(s, q, grid);
    } else {
        gemm_launch<F, DOWN, 3>(s, q, grid);
    }
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

bool gemm_takes_always(int dt) { return unit_format_block(dt) != 0 && !grouped_reads_units(dt); }

// Tiles of 64 pairs on three workgroups per CU, or of 128 on two?  128 tokens share a weight's unpacking, and the kernel of two has
// the LDS for two steps of weights ahead of a small tile; three hide more of everything else.  us per layer, 64 | 128 (128 experts of
// 2048 x 768 unless said otherwise; uniform routing, then Zipf(1.1) where given):
//   Q4_K / Q6_K   34 rows 114 | 111, 64 rows 119 | 118, 90 rows 122 82 | 121 83, 200 rows 132 105 | 132 100, 300 rows 140 119 | 142 116,
//                 512 rows 167 165 | 175 164, 1024 rows 237 242 | 227 236, 2048 rows 383 372 | 373 355
//   Q5_K / Q6_K   34 rows 124 | 121, 64 rows 130 | 128, 130 rows 137 92 | 136 96, 200 rows 143 111 | 143 105, 300 rows 150 124 | 153 122,
//                 512 rows 181 179 | 186 174, 1024 rows 256 262 | 238 250
//   Q8_0          34 rows 156 | 152, 90 rows 169 106 | 165 99, 200 rows 178 131 | 176 123, 512 rows 214 210 | 208 199, 2048 rows 437 413 | 406 387
//   Q4_0          34 rows 110 | 112, 90 rows 115 77 | 119 78, 200 rows 125 99 | 126 96, 300 rows 130 111 | 138 109, 512 rows 161 154 | 172 156
//   IQ4_XS        34 rows 126 | 127, 90 rows 132 86 | 133 86, 300 rows 143 121 | 151 117, 512 rows 171 169 | 180 166, 1024 rows 244 255 | 231 243
//   MXFP4         34 rows 99 | 97, 90 rows 108 71 | 105 70, 200 rows 116 92 | 113 86, 300 rows 123 103 | 121 100, 512 rows 148 140 | 157 137
//   256 experts of 4096 x 1536 beside one: Q4_K / Q6_K 34 rows 524 | 539, 64 rows 689 | 706, 90 rows 797 465 | 810 471;  Q5_K / Q6_K 64 rows
//                 787 | 797, 90 rows 914 524 | 919 526;  Q4_0 200 rows 670 416 | 697 416;  Q8_0 34 rows 767 | 760, 200 rows 1137 656 | 1102 630;
//                 MXFP4 34 rows 614 | 614, 200 rows 611 379 | 596 371
//   32 experts of 1024 x 512: Q8_0 34 rows 48.5 | 43.5, 90 rows 51.8 53.0 | 48.5 55.8, 130 rows 53.4 54.8 | 51.8 58.1, 200 rows 55.0 56.1 |
//                 54.5 59.6;  Q4_K / Q6_K 34 rows 43.3 | 42.8, 90 rows 46.7 49.8 | 47.6 54.2, 200 rows 52.6 52.0 | 51.9 58.6;  64 rows in Q4_K /
//                 Q6_K 45.5 | 46.1, Q5_K / Q6_K 47.2 | 47.5, MXFP4 43.4 | 40.9
//   8 experts of 4096 x 14336, top-2, Q4_K / Q6_K: 34 rows 241 | 230, 100 rows 272 328 | 264 323, 1000 rows 1155 1161 | 1003 1021;  64 of
//                 4352 x 1024, top-4: 64 rows 164 | 155, 100 rows 167 136 | 158 140, 1000 rows 289 297 | 266 286;  32 of 2048 x 5120, top-4:
//                 64 rows 178 | 175, 100 rows 182 172 | 182 179, 1000 rows 486 511 | 453 465;  Q8_0 and Q5_K / Q6_K on these shapes alike
// So with 128: rows beyond 4096; from 40 pairs per expert on if that leaves three rounds of workgroups; Q8_0; below 24 pairs per expert MXFP4 and, in
// rows of 2048 and less (longer ones hide a workgroup's start by themselves), Q4_K and Q5_K.  Launches that do not fill the chip
// once: 64, so that a large bucket is spread over more workgroups, but up to 64 rows, which both cut alike, and for Q8_0 below 40 pairs per
// expert (uniform routing gains what skewed loses) 128.
int gemm_tile_log2(int gate_dt, int down_dt, int rows, int n_pairs, int n_expert, int ne, int nff) {
    if (grouped_reads_units(gate_dt) || grouped_reads_units(down_dt)) return 6;
    const int mean = n_pairs / n_expert;
    const bool k_quant = gate_dt == INFR_Q4K || gate_dt == INFR_Q5K;
    if (ne > 4096 || nff > 4096) return 7;
    if ((int64_t)gemm_max_tiles(n_pairs, n_expert, 128) * ((nff + 63) / 64) < 512) return rows <= 64 || (gate_dt == INFR_Q8_0 && mean < 40) ? 7 : 6;
    if (gate_dt == INFR_Q8_0) return 7;
    if (mean >= 40) return (int64_t)gemm_max_tiles(n_pairs, n_expert, 128) * ((nff + 63) / 64) >= 3 * 512 ? 7 : 6;
    return mean < 24 && (gate_dt == INFR_MXFP4 || (k_quant && ne <= 2048)) ? 7 : 6;
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
