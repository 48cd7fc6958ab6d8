// Decode batches of Op::MoeFfn (a few to some dozen token rows) whose pairs share experts: the two expert stages over the
// buckets, every weight row read once for up to 8 tokens of its expert, in the arithmetic of the per-token kernels.
//
// Those contract fixed-point activations with the weight codes as three or four byte planes, exact integer sums joined in
// f32 (k_gemv.hip), with 24 or 32 dot instructions per 32 elements and token.  Here the matrix cores take the byte products:
//   * v_mfma_i32_16x16x32_i8: operand A is four tokens x (plane A, B, C, and D or ones) by 32 k, operand B the codes of 16
//     weight rows; a lane receives the plane sums of one token and weight row in its four registers, so the fourth plane of
//     the formats that have one costs no instruction.  Q4_K and Q6_K take three planes as their per-token kernels do, A signed
//     and B, C unsigned, the latter less 128, which the sum of the codes in the fourth register makes good: the same integers,
//     so the same bits; the others balanced digits.
//   * Scales apply per 32 elements (Q6_K: per 16, the codes of the other half masked off), and sums join in the per-token
//     kernels' order: two groups of a lane first (Q6_K: the four 16-groups of a lane), then a binary tree over a block's
//     four lanes and over blocks (a counter of pending partial sums per level).  So a row has the same bits alone, in a small
//     batch and here, wherever the per-token kernels of the format contract the same byte planes: all formats but MXFP4
//     (whose per-token kernel multiplies floats), rows that fit a wavefront.
//   * Weights come as in the grouped GEMM (k_grouped_gemm.hip): 16-byte chunks of consecutive lanes, two steps ahead
//     in registers, through a small LDS region of the wave to a row per lane.  Activations are f32 rows in memory and become
//     planes here, 256 k at a time into alternating LDS buffers: no launch and no buffer for the conversion.
// Bound by the stream of weight rows and, with look-up codes (MXFP4, IQ4_XS), by their unpacking: 16 token rows of 128 experts of
// 2048 x 768 in Q8_0 60 and 32 us (81 distinct experts at 4.5 TB/s; the per-token kernels read 128: 83 and 45); 20 rows of 8
// experts of 4096 x 14336, Q5_K / Q6_K, 179 and 123 us (the unit kernels 1240 and 572).  Tiles of 16 tokens would need more registers than three workgroups per CU leave
// (100 of them spilled) and be bound by the vector instructions.
#include "grouped_fmt.h"
#include "gemv_fmt.h"

namespace infr {

namespace {

constexpr int kIW = 4;   // waves per workgroup
typedef int int4v __attribute__((ext_vector_type(4)));

// Per format, on top of the row layout: the lane's eight codes of a group, in the k order of its bytes (kNibble: elements
// 4 kq .. + 3 and 16 further, else 8 kq .. + 7), and the group scales.
struct PairScale {
    float s0, s1, m0, m1;   // groups 2j, 2j + 1: value = s * code - m
};

// The two groups of a lane as the per-token kernels of one lane per two groups add them up: acc = 0, then acc += scale * sum twice.
__device__ __forceinline__ float two_terms(float s0, float f0, float s1, float f1) { return fmaf(s1, f1, fmaf(s0, f0, 0.0f)); }

struct I4K : G4K {
    static constexpr int kPlanes = 3;
    static constexpr bool kUnsigned = true, kNibble = false, kHalves = false, kSums = true;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        const uint2 q = v.q[g >> 1];
        return g & 1 ? make_uint2((q.x >> 4) & kLo4, (q.y >> 4) & kLo4) : make_uint2(q.x & kLo4, q.y & kLo4);
    }
    static __device__ __forceinline__ PairScale header_scales(const uint4& h, int j) {
        const float d = f16_bits_to_f32(h.x & 0xFFFFu), dmin = f16_bits_to_f32(h.x >> 16);
        const uint32_t sc = j < 2 ? h.y & 0x3F3F3F3Fu : (h.w & kLo4) | ((h.y >> 2) & 0x30303030u);
        const uint32_t mn = j < 2 ? h.z & 0x3F3F3F3Fu : ((h.w >> 4) & kLo4) | ((h.z >> 2) & 0x30303030u);
        const int at = 16 * (j & 1);
        return PairScale{d * (float)((sc >> at) & 0xFFu), d * (float)((sc >> (at + 8)) & 0xFFu),
                         dmin * (float)((mn >> at) & 0xFFu), dmin * (float)((mn >> (at + 8)) & 0xFFu)};
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) { return header_scales(v.h, j); }
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float x0, float x1) {
        return Q4KFmt::two_groups(p.s0, p.s1, p.m0, p.m1, f0, f1, x0, x1);
    }
};

struct I5K : G5K {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false, kNibble = false, kHalves = false, kSums = true;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        const uint2 q = v.q[g >> 1];
        auto five = [&](uint32_t w, uint32_t h) { return ((g & 1 ? w >> 4 : w) & kLo4) | (((h >> g) & kB0) << 4); };
        return make_uint2(five(q.x, v.t.x), five(q.y, v.t.y));
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) { return I4K::header_scales(v.h, j); }
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float x0, float x1) { return I4K::pair(p, f0, f1, x0, x1); }
};

struct I6K : G6K {
    static constexpr int kPlanes = 3;
    static constexpr bool kUnsigned = true, kNibble = false, kHalves = true, kSums = true;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        const int hh = g >> 2, w = g & 3;
        const uint2 l = v.l[2 * hh + (w & 1)], h = v.h[hh];
        auto six = [&](uint32_t q, uint32_t t) {
            return ((w & 2 ? q >> 4 : q) & kLo4) | ((w == 0 ? t << 4 : w == 1 ? t << 2 : w == 2 ? t : t >> 2) & 0x30303030u);
        };
        return make_uint2(six(l.x, h.x), six(l.y, h.y));
    }
    // d * scale of 16-group `odd` of group g
    static __device__ __forceinline__ float scale16(const Raw& v, int g, int odd) {
        const int at = 8 * (g >> 2) + 2 * (g & 3) + odd;
        const uint32_t w = at < 4 ? v.sc.x : at < 8 ? v.sc.y : at < 12 ? v.sc.z : v.sc.w;
        return f16_bits_to_f32(v.d) * (float)(int)(int8_t)((w >> (8 * (at & 3))) & 0xFFu);
    }
};

struct I80 : G80 {
    static constexpr int kPlanes = 3;
    static constexpr bool kUnsigned = false, kNibble = false, kHalves = false, kSums = false;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        if (g & 1) return make_uint2(v.x[g], v.y[g]);
        return make_uint2(__builtin_amdgcn_alignbyte(v.y[g], v.x[g], 2), __builtin_amdgcn_alignbyte(v.z[g >> 1], v.y[g], 2));
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) {
        return PairScale{f16_bits_to_f32(v.d[2 * j]), f16_bits_to_f32(v.d[2 * j + 1]), 0.0f, 0.0f};
    }
    // (a lane per group in the per-token kernel: both products are rounded)
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float, float) { return __fadd_rn(__fmul_rn(p.s0, f0), __fmul_rn(p.s1, f1)); }
};

struct I40 : G40 {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false, kNibble = true, kHalves = false, kSums = false;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        const uint32_t x = g & 1 ? v.x[g] : __builtin_amdgcn_alignbyte(v.y[g >> 1], v.x[g], 2);
        return make_uint2(nibbles_less8(x, false), nibbles_less8(x, true));
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) {
        return PairScale{0.0625f * f16_bits_to_f32(v.d[2 * j]), 0.0625f * f16_bits_to_f32(v.d[2 * j + 1]), 0.0f, 0.0f};
    }
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float, float) { return two_terms(p.s0, f0, p.s1, f1); }
};

struct IMX : GMX {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false, kNibble = true, kHalves = false, kSums = false;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {   // twice the value
        const uint32_t x = (g + 1) & 3 ? __builtin_amdgcn_alignbyte(v.y[g], v.x[g], (g + 1) & 3) : v.x[g];
        return make_uint2(signed_book(x << 4, x, 0x03020100u, 0x0C080604u, 0xFDFEFF00u, 0xF4F8FAFCu),
                          signed_book(x, x >> 4, 0x03020100u, 0x0C080604u, 0xFDFEFF00u, 0xF4F8FAFCu));
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) { return PairScale{e8m0_half(v.e[2 * j]), e8m0_half(v.e[2 * j + 1]), 0.0f, 0.0f}; }
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float x0, float x1) { return I80::pair(p, f0, f1, x0, x1); }
};

struct IIX : GIX {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false, kNibble = true, kHalves = false, kSums = false;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {
        return make_uint2(signed_book(v.x[g] << 4, v.x[g], 0xBFAD9881u, 0xF6EADDCFu, 0x26190D01u, 0x71594535u),
                          signed_book(v.x[g], v.x[g] >> 4, 0xBFAD9881u, 0xF6EADDCFu, 0x26190D01u, 0x71594535u));
    }
    static __device__ __forceinline__ float scale(const Raw& v, int g) {
        const int ls = (int)((v.h.y >> (4 * g)) & 15u) | (int)(((v.h.x >> (16 + 2 * g)) & 3u) << 4);
        return f16_bits_to_f32(v.h.x & 0xFFFFu) * (float)(ls - 32);
    }
    static __device__ __forceinline__ PairScale scales(const Raw& v, int j) { return PairScale{scale(v, 2 * j), scale(v, 2 * j + 1), 0.0f, 0.0f}; }
    static __device__ __forceinline__ float pair(const PairScale& p, float f0, float f1, float, float) { return two_terms(p.s0, f0, p.s1, f1); }
};

// Rows too wide for a wavefront of the per-token kernels are f32 sums when they come alone: four planes here.
struct W4K : I4K {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false;
};
struct W6K : I6K {
    static constexpr int kPlanes = 4;
    static constexpr bool kUnsigned = false, kSums = false;
    static __device__ __forceinline__ uint2 codes(const Raw& v, int g) {   // less 32, four times
        const uint2 c = I6K::codes(v, g);
        return make_uint2((c.x << 2) ^ 0x80808080u, (c.y << 2) ^ 0x80808080u);
    }
    static __device__ __forceinline__ float scale16(const Raw& v, int g, int odd) { return 0.25f * I6K::scale16(v, g, odd); }
};
struct W80 : I80 {
    static constexpr int kPlanes = 4;
};

template <class F>
constexpr int kIStage = 256 * F::kChunks;              // LDS bytes of 16 rows' step
template <class F>
constexpr int kIGroups = F::kHalves ? 16 : 8;          // scale groups of 256 k
constexpr int kIGroup = 544;                           // bytes of 16 plane rows x 32 k (32 more, so that the groups start on different banks)
constexpr int kIPlanes = kIntTok / 4 * 8 * kIGroup;    // planes of the tile's tokens x 256 k
template <class F>
constexpr size_t int_lds() { return (size_t)kIW * kIStage<F> + 2 * kIPlanes + 2 * kIntTok * kIGroups<F> * 8; }

// TQ: groups of four tokens.  A wave owns 16 weight rows (gate/up: waves 0 and 1 gate rows, 2 and 3 the up rows of the same features).
template <class F, bool DOWN, int TQ>
__device__ __forceinline__ void int_tile(const GroupedParams& p, const Tile& t, int n0, uint8_t* lds, const uint64_t* s_tab) {
    constexpr int NC = 16 * F::kChunks, NL = (NC + 63) / 64;
    constexpr bool kPartial = F::kBlock < F::kStep;
    constexpr int SPP = 256 / F::kStep;                                // steps per 256-k piece of the activations
    constexpr int GR = kIGroups<F>, E = 4 * TQ;                        // scale groups and elements a thread converts per piece
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, kq = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* const wl = lds + wave * kIStage<F>;
    uint8_t* const al = lds + kIW * kIStage<F>;                        // [2][TQ][8 groups][16 rows: token, plane][32 bytes]
    float2* const sl = reinterpret_cast<float2*>(al + 2 * kIPlanes);   // [2][4 TQ tokens][GR] scale, sum

    const int tok_x = tid / (256 / E), e_x = tid % (256 / E);          // the thread's token and E elements of a piece
    const float* xrow;
    {
        const int pr = t.p0 + min(tok_x, t.cnt - 1);
        xrow = p.xf + (size_t)(DOWN ? pr : p.pair_row[pr]) * p.K + E * e_x;
    }
    constexpr int kStepBytes = F::kStep / F::kBlock * F::kBlockBytes;
    const uint32_t row_bytes = (uint32_t)(p.K / F::kBlock) * F::kBlockBytes;
    const bool up = !DOWN && wave >= 2;
    const uint8_t* const bank = (up ? p.w1 + (size_t)t.e * p.w1_stride : p.w0 + (size_t)t.e * p.w0_stride);
    const int f_wave = n0 + 16 * (DOWN ? wave : wave & 1);
    uint32_t woff[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {          // rows beyond the matrix's last one repeat it
        const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, c = idx - r * F::kChunks;
        woff[i] = (uint32_t)min(f_wave + r, p.N - 1) * row_bytes + F::src(c, r);
    }
    uint4v w[2][NL];   // the steps under way: even, odd
    // the steps of this part of K (down may be cut into parts, see launch_grouped_int_down)
    const int base = (int)blockIdx.y * p.k_part_steps;
    const int n_steps = min(p.k_part_steps, (p.K + F::kStep - 1) / F::kStep - base);
    auto request = [&](int s, uint4v (&to)[NL]) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const uint8_t* const b = bank + (uint32_t)(kStepBytes * (base + s));
            uint32_t off = woff[i];
            if (kPartial && (base + s + 1) * F::kStep > p.K) {   // chunks behind the row's end are not read (the step's first one instead)
                const int idx = min(64 * i + lane, NC - 1), r = idx / F::kChunks, at = F::src(idx - r * F::kChunks, r);
                if (kStepBytes * (base + s) + at >= (int)row_bytes) off -= (uint32_t)at;
            }
            to[i] = ldu<uint4v>(b + off);
        }
    };
    float xv[E];
    auto x_load = [&](int piece) {
        const int k = F::kStep * base + 256 * piece;
#pragma unroll
        for (int q = 0; q < E; q += 4) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!kPartial || k + E * e_x < p.K) v = *reinterpret_cast<const float4*>(xrow + k + q);
            xv[q] = v.x; xv[q + 1] = v.y; xv[q + 2] = v.z; xv[q + 3] = v.w;
        }
    };
    auto x_store = [&](int buf) {
        const Digits<E, F::kPlanes> d = digits_of<E, F::kHalves ? 16 : 32, !F::kUnsigned, F::kPlanes>(xv);
        const int g = e_x / (32 / E), o = e_x % (32 / E);              // group, place in it
        uint8_t* const row = al + buf * kIPlanes + ((tok_x >> 2) * 8 + g) * kIGroup + 4 * (tok_x & 3) * 32;
#pragma unroll
        for (int i = 0; i < E / 4; i++) {
            const int q = o * (E / 4) + i;                             // four elements
            uint8_t* const at = row + (F::kNibble ? 8 * (q & 3) + 4 * (q >> 2) : 4 * q);
            const uint32_t flip = F::kUnsigned ? 0x80808080u : 0u;
            *reinterpret_cast<uint32_t*>(at) = d.a[i];
            *reinterpret_cast<uint32_t*>(at + 32) = d.b[i] ^ flip;
            *reinterpret_cast<uint32_t*>(at + 64) = d.c[i] ^ flip;
            if constexpr (F::kPlanes == 4) *reinterpret_cast<uint32_t*>(at + 96) = d.d[i];
        }
        constexpr int kPer = (F::kHalves ? 16 : 32) / E;               // threads of a scale group
        if (e_x % kPer == 0) sl[buf * kIntTok * GR + tok_x * GR + e_x / kPer] = make_float2(d.scale, F::kSums ? d.sum : 0.0f);
    };
    const int n_pieces = (n_steps + SPP - 1) / SPP;
    x_load(0);
    request(0, w[0]);
    if (n_steps > 1) request(1, w[1]);
    x_store(0);
    if (n_pieces > 1) x_load(1);
    // with unsigned codes the fourth row of every token: ones (both buffers, once)
    for (int i = F::kUnsigned ? tid : 2 * TQ * 8 * 4 * 8; i < 2 * TQ * 8 * 4 * 8; i += 256) {   // dwords: buffer, token quad and group, token, dword
        const int dw = i & 7, tk = (i >> 3) & 3, tg = (i >> 5) % (TQ * 8), buf = (i >> 5) / (TQ * 8);
        *reinterpret_cast<uint32_t*>(al + buf * kIPlanes + tg * kIGroup + (4 * tk + 3) * 32 + 4 * dw) = kB0;
    }

    float lv[4][TQ], tot[TQ];   // partial sums that wait for their neighbour, per level; sums of 16 steps
#pragma unroll
    for (int m = 0; m < TQ; m++) {
        tot[m] = 0.0f;
#pragma unroll
        for (int l = 0; l < 4; l++) lv[l][m] = 0.0f;
    }
    // join3 of the three plane sums; the lower two in integers first (below 2^28), which rounds as its inner fma does
    auto join = [&](const int4v& y) {
        if constexpr (F::kPlanes == 4) return join4(y[0], y[1], y[2], y[3]);
        int low = y[1] * 256 + y[2];
        if (F::kUnsigned) low += __mul24(y[3], 128 * 256 + 128);
        return fmaf((float)y[0], 65536.0f, (float)low);
    };
    // The arithmetic of a pair of groups is done where it stands: drawn together, or left until a later step needs its result,
    // the operands would not fit the registers (some hundred spilled).
    auto pin = [](float& v) { asm volatile("" : "+v"(v)); };
    // step s, whose weights are in wr; more: step s + 2 exists and is requested into the same registers
    auto step = [&](int s, uint4v (&wr)[NL], auto always) __attribute__((always_inline)) {
        const bool more = decltype(always)::value || s + 2 < n_steps;
        typename F::Raw raw;   // in rows of the wave's LDS region, out as every lane's share of its row (in order: no waiting between)
#pragma unroll
        for (int i = 0; i < NL; i++)
            if (64 * i + 63 < NC || 64 * i + lane < NC) *reinterpret_cast<uint4v*>(wl + 16 * (64 * i + lane)) = wr[i];
        asm volatile("" ::: "memory");
        F::load(wl, col, kq, raw);
        asm volatile("" ::: "memory");
        if (more) request(s + 2, wr);
        asm volatile("" ::: "memory");
        const int piece = s / SPP, buf = piece & 1;
        if (s % SPP == 0) {
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            // the next piece, beside this one's arithmetic: its buffer's last readers are behind the barrier
            if (decltype(always)::value || piece + 1 < n_pieces) x_store(buf ^ 1);
            if (decltype(always)::value) x_load(min(piece + 2, n_pieces - 1));   // (no branch: see the loop)
            else if (piece + 2 < n_pieces) x_load(piece + 2);
        }
        const uint8_t* const ab = al + buf * kIPlanes + (SPP > 1 ? (s % SPP) * (F::kStep / 32) * kIGroup : 0) + col * 32 + kq * 8;
        const float2* const sb = sl + buf * kIntTok * GR + kq * GR + (SPP > 1 ? (s % SPP) * (F::kStep / 32) : 0);
        float blk[TQ], part[TQ];
        if constexpr (F::kHalves) {
#pragma unroll
            for (int hh = 0; hh < 2; hh++) {
                float odd0[TQ], odd1[TQ];
#pragma unroll
                    for (int m = 0; m < TQ; m++) odd0[m] = odd1[m] = 0.0f;
#pragma unroll
                for (int g4 = 0; g4 < 4; g4++) {
                    const int g = 4 * hh + g4;
                    long b[2];
                    float sc[2];
                    const uint2 c = F::codes(raw, g);
                    const uint32_t mask = kq < 2 ? 0xFFFFFFFFu : 0u;
                    b[0] = __builtin_bit_cast(long, make_uint2(c.x & mask, c.y & mask));
                    b[1] = __builtin_bit_cast(long, make_uint2(c.x & ~mask, c.y & ~mask));
                    sc[0] = F::scale16(raw, g, 0);
                    sc[1] = F::scale16(raw, g, 1);
#pragma unroll
                    for (int m = 0; m < TQ; m++) {
                        const long a = *reinterpret_cast<const long*>(ab + (m * 8 + g) * kIGroup);
                        const float4 ks = *reinterpret_cast<const float4*>(sb + 4 * m * GR + 2 * g);
                        const float f0 = join(__builtin_amdgcn_mfma_i32_16x16x32_i8(a, b[0], int4v{0, 0, 0, 0}, 0, 0, 0)) * ks.x;
                        const float f1 = join(__builtin_amdgcn_mfma_i32_16x16x32_i8(a, b[1], int4v{0, 0, 0, 0}, 0, 0, 0)) * ks.z;
                        odd0[m] += sc[0] * (F::kSums ? f0 - 32.0f * ks.y : f0);
                        odd1[m] += sc[1] * (F::kSums ? f1 - 32.0f * ks.w : f1);
                        pin(odd0[m]);
                        pin(odd1[m]);
                    }
                }
#pragma unroll
                for (int m = 0; m < TQ; m++) {
                    const float v = odd0[m] + odd1[m];
                    blk[m] = hh ? blk[m] + v : v;
                }
            }
        } else {
            const int groups = kPartial ? (p.K - (base + s) * F::kStep) / 32 : F::kStep / 32;   // groups from here to the row's end
#pragma unroll
            for (int j = 0; j < F::kStep / 64; j++) {
                if (kPartial && 2 * j >= groups) break;
                long b[2];
                PairScale ps;
                ps = F::scales(raw, j);
                if (kPartial && 2 * j + 1 >= groups) ps.s1 = -0.0f;   // its sum is +0: adds -0.0, the identity
                b[0] = __builtin_bit_cast(long, F::codes(raw, 2 * j));
                b[1] = __builtin_bit_cast(long, F::codes(raw, 2 * j + 1));
#pragma unroll
                for (int m = 0; m < TQ; m++) {
                    const long a0 = *reinterpret_cast<const long*>(ab + (m * 8 + 2 * j) * kIGroup), a1 = *reinterpret_cast<const long*>(ab + (m * 8 + 2 * j + 1) * kIGroup);
                    const float4 ks = *reinterpret_cast<const float4*>(sb + 4 * m * GR + 2 * j);
                    const float f0 = join(__builtin_amdgcn_mfma_i32_16x16x32_i8(a0, b[0], int4v{0, 0, 0, 0}, 0, 0, 0)) * ks.x;
                    const float f1 = join(__builtin_amdgcn_mfma_i32_16x16x32_i8(a1, b[1], int4v{0, 0, 0, 0}, 0, 0, 0)) * ks.z;
                    const float v = F::pair(ps, f0, f1, ks.y, ks.w);
                    // ((0 + 1) + (2 + 3)): an even pair waits, an odd one joins it
                    if (j & 1) {
                        const float u = part[m] + v;
                        blk[m] = j == 3 ? blk[m] + u : u;
                        pin(blk[m]);
                    } else {
                        part[m] = v;
                        pin(part[m]);
                    }
                }
                if (kPartial && !(j & 1) && 2 * j + 2 >= groups) {   // no odd pair follows
#pragma unroll
                        for (int m = 0; m < TQ; m++) blk[m] = j == 2 ? blk[m] + part[m] : part[m];
                }
            }
        }
        // the step's sums into the counter of partial sums: level l waits while bit l of s is clear
        auto carry = [&](float (&wait)[TQ], bool join_it) {
#pragma unroll
                for (int m = 0; m < TQ; m++) {
                    if (join_it) blk[m] = wait[m] + blk[m];
                    else wait[m] = blk[m];
                }
        };
        carry(lv[0], s & 1);
        if (s & 1) {
            carry(lv[1], s & 2);
            if (s & 2) {
                carry(lv[2], s & 4);
                if (s & 4) {
                    carry(lv[3], s & 8);
                    if (s & 8) {
#pragma unroll
                            for (int m = 0; m < TQ; m++) tot[m] = s == 15 ? blk[m] : tot[m] + blk[m];
                    }
                }
            }
        }
    };
    int s0 = 0;
    for (; s0 + 4 <= n_steps; s0 += 2) {   // no branch around the requests: the waits count exactly the younger ones
        step(s0, w[0], std::true_type{});
        step(s0 + 1, w[1], std::true_type{});
    }
    for (; s0 < n_steps; s0 += 2) {
        step(s0, w[0], std::false_type{});
        if (s0 + 1 < n_steps) step(s0 + 1, w[1], std::false_type{});
    }
    // what still waits, small levels first
    float sum[TQ];
#pragma unroll
        for (int m = 0; m < TQ; m++) {
            float v = -0.0f;   // x + -0.0 is x
#pragma unroll
            for (int l = 0; l < 4; l++)
                if (n_steps & (1 << l)) v = lv[l][m] + v;
            sum[m] = n_steps >= 16 ? tot[m] + v : v;
        }
    const int f = f_wave + col;
    if constexpr (!DOWN) {   // the up rows' sums to the waves of the gate rows
        float* const xch = reinterpret_cast<float*>(lds + (wave & 1) * kIStage<F>);   // (the gate waves' own region, read for the last time)
        if (up) {
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int m = 0; m < TQ; m++) xch[64 * m + lane] = sum[m];
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            return;
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int m = 0; m < TQ; m++) {
            const int tok = 4 * m + kq, pr = t.p0 + tok;
            float gs = sum[m], us = xch[64 * m + lane];
            if (tok >= t.cnt || f >= p.N) continue;
            if (p.weight_before) {
                const float wp = p.route_w[p.pair_src[pr]];
                gs = __fmul_rn(wp, gs);
                us = __fmul_rn(wp, us);
            }
            p.out[(size_t)pr * p.N + f] = gated_act_fn(p.act, p.has_clamp, p.clamp, gs, us, s_tab);
        }
    } else {
#pragma unroll
        for (int m = 0; m < TQ; m++) {
            const int tok = 4 * m + kq;
            if (tok < t.cnt && f < p.N)
                p.out[((size_t)blockIdx.y * p.n_pairs + t.p0 + tok) * p.N + f] = p.down_scale ? __fmul_rn(sum[m], p.down_scale[t.e]) : sum[m];
        }
    }
}

template <class F, bool DOWN>
__global__ __launch_bounds__(kIW * 64, 3) void grouped_int(GroupedParams p) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_int[];
    __shared__ uint64_t s_tab[32];
    Tile t;
    int n0;
    if (!tile_item(p.tiles, p.n_tiles_n, p.n_tiles_rcp, kIntTok, t, n0)) return;
    n0 *= (DOWN ? 16 : 8) * kIW;
    if (!DOWN && threadIdx.x < 32) s_tab[threadIdx.x] = kExp2Table[threadIdx.x];   // read behind barriers
    if (t.cnt <= 4) int_tile<F, DOWN, 1>(p, t, n0, lds_int, s_tab);
    else int_tile<F, DOWN, 2>(p, t, n0, lds_int, s_tab);
}

// Steps of a part when K is asked for in `parts`: whole pieces of 256 k.
int part_steps(int steps, int parts) { return parts < 2 ? steps : ((steps + parts - 1) / parts + 1) & ~1; }

template <class F, bool DOWN>
void int_gemm(hipStream_t s, const GroupedParams& p) {
    const int width = (DOWN ? 16 : 8) * kIW;
    GroupedParams q = p;
    q.n_tiles_n = (p.N + width - 1) / width;
    q.n_tiles_rcp = (uint32_t)((0x100000000ull + q.n_tiles_n - 1) / q.n_tiles_n);
    const int steps = (p.K + F::kStep - 1) / F::kStep;
    q.k_part_steps = DOWN ? part_steps(steps, p.k_parts) : steps;
    const dim3 grid((unsigned)((gemm_max_tiles(p.n_pairs, p.n_expert, kIntTok) * q.n_tiles_n + 7) & ~7), (steps + q.k_part_steps - 1) / q.k_part_steps);
    INFR_LDS_LIMIT((grouped_int<F, DOWN>), (int)int_lds<F>());
    INFR_LAUNCH((grouped_int<F, DOWN>), grid, dim3(kIW * 64), int_lds<F>(), s, q);
}

template <bool DOWN>
void int_any(hipStream_t s, int dt, const GroupedParams& p) {
    auto go = [&](auto f) { int_gemm<decltype(f), DOWN>(s, p); };
    switch (dt) {
        case INFR_Q4K: p.K > 4096 ? go(W4K{}) : go(I4K{}); break;
        case INFR_Q5K: go(I5K{}); break;
        case INFR_Q6K: p.K > 4096 ? go(W6K{}) : go(I6K{}); break;
        case INFR_Q8_0: p.K > 2048 ? go(W80{}) : go(I80{}); break;
        case INFR_Q4_0: go(I40{}); break;
        case INFR_MXFP4: go(IMX{}); break;
        case INFR_IQ4_XS: go(IIX{}); break;
        default: break;
    }
}

}  // namespace

bool grouped_int_supported(int dt, int k) {
    switch (dt) {
        case INFR_Q4K: case INFR_Q5K: case INFR_Q6K: case INFR_IQ4_XS: return k > 0 && k % 256 == 0;
        case INFR_Q8_0: case INFR_Q4_0: case INFR_MXFP4: return k > 0 && k % 32 == 0;
        default: return false;
    }
}

// Rows of many blocks on few columns leave most compute units without a workgroup: the down rows then go in parts of K, whose
// sums the combine adds.  Rows of up to sixteen 256-k steps stay whole: their sums have the per-token kernels' order.  Longer
// ones are cut by their length alone, so that a row's bits do not depend on how many others are in the batch (8 experts of
// 4096 x 14336, Q6_K, four parts: 5 rows 72 us, 31 rows 158; in the one or two parts that the batch alone would ask for 88 and 172).
int grouped_int_down_parts(int k) { return (k + 4095) / 4096; }
int grouped_int_parts(int dt, int k, int k_parts) {
    const int step = dt == INFR_Q8_0 ? 128 : 256, steps = (k + step - 1) / step, per = part_steps(steps, k_parts);
    return (steps + per - 1) / per;
}

void launch_grouped_int_gate_up(hipStream_t s, int dt, const GroupedParams& p) { int_any<false>(s, dt, p); }
void launch_grouped_int_down(hipStream_t s, int dt, const GroupedParams& p) { int_any<true>(s, dt, p); }

}  // namespace infr
