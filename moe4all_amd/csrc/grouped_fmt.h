// How the rows of the block formats travel from memory to the lanes of a wave in the kernels that contract 16-row operands
// (k_grouped_gemm.hip, k_grouped_int.hip), and the formats as f16 operands.
#pragma once

#include "grouped_common.h"
#include "units.h"

namespace infr {

namespace {

typedef float float4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));   // (arrays of HIP's uint4 written under a condition end up in scratch memory)

constexpr float kTwo24 = 16777216.0f;       // undoes the 2^-24 of subnormal codes


__device__ __forceinline__ half8 pack8(half2v a, half2v b, half2v c, half2v d) {
    return __builtin_bit_cast(half8, make_uint4(as_u32(a), as_u32(b), as_u32(c), as_u32(d)));
}

// Weight formats.
//   kStep k elements of a row are one step: kChunks 16-byte chunks per row; chunk c of row r (of 16) of step s comes from
//   byte kStepBytes s + src(c, r) of the row and lies at 16 (kChunks r + c) in LDS, where sixteen rows reading the same
//   place of a row hit distinct banks (at most two for the same).  A row may end inside a step (K a multiple of 64); a
//   chunk that starts inside the row may run up to 15 bytes past it, which every buffer of the backend has room for.
//   Raw: the lane's share of its row for the step (a quarter of every group of 32 k), in registers; St: what is derived
//   from it once per step; frag(g) = the lane's eight k of group g of the step, in the order of activation chunk
//   a_lane(kq) | a_group(g) (four groups cover 16 chunks, disjoint bits).
//   kScale: the sums are kept in units of the block's d; kMin: the format has minimums (St::mins: those of eight groups).
struct G4K {
    static constexpr int kStep = 256, kChunks = 9;
    static constexpr bool kScale = true, kMin = true, kUnits = false;
    static constexpr int kBlock = 256, kBlockBytes = 144;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return 4 * (kq >> 1) + (kq & 1); }
    static constexpr __device__ int a_group(int g) { return 8 * (g >> 1) | 2 * (g & 1); }
    struct Raw {
        uint4 h;
        uint2 q[4];
    };
    struct St {
        uint32_t s[2];     // integer scales of groups 0..3, 4..7
        half8 mins;
        float d, dmin;
    };
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 144 * r;
        v.h = *reinterpret_cast<const uint4*>(row);
#pragma unroll
        for (int j = 0; j < 4; j++) v.q[j] = *reinterpret_cast<const uint2*>(row + 16 + 32 * j + 8 * kq);
    }
    static __device__ __forceinline__ St prep(const Raw& v, int kq) { return prep_header(v.h, kq); }
    static __device__ __forceinline__ St prep_header(const uint4& h, int kq) {
        St t;
        t.d = f16_bits_to_f32(h.x & 0xFFFFu);
        t.dmin = f16_bits_to_f32(h.x >> 16);
        // get_scale_min_k4 (crates/infr-gguf/src/dequant.rs:77-87), four scales or minimums per dword
        t.s[0] = h.y & 0x3F3F3F3Fu;
        t.s[1] = (h.w & 0x0F0F0F0Fu) | ((h.y >> 2) & 0x30303030u);
        if (t.d == 0.0f) t.s[0] = t.s[1] = 0;   // the sums keep the unit of the block before
        const uint32_t ml = h.z & 0x3F3F3F3Fu, mh = ((h.w >> 4) & 0x0F0F0F0Fu) | ((h.z >> 2) & 0x30303030u);
        // k slots 0..7 meet the high halves of the sums, 8..15 their low halves, the rest is zero
        uint32_t m[4] = {__builtin_amdgcn_perm(0x64u, ml, 0x04010400u), __builtin_amdgcn_perm(0x64u, ml, 0x04030402u),
                         __builtin_amdgcn_perm(0x64u, mh, 0x04010400u), __builtin_amdgcn_perm(0x64u, mh, 0x04030402u)};
#pragma unroll
        for (int i = 0; i < 4; i++) m[i] = kq < 2 ? m[i] : 0x64006400u;
        t.mins = pack8(unbias(m[0], 1024.f), unbias(m[1], 1024.f), unbias(m[2], 1024.f), unbias(m[3], 1024.f));
        return t;
    }
    // odd groups sit in the high nibbles, code * 16: their scale is a sixteenth
    static __device__ __forceinline__ half2v scale(const St& t, int g) {
        const uint32_t sc = __builtin_amdgcn_perm(0x64u, t.s[g >> 2], 0x04000400u + 0x00010001u * (g & 3));
        return g & 1 ? __builtin_elementwise_fma(as_h2(sc), splat(0.0625f), splat(-64.0f)) : as_h2(sc) - splat(1024.0f);
    }
    static __device__ __forceinline__ half8 frag(const Raw& r, const St& t, int g) {
        const uint2 v = r.q[g >> 1];
        const half2v f = scale(t, g);
        const uint32_t mask = g & 1 ? 0x00F000F0u : 0x000F000Fu;
        return pack8(as_h2(v.x & mask) * f, as_h2((v.x >> 8) & mask) * f, as_h2(v.y & mask) * f, as_h2((v.y >> 8) & mask) * f);
    }
};

// Bytes 0..207 of a block as thirteen chunks, bytes 194..209 (d in the last two) as the fourteenth.  (A step of half a block
// would fetch 64 + 32 + 2 x 16 bytes from four places of it: 9 cache lines per row and block instead of 2.6, and the load
// path, not the memory, would set the pace: a launch that only reads 165 MB that way takes 41 us, this way 32.)
struct G6K {
    static constexpr int kStep = 256, kChunks = 14;
    static constexpr bool kScale = true, kMin = false, kUnits = false;
    static constexpr int kBlock = 256, kBlockBytes = 210;
    // rows 8..15 hold chunk c at c ^ 1 (rows of 224 bytes: r and r + 8 start on the same bank)
    static __device__ __forceinline__ int src(int c, int r) { c ^= r >> 3; return c < 13 ? 16 * c : 194; }
    static __device__ __forceinline__ int a_lane(int kq) { return 4 * (kq >> 1) + (kq & 1); }
    static constexpr __device__ int a_group(int g) { return 8 * (g >> 1) | 2 * (g & 1); }
    struct Raw {
        uint2 l[4], h[2];
        uint4 sc;
        uint32_t d;
    };
    struct St {
        float d;
        int sh;
    };
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const int x = r >> 3;
        const uint8_t* const row = w + 224 * r;
        const uint8_t* const q = row + 16 * ((kq >> 1) ^ x) + 8 * (kq & 1);
#pragma unroll
        for (int j = 0; j < 4; j++) v.l[j] = *reinterpret_cast<const uint2*>(q + 32 * j);
#pragma unroll
        for (int j = 0; j < 2; j++) v.h[j] = *reinterpret_cast<const uint2*>(q + 128 + 32 * j);
        v.sc = *reinterpret_cast<const uint4*>(row + 192 + 16 * x);
        v.d = *reinterpret_cast<const uint16_t*>(row + 222 - 16 * x);
    }
    static __device__ __forceinline__ St prep(const Raw& v, int kq) { return St{f16_bits_to_f32(v.d), 8 * (kq >> 1)}; }
    // virtual 64-k chunk g / 2 = 2 half + ab: group 2 ab the low codes of ql bytes 64 half + 32 ab .., group 2 ab + 1 their
    // high codes (64 elements further)
    static __device__ __forceinline__ half8 frag(const Raw& v, const St& t, int g) {
        const int hh = g >> 2, ab = (g >> 1) & 1, high = g & 1;
        const uint32_t sw = hh ? (high ? v.sc.w : v.sc.z) : (high ? v.sc.y : v.sc.x);   // scales 8 hh + 4 high + 2 ab + kq / 2
        const float sc = (float)(int8_t)((sw >> (16 * ab)) >> t.sh);
        const half2v f = splat(t.d == 0.0f ? 0.0f : sc);   // (d = 0: the sums keep the unit of the block before)
        const half2v bias = as_h2(0x80208020u);   // -32 * 2^-24
        const int up = high ? -2 * ab : 4 - 2 * ab;   // the codes' two top bits to bits 4, 5
        auto top = [&](uint32_t h) { return up >= 0 ? h << up : h >> -up; };
        auto two = [&](uint32_t q, uint32_t h) { return (as_h2((q & 0x000F000Fu) | (h & 0x00300030u)) + bias) * f; };
        const uint2 l = v.l[g >> 1], h = v.h[hh];
        const uint32_t q0 = high ? l.x >> 4 : l.x, q1 = high ? l.y >> 4 : l.y, h0 = top(h.x), h1 = top(h.y);
        return pack8(two(q0, h0), two(q0 >> 8, h0 >> 8), two(q1, h1), two(q1 >> 8, h1 >> 8));
    }
};

// Four blocks per step.
struct G80 {
    static constexpr int kStep = 128, kChunks = 9;
    static constexpr bool kScale = false, kMin = false, kUnits = false;
    static constexpr int kBlock = 32, kBlockBytes = 34;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return kq; }
    static constexpr __device__ int a_group(int g) { return 4 * g; }
    struct Raw {
        uint32_t x[4], y[4], z[2], d[4];   // block g: eight codes at byte 34 g + 2 + 8 kq; even blocks start two bytes off a dword
    };
    struct St {};
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 144 * r;
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const uint8_t* q = row + 34 * g + 2 + 8 * kq;
            if (!(g & 1)) {
                q -= 2;
                v.z[g >> 1] = *reinterpret_cast<const uint32_t*>(q + 8);
            }
            v.x[g] = *reinterpret_cast<const uint32_t*>(q);
            v.y[g] = *reinterpret_cast<const uint32_t*>(q + 4);
            v.d[g] = *reinterpret_cast<const uint16_t*>(row + 34 * g);
        }
    }
    static __device__ __forceinline__ St prep(const Raw&, int) { return St{}; }
    // f16(d * code): rounded once
    static __device__ __forceinline__ half8 frag(const Raw& v, const St&, int g) {
        uint32_t x = v.x[g], y = v.y[g];
        if (!(g & 1)) {
            x = __builtin_amdgcn_alignbyte(y, x, 2);
            y = __builtin_amdgcn_alignbyte(v.z[g >> 1], y, 2);
        }
        x ^= 0x80808080u;
        y ^= 0x80808080u;
        const half2v d = as_h2(__builtin_amdgcn_perm(v.d[g], v.d[g], 0x01000100u));
        const uint32_t a = __builtin_amdgcn_perm(0x64u, x, 0x04010400u), b = __builtin_amdgcn_perm(0x64u, x, 0x04030402u);
        const uint32_t c = __builtin_amdgcn_perm(0x64u, y, 0x04010400u), e = __builtin_amdgcn_perm(0x64u, y, 0x04030402u);
        return pack8(unbias(a, 1152.f) * d, unbias(b, 1152.f) * d, unbias(c, 1152.f) * d, unbias(e, 1152.f) * d);
    }
};

// (Before they had operands of their own the formats from here on went through the 32-element unit decoder on tiles of 128
// tokens: 333 token rows of 128 experts of 2048 x 768, gate/up in Q5_K 113 us, 64 here.)
// Q5_K as Q4_K with a fifth code bit per element (bit g of byte l of the 32 high-bit bytes): scale * code <= 63 * 31 fits a half.
struct G5K {
    static constexpr int kStep = 256, kChunks = 11;
    static constexpr bool kScale = true, kMin = true, kUnits = false;
    static constexpr int kBlock = 256, kBlockBytes = 176;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return G4K::a_lane(kq); }
    static constexpr __device__ int a_group(int g) { return G4K::a_group(g); }
    struct Raw {
        uint4 h;
        uint2 t, q[4];
    };
    typedef G4K::St St;
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 176 * r;
        v.h = *reinterpret_cast<const uint4*>(row);
        v.t = *reinterpret_cast<const uint2*>(row + 16 + 8 * kq);
#pragma unroll
        for (int j = 0; j < 4; j++) v.q[j] = *reinterpret_cast<const uint2*>(row + 48 + 32 * j + 8 * kq);
    }
    static __device__ __forceinline__ St prep(const Raw& v, int kq) { return G4K::prep_header(v.h, kq); }
    static __device__ __forceinline__ half8 frag(const Raw& r, const St& t, int g) {
        const uint2 v = r.q[g >> 1];
        const half2v f = G4K::scale(t, g);
        // even groups: code in bits 0..4; odd groups: code * 16 in bits 4..8
        const int at = g & 1 ? 8 : 4;
        const uint32_t mask = g & 1 ? 0x00F000F0u : 0x000F000Fu, top = 0x00010001u << at;
        auto bit = [&](uint32_t h) { return at >= g ? h << (at - g) : h >> (g - at); };
        auto two = [&](uint32_t q, uint32_t h) { return as_h2((q & mask) | (bit(h) & top)) * f; };
        return pack8(two(v.x, r.t.x), two(v.x >> 8, r.t.x >> 8), two(v.y, r.t.y), two(v.y >> 8, r.t.y >> 8));
    }
};

// Q4_0: a lane's dword of a block's 16 code bytes holds elements 4 kq .. + 3 (low nibbles) and 16 further (high nibbles).
struct G40 {
    static constexpr int kStep = 256, kChunks = 9;
    static constexpr bool kScale = false, kMin = false, kUnits = false;
    static constexpr int kBlock = 32, kBlockBytes = 18;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return kq; }
    static constexpr __device__ int a_group(int g) { return 4 * g; }
    struct Raw {
        uint32_t x[8], y[4], d[8];   // even blocks start two bytes off a dword
    };
    struct St {};
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 144 * r;
#pragma unroll
        for (int g = 0; g < 8; g++) {
            const uint8_t* q = row + 18 * g + 2 + 4 * kq;
            if (!(g & 1)) {
                q -= 2;
                v.y[g >> 1] = *reinterpret_cast<const uint32_t*>(q + 4);
            }
            v.x[g] = *reinterpret_cast<const uint32_t*>(q);
            v.d[g] = *reinterpret_cast<const uint16_t*>(row + 18 * g);
        }
    }
    static __device__ __forceinline__ St prep(const Raw&, int) { return St{}; }
    // f16(d * (code - 8)): rounded once
    static __device__ __forceinline__ half8 frag(const Raw& v, const St&, int g) {
        const uint32_t x = g & 1 ? v.x[g] : __builtin_amdgcn_alignbyte(v.y[g >> 1], v.x[g], 2);
        const half2v d = as_h2(__builtin_amdgcn_perm(v.d[g], v.d[g], 0x01000100u));
        auto two = [&](uint32_t q) { return unbias((q & 0x000F000Fu) | 0x64006400u, 1032.f) * d; };
        return pack8(two(x), two(x >> 8), two(x >> 4), two(x >> 12));
    }
};

// MXFP4: the conversion instruction takes a byte of two codes and the block's exponent to two halves; a byte holds elements
// l and l + 16.
struct GMX {
    static constexpr int kStep = 256, kChunks = 9;
    static constexpr bool kScale = false, kMin = false, kUnits = false;
    static constexpr int kBlock = 32, kBlockBytes = 17;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return kq; }
    static constexpr __device__ int a_group(int g) { return 4 * g; }
    struct Raw {
        uint32_t x[8], y[8], e[8];
    };
    struct St {};
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 144 * r;
#pragma unroll
        for (int g = 0; g < 8; g++) {   // codes at 17 g + 1 + 4 kq: (g + 1) % 4 bytes behind a dword
            const uint8_t* const q = row + 17 * g + 1 - ((g + 1) & 3) + 4 * kq;
            v.x[g] = *reinterpret_cast<const uint32_t*>(q);
            if ((g + 1) & 3) v.y[g] = *reinterpret_cast<const uint32_t*>(q + 4);
            v.e[g] = row[17 * g];
        }
    }
    static __device__ __forceinline__ St prep(const Raw&, int) { return St{}; }
    static __device__ __forceinline__ half8 frag(const Raw& v, const St&, int g) {
        const uint32_t x = (g + 1) & 3 ? __builtin_amdgcn_alignbyte(v.y[g], v.x[g], (g + 1) & 3) : v.x[g];
        const float e = __uint_as_float(min(v.e[g], 254u) << 23);   // (255 decodes as 2^127 here, a NaN to the instruction)
        return pack8(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(x, e, 0), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(x, e, 1),
                     __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(x, e, 2), __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(x, e, 3));
    }
};

// IQ4_XS: elements as Q4_0's, sixteen bytes per sub-block; book value (-127 .. 113) times the sub-block's signed 6-bit scale,
// products beyond 2048 rounded once.
struct GIX {
    static constexpr int kStep = 256, kChunks = 9;
    static constexpr bool kScale = true, kMin = false, kUnits = false;
    static constexpr int kBlock = 256, kBlockBytes = 136;
    static __device__ __forceinline__ int src(int c, int) { return 16 * c; }
    static __device__ __forceinline__ int a_lane(int kq) { return kq; }
    static constexpr __device__ int a_group(int g) { return 4 * g; }
    struct Raw {
        uint2 h;
        uint32_t x[8];
    };
    struct St {
        float d;
    };
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 144 * r;
        v.h = *reinterpret_cast<const uint2*>(row);
#pragma unroll
        for (int g = 0; g < 8; g++) v.x[g] = *reinterpret_cast<const uint32_t*>(row + 8 + 16 * g + 4 * kq);
    }
    static __device__ __forceinline__ St prep(const Raw& v, int) { return St{f16_bits_to_f32(v.h.x & 0xFFFFu)}; }
    static __device__ __forceinline__ half8 frag(const Raw& v, const St& t, int g) {
        const int ls = (int)((v.h.y >> (4 * g)) & 15u) | (int)(((v.h.x >> (16 + 2 * g)) & 3u) << 4);
        const half2v f = splat(t.d == 0.0f ? 0.0f : (float)(ls - 32));   // (d = 0: the sums keep the unit of the block before)
        const uint32_t lo = iq4nl4(v.x[g] & kLo4), hi = iq4nl4((v.x[g] >> 4) & kLo4);   // book + 127
        const half2v bias = as_h2(0x807F807Fu);   // -127 * 2^-24
        auto two = [&](uint32_t c, uint32_t sel) { return (as_h2(__builtin_amdgcn_perm(0u, c, sel)) + bias) * f; };
        return pack8(two(lo, 0x0C010C00u), two(lo, 0x0C030C02u), two(hi, 0x0C010C00u), two(hi, 0x0C030C02u));
    }
};

// Every other block format through the 32-element unit decoder (units.h): a lane decodes whole units, 4 i + kq of a step, and
// rounds scale * code + min once; group 4 i + m contracts elements 8 m .. 8 m + 7 of the four lanes' units.  The decoding
// bounds it: 333 token rows of 128 experts of 2048 x 768 in Q2_K 73 and 42 us, IQ3_S 125 and 66 (the kernel that decoded from
// rows fetched a lane per row, for 128 tokens: 121 and 71, 215 and 118).
template <int DT>
struct GU {
    static constexpr int kBlock = unit_geometry(DT).elems, kBlockBytes = unit_geometry(DT).bytes;
    static constexpr int kStep = 256, kChunks = ((256 / kBlock * kBlockBytes + 15) / 16) | 1;
    static constexpr bool kScale = false, kMin = false, kUnits = true;
    static __device__ __forceinline__ int src(int c, int) { return 16 * min(c, (256 / kBlock * kBlockBytes - 1) / 16); }
    static __device__ __forceinline__ int a_lane(int kq) { return 4 * kq; }
    static constexpr __device__ int a_group(int g) { return 16 * (g >> 2) | (g & 3); }
    struct Raw {
        Unit u[2];
    };
    struct St {};
    static __device__ __forceinline__ void load(const uint8_t* w, int r, int kq, Raw& v) {
        const uint8_t* const row = w + 16 * kChunks * r;
#pragma unroll
        for (int i = 0; i < 2; i++) load_unit<DT>(row, 4 * i + kq, v.u[i]);
    }
    // the units of a row's last, partial step beyond its end count for nothing
    static __device__ __forceinline__ void cut(Raw& v, int kq, int units) {
#pragma unroll
        for (int i = 0; i < 2; i++)
            if (4 * i + kq >= units) {
#pragma unroll
                for (int h = 0; h < 2; h++) v.u[i].sc[h] = v.u[i].mn[h] = 0.0f;
            }
    }
    static __device__ __forceinline__ St prep(const Raw&, int) { return St{}; }
    static __device__ __forceinline__ half8 frag(const Raw& v, const St&, int g) {
        const Unit& u = v.u[g >> 2];
        const int m = g & 3;
        const float sc = u.sc[m >> 1], mn = u.mn[m >> 1];
        const uint32_t a = u.q[2 * m], b = u.q[2 * m + 1];
        half8 h;
        h[0] = (_Float16)fmaf(sc, (float)(a & 0xFFu), mn);
        h[1] = (_Float16)fmaf(sc, (float)((a >> 8) & 0xFFu), mn);
        h[2] = (_Float16)fmaf(sc, (float)((a >> 16) & 0xFFu), mn);
        h[3] = (_Float16)fmaf(sc, (float)(a >> 24), mn);
        h[4] = (_Float16)fmaf(sc, (float)(b & 0xFFu), mn);
        h[5] = (_Float16)fmaf(sc, (float)((b >> 8) & 0xFFu), mn);
        h[6] = (_Float16)fmaf(sc, (float)((b >> 16) & 0xFFu), mn);
        h[7] = (_Float16)fmaf(sc, (float)(b >> 24), mn);
        return h;
    }
};

}  // namespace

}  // namespace infr
