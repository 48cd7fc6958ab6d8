// Shared by the kernels of Op::MoeFfn's batched path (k_grouped.hip: bucketing, conversion, combine; k_grouped_gemm.hip: the
// GEMMs on block formats; k_grouped_float.hip: float weights): k orders of the f16
// activations, the kernels' work item look-ups, the float kernel's tile epilogue.
#pragma once

#include <type_traits>

#include "device_common.h"
#include "kernels.h"

namespace infr {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float16v __attribute__((ext_vector_type(16)));

namespace {

constexpr int kBM = 128;        // token rows per tile
constexpr int kSlice = 64;      // k elements per LDS stage

// Rotation of the eight 16-byte chunks of row t in an LDS tile whose rows are 128 bytes.  The LDS has 64 banks of 4
// bytes and serves a 16-byte read of a wavefront 16 lanes at a time: rows t and t + 1 start half the banks apart, so 16
// consecutive rows reading the same chunk hit 64 distinct banks when rows 2 u and 2 u + 1 share a rotation (measured:
// 205 B/clk per CU against 139 with a rotation by t & 7, 43 without any).
__device__ __forceinline__ int rot7(int t) { return (t >> 1) & 7; }

__device__ __forceinline__ half2v as_h2(uint32_t v) { return __builtin_bit_cast(half2v, v); }
__device__ __forceinline__ uint32_t as_u32(half2v v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ half2v splat(float v) {
    _Float16 h = (_Float16)v;
    return half2v{h, h};
}
// (1024 + code pair) -> code pair - bias, exact
__device__ __forceinline__ half2v unbias(uint32_t magic_pair, float bias) { return as_h2(magic_pair) - splat(bias); }

// --------------------------------------------------------------------------------------------
// K orders of the f16 activation rows, so that the order in which codes fall out of a weight block's dwords is the order in
// which a row lies: virtual chunk c (8 halves) is made of the elements lo .. lo + 3 (a) and hi .. hi + 3 (b), mixed as
// kPlain: a0 a1 a2 a3 b0 b1 b2 b3; kSwapped: a0 a2 a1 a3 b0 b2 b1 b3 (nibbles under a half-word mask);
// kPairs: a0 b0 a1 b1 a2 b2 a3 b3 (both nibbles of a byte).
// kHasMin: the weight format has minimums and a float scale per 256 k, so the sums over groups of 32 are wanted too.
enum KMix { kPlain, kSwapped, kPairs };
struct Order4K {   // Q4_K, Q5_K.  64-k slice of a super-block: 32 bytes, low nibbles = its first 32 elements; chunk 4 h + 2 b + i = bytes 16 h + 8 i ..
    static constexpr bool kHasMin = true;
    static constexpr KMix kMix = kSwapped;
    static __device__ __forceinline__ int lo(int c) { return (c >> 3) * 64 + 32 * ((c >> 1) & 1) + 16 * ((c >> 2) & 1) + 8 * (c & 1); }
    static __device__ __forceinline__ int hi(int c) { return lo(c) + 4; }
};
struct Order6K {   // virtual slice t = 2 half + ab of a block = ql bytes 32 t ..: low nibbles elements 128 half + 32 ab .., high nibbles 64 further
    static constexpr bool kHasMin = false;
    static constexpr KMix kMix = kSwapped;
    static __device__ __forceinline__ int lo(int c) {
        const int t = (c >> 3) & 3;
        return (c >> 5) * 256 + 128 * (t >> 1) + 32 * (t & 1) + 64 * ((c >> 1) & 1) + 16 * ((c >> 2) & 1) + 8 * (c & 1);
    }
    static __device__ __forceinline__ int hi(int c) { return lo(c) + 4; }
};
template <KMix MIX>
struct OrderNibbles {   // 32-element blocks whose byte l holds elements l and 16 + l: chunk c & 3 = bytes 4 (c & 3) ..
    static constexpr bool kHasMin = false;
    static constexpr KMix kMix = MIX;
    static __device__ __forceinline__ int lo(int c) { return 32 * (c >> 2) + 4 * (c & 3); }
    static __device__ __forceinline__ int hi(int c) { return lo(c) + 16; }
};
struct OrderPlain {
    static constexpr bool kHasMin = false;
    static constexpr KMix kMix = kPlain;
    static __device__ __forceinline__ int lo(int c) { return 8 * c; }
    static __device__ __forceinline__ int hi(int c) { return 8 * c + 4; }
};

// Activation for the matrix-core path: hardware exp (about 1e-6 relative), since operands were
// already rounded to f16.  Same formulas as act_fn / gated_act_fn (crates/infr-cpu/src/kernels.rs:6664-6683).
__device__ __forceinline__ float act_fast(int act, float g) {
    if (act == INFR_ACT_SILU) return g / (1.0f + __expf(-g));
    if (act == INFR_ACT_GELU) {
        const float inner = 0.7978846f * (g + 0.044715f * g * g * g);
        return 0.5f * g * (1.0f + tanhf(inner));
    }
    return 1.0f / (1.0f + __expf(-g));
}
// silu with the hardware exp2 and reciprocal (1 ulp each).  The product g * log2(e) is rounded, so the exponential is off by up to
// |g| 2^-24 of itself: 10 ulp at |g| = 20, where the f16 rounding of the result still hides it.  The reciprocal comes first:
// g * up may overflow where silu(g) is 0 (g < -88), and infinity times 0 is NaN.
__device__ __forceinline__ float silu_fast(float g) {
    return g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f));
}
__device__ __forceinline__ float gated_act_fast(int act, bool has_clamp, float clamp, float gate, float up) {
    if (has_clamp) {
        gate = gate < clamp ? gate : clamp;
        up = up < -clamp ? -clamp : up > clamp ? clamp : up;   // (a NaN stays)
    }
    return act_fast(act, gate) * up;
}

// One 16-byte load per lane straight from global memory into LDS: lane i's bytes land at lds_base + 16 i.  Inline assembly,
// so the compiler neither counts it nor orders LDS reads against it: the caller waits (vmcnt) before a barrier.
// M0 carries the LDS base of the transfer.  The statement writes M0 immediately before its only use, and nothing
// else in these kernels uses M0 (no other LDS-direct load, no indirect register addressing, no message), so no
// value of the compiler's can be live in it across the statement.  M0 cannot be named as a clobber: the compiler
// reserves the register and warns that it does not honour such a clobber.
__device__ __forceinline__ void dma16(const void* gsrc, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(gsrc), "s"(__builtin_amdgcn_readfirstlane(lds_base)) : "memory");
}
// the same from 32-bit offsets behind a uniform address
__device__ __forceinline__ void dma16(const void* gbase, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(gbase), "s"(__builtin_amdgcn_readfirstlane(lds_base)) : "memory");
}
// 4 bytes per lane, to lds_base + 4 i
__device__ __forceinline__ void dma4(const void* gbase, uint32_t off, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(gbase), "s"(__builtin_amdgcn_readfirstlane(lds_base)) : "memory");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}

// --------------------------------------------------------------------------------------------
struct Tile {
    int e, p0, cnt;
};
// The workgroup's item of the integer kernels, by the tile table of launch_bucket: (tile, column tile).  Items are ordered by
// (expert, group of up to kGroupTiles tiles of its bucket, column tile, tile), and each of the 8 XCDs, which workgroups go to
// round-robin and which have an L2 each, takes a contiguous eighth of them: the tiles of a group run beside each other on
// the same weights, which then come from memory once per group, while the group's activations stay in the L2 for its
// columns.  Uniform; false when there is nothing to do (the grid is an upper bound).
constexpr int kGroupTiles = 4;
__device__ __forceinline__ int group_column(uint32_t r, int in_group) {   // item r of a group of in_group tiles: r / in_group
    return (int)(in_group == 1 ? r : in_group == 2 ? r >> 1 : in_group == 3 ? __umulhi(r, 0x55555556u) : r >> 2);
}
__device__ __forceinline__ bool tile_item(const int4* __restrict__ tiles, int n_cols, uint32_t n_cols_rcp, int tile_pairs, Tile& t, int& col) {
    const int n_items = tiles[0].x * n_cols, per = (n_items + 7) >> 3, k = (int)(blockIdx.x >> 3);
    const int item = (int)(blockIdx.x & 7) * per + k;
    if (k >= per || item >= n_items) return false;
    const int some = n_cols == 1 ? item : (int)__umulhi((uint32_t)item, n_cols_rcp);   // item / n_cols: exact below 2^32 / n_cols
    const int4 b = tiles[1 + some];   // expert, its first pair, its pairs, its first tile
    const int first = (some - b.w) & ~(kGroupTiles - 1), in_group = min(kGroupTiles, (b.z + tile_pairs - 1) / tile_pairs - first);
    const int r = item - (b.w + first) * n_cols, c = group_column((uint32_t)r, in_group);
    const int at = (first + r - c * in_group) * tile_pairs;
    t = Tile{b.x, b.y + at, min(tile_pairs, b.z - at)};
    col = c;
    return true;
}

// The block's work item of the float kernel: (expert, kBM-row tile of its bucket, column tile nt), items ordered by
// expert, row tile, column tile.  Workgroups go to the chip's 8 XCDs round-robin by workgroup id
// and every XCD has its own L2, so each XCD takes a contiguous eighth of the items: the column
// tiles of one row tile, which read the same activation tile, then sit behind the same L2.
// Uniform per wave; false when the block has nothing to do (the grid is an upper bound).
__device__ __forceinline__ bool find_item(const int32_t* __restrict__ offsets, int n_expert, int n_tiles_n, int lane,
                                          Tile& t, int& nt) {
    const int epl = (n_expert + 63) >> 6;
    const int e_lo = lane * epl, e_hi = min(n_expert, e_lo + epl);
    int mine = 0;
    for (int e = e_lo; e < e_hi; e++) mine += (offsets[e + 1] - offsets[e] + kBM - 1) / kBM;
    int incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    const int n_items = __shfl(incl, 63, 64) * n_tiles_n;
    const int per = (n_items + 7) >> 3;
    const int k = (int)(blockIdx.x >> 3);
    const int item = (int)(blockIdx.x & 7) * per + k;
    if (k >= per || item >= n_items) return false;
    nt = item % n_tiles_n;
    const int tile = item / n_tiles_n;
    const unsigned long long past = __ballot(incl > tile);
    if (past == 0) return false;
    const int owner = __ffsll((long long)past) - 1;
    int rem = tile - (__shfl(incl, owner, 64) - __shfl(mine, owner, 64));
    const int o_lo = owner * epl, o_hi = min(n_expert, o_lo + epl);
    for (int e = o_lo; e < o_hi; e++) {
        const int cnt = offsets[e + 1] - offsets[e];
        const int ntile = (cnt + kBM - 1) / kBM;
        if (rem < ntile) {
            t.e = e;
            t.p0 = offsets[e] + rem * kBM;
            t.cnt = min(kBM, cnt - rem * kBM);
            return true;
        }
        rem -= ntile;
    }
    return false;
}

// Epilogue of a tile whose accumulators are acc0/acc1[M] (column tiles of the wave, M 32-row
// sub-tiles): SwiGLU of (gate, up) or the scaled down-projection row, stored to p.out.
template <bool DOWN, int M>
__device__ __forceinline__ void tile_epilogue(const GroupedParams& p, const Tile& t, int n0, int wave, int lane,
                                              const float* s_scale, const float16v (&acc0)[M], const float16v (&acc1)[M]) {
    // accumulator register r of a 32x32 tile: row 8*(r/4) + 4*(lane/32) + r%4, column lane%32.
    // The epilogue variant is chosen once, outside the loops; rows below the last 32-row sub-tile
    // are all inside the tile, so only that sub-tile tests the row count.
    const int fc0 = n0 + (DOWN ? 64 : 32) * wave + (lane & 31);   // the lane's column (second column tile of DOWN: + 32)
    float* const obase = p.out + (size_t)t.p0 * p.N + fc0;
    const int mrow = 4 * (lane >> 5);
    auto for_each = [&](auto&& body) {
#pragma unroll
        for (int mi = 0; mi < M; mi++) {
#pragma unroll
            for (int r4 = 0; r4 < 4; r4++) {
                const int m0 = 32 * mi + 8 * r4 + mrow;   // rows m0 .. m0 + 3
                const float4 sc4 = *reinterpret_cast<const float4*>(s_scale + m0);
                const float scs[4] = {sc4.x, sc4.y, sc4.z, sc4.w};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int m = m0 + i;
                    if (mi < M - 1 || m < t.cnt) body(mi, 4 * r4 + i, m, scs[i], obase + (size_t)m * p.N);
                }
            }
        }
    };
    if (DOWN && p.out_f16) {
        // f16 without the row's power-of-two scale (|acc| stays far inside the f16 range: the
        // activation rows were normalised below 1); the combine multiplies the scale back in
        const float ds = p.down_scale ? p.down_scale[t.e] : 1.0f;
        const bool ok0 = fc0 < p.N, ok1 = fc0 + 32 < p.N;
        _Float16* const hbase = reinterpret_cast<_Float16*>(p.out) + (size_t)t.p0 * p.N + fc0;
        if (ok0) {
            for_each([&](int mi, int r, int m, float, float*) {
                _Float16* o = hbase + (size_t)m * p.N;
                o[0] = (_Float16)(acc0[mi][r] * ds);
                if (ok1) o[32] = (_Float16)(acc1[mi][r] * ds);
            });
        }
    } else if (DOWN) {
        const float ds = p.down_scale ? p.down_scale[t.e] : 1.0f;
        const bool ok0 = fc0 < p.N, ok1 = fc0 + 32 < p.N;
        if (ok1) {
            for_each([&](int mi, int r, int, float sc, float* o) {
                o[0] = acc0[mi][r] * sc * ds;
                o[32] = acc1[mi][r] * sc * ds;
            });
        } else if (ok0) {
            for_each([&](int mi, int r, int, float sc, float* o) { o[0] = acc0[mi][r] * sc * ds; });
        }
    } else if (fc0 < p.N) {
        if (p.act == INFR_ACT_SILU && !p.has_clamp && !p.weight_before) {
            for_each([&](int mi, int r, int, float sc, float* o) {
                const float g = acc0[mi][r] * sc, u = acc1[mi][r] * sc;
                o[0] = silu_fast(g) * u;
            });
        } else {
            for_each([&](int mi, int r, int m, float sc, float* o) {
                float g = acc0[mi][r] * sc, u = acc1[mi][r] * sc;
                if (p.weight_before) {
                    const float wp = p.route_w[p.pair_src[t.p0 + min(m, t.cnt - 1)]];
                    g *= wp;
                    u *= wp;
                }
                o[0] = gated_act_fast(p.act, p.has_clamp, p.clamp, g, u);
            });
        }
    }
}

}  // namespace

}  // namespace infr
