// Batched Op::MoeFfn: token -> expert bucketing and per-expert grouped GEMMs on the matrix cores.
//
// The CPU reference groups the (token row, rank) pairs of a batch by expert, experts ascending
// and rows ascending inside a bucket (crates/infr-cpu/src/lib.rs:3874-3908), and runs one GEMM
// per bucket (crates/infr-cpu/src/moe.rs:142-173).  Here:
//
//   bucket_kernel         offsets[e] = number of pairs whose expert id is below e, and the stable
//                         scatter of the pairs into that order (one block per expert; order is
//                         an integer contract and is reproduced exactly).  route_bucket_kernel: the same behind the routing
//                         of a few rows, in one launch.
//   rows_to_f16_kernel    activation rows -> f16 with one power-of-two scale per row (so any f32
//                         magnitude fits), laid out in the k order the weight format unpacks to
//                         (the token rows beside the bucketing, in its launch)
//   grouped_gemm / grouped_float_mfma   the GEMMs (k_grouped_gemm.hip, k_grouped_float.hip)
//   unbucket_combine      dst[row] = sum over ranks (rank order, separate mul and add,
//                         lib.rs:4290-4302) of w * y[pair of (row, rank)].
//
// The order in which codes fall out of a dword is not the element order; since a dot product does not care about the order
// of its terms, the activation rows are stored in that same ("virtual") order.
#include "grouped_common.h"
#include "route.h"

namespace infr {

namespace {

// --------------------------------------------------------------------------------------------
// A row's power-of-two scale from its largest magnitude.
__device__ __forceinline__ int row_exponent(float m) {
    int e = 0;
    if (m > 0.0f && m < __builtin_inff()) (void)frexpf(m, &e);  // m = f * 2^e, f in [0.5, 1)
    return e;
}
// Chunk c of a row (elements lo .. lo + 3 and hi .. hi + 3) times `inv` as f16; formats with minimums: also the sum of the rounded
// values over each group of 32 (four chunks: c ^ 1, c ^ 4, in the lanes ^ 1 and ^ 4), as an f16 pair high + low:
// sums[row][256 k][high, low][8 groups].
template <class F>   // F: k order of a weight format (grouped_common.h)
__device__ __forceinline__ uint4 chunk_to_f16(float4 a, float4 b, float inv, int c, uint32_t* __restrict__ row_sums) {
    auto two = [&](float u, float v) { return half2v{(_Float16)(u * inv), (_Float16)(v * inv)}; };
    half2v h0, h1, h2, h3;
    if constexpr (F::kMix == kSwapped) {
        h0 = two(a.x, a.z), h1 = two(a.y, a.w), h2 = two(b.x, b.z), h3 = two(b.y, b.w);
    } else if constexpr (F::kMix == kPairs) {
        h0 = two(a.x, b.x), h1 = two(a.y, b.y), h2 = two(a.z, b.z), h3 = two(a.w, b.w);
    } else {
        h0 = two(a.x, a.y), h1 = two(a.z, a.w), h2 = two(b.x, b.y), h3 = two(b.z, b.w);
    }
    if constexpr (F::kHasMin) {
        float s = ((float)h0[0] + (float)h0[1]) + ((float)h1[0] + (float)h1[1]) + (((float)h2[0] + (float)h2[1]) + ((float)h3[0] + (float)h3[1]));
        s += __shfl_xor(s, 1, 64);
        s += __shfl_xor(s, 4, 64);
        if ((c & 5) == 0) {
            const int g = c >> 3 << 1 | (c >> 1 & 1);
            _Float16* o = reinterpret_cast<_Float16*>(row_sums) + (g >> 3) * 16 + (g & 7);
            const _Float16 hi = (_Float16)s;
            o[0] = hi;
            o[8] = (_Float16)(s - (float)hi);
        }
    }
    return uint4{as_u32(h0), as_u32(h1), as_u32(h2), as_u32(h3)};
}

// A row by 256 threads (t: the thread's place among them): amax -> power-of-two scale -> f16 in the virtual k order of format F.
// Rows of up to 2048 kHold wait in registers for their scale, longer ones are read twice.  All threads of the block pass the one barrier.
template <class F>
__device__ __forceinline__ void row_to_f16(const float* __restrict__ src, int n, _Float16* __restrict__ dst, float* __restrict__ scale,
                                           size_t row, int t, float* s_max, uint32_t* __restrict__ sums, bool live = true) {
    constexpr int kHold = 2;   // chunks of 8 elements a thread holds
    const float* x = src + row * n;
    uint4* out = reinterpret_cast<uint4*>(dst + row * n);
    uint32_t* row_sums = sums + row * (n / 32);
    const bool held = n <= 2048 * kHold;
    float4 a[kHold], b[kHold];
    float m = 0.0f;
    if (held) {
#pragma unroll
        for (int i = 0; i < kHold; i++) {   // (threads behind the row's end repeat its last chunk)
            const int c = min(256 * i + t, n / 8 - 1);
            a[i] = *reinterpret_cast<const float4*>(x + F::lo(c));
            b[i] = *reinterpret_cast<const float4*>(x + F::hi(c));
        }
#pragma unroll
        for (int i = 0; i < kHold; i++) {
            m = fmaxf(fmaxf(m, fmaxf(fabsf(a[i].x), fabsf(a[i].y))), fmaxf(fabsf(a[i].z), fabsf(a[i].w)));
            m = fmaxf(fmaxf(m, fmaxf(fabsf(b[i].x), fabsf(b[i].y))), fmaxf(fabsf(b[i].z), fabsf(b[i].w)));
        }
    } else {
        for (int k = t * 4; k < n; k += 1024) {
            const float4 v = *reinterpret_cast<const float4*>(x + k);
            m = fmaxf(fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y))), fmaxf(fabsf(v.z), fabsf(v.w)));
        }
    }
    m = wave_max(m);
    if ((t & 63) == 0) s_max[t >> 6] = m;
    __syncthreads();
    if (!live) return;
    m = fmaxf(fmaxf(s_max[0], s_max[1]), fmaxf(s_max[2], s_max[3]));
    const int e = row_exponent(m);
    const float inv = ldexpf(1.0f, -e);
    if (t == 0) scale[row] = ldexpf(1.0f, e);
    if (held) {
#pragma unroll
        for (int i = 0; i < kHold; i++)
            if (256 * i + t < n / 8) out[256 * i + t] = chunk_to_f16<F>(a[i], b[i], inv, 256 * i + t, row_sums);
    } else {
        for (int c = t; c < n / 8; c += 256)
            out[c] = chunk_to_f16<F>(*reinterpret_cast<const float4*>(x + F::lo(c)), *reinterpret_cast<const float4*>(x + F::hi(c)), inv, c, row_sums);
    }
}

// The f16 conversion of a batch's token rows for the gate/up GEMM, which a bucketing launch takes along: it depends on nothing that the
// routing made, and the bucketing is a chain of latencies on n_expert + 1 blocks.  The blocks behind those convert a row per 256 threads.
// In the routing's launch, ahead of a row's routing on the same wavefronts, it took us a pass: two layers of 64 rows 238.2 and here 236.2,
// 333 rows 127.9 and 126.5, 2048 rows 326.5 and 324.1 (2048 rows, us a launch: routing with conversion 14.9, bucketing 14.3; now 8 and 16).
template <class F, int NT>
__device__ __forceinline__ void rows_beside(const RowsToF16& c, int block) {
    __shared__ float s_max[NT / 64];
    const int q = threadIdx.x >> 8, row = block * (NT / 256) + q;
    row_to_f16<F>(c.src, c.n, reinterpret_cast<_Float16*>(c.dst), c.scale, (size_t)min(row, c.rows - 1), threadIdx.x & 255, s_max + 4 * q, c.sums, row < c.rows);
}

// A wavefront per row of up to 512 NC elements, four rows per block: the row is read once and waits in registers for its scale
// (a block per row, read twice across a barrier: 16384 rows of 768 18.1 us, so 13.5).
template <class F, int NC>
__global__ __launch_bounds__(256) void rows_to_f16_wave_kernel(const float* __restrict__ src, int rows, int n, _Float16* __restrict__ dst,
                                                               float* __restrict__ scale, uint32_t* __restrict__ sums) {
    const int lane = threadIdx.x & 63;
    const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= (size_t)rows) return;
    const float* x = src + row * n;
    float4 a[NC], b[NC];
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < NC; i++) {   // (lanes behind the row's end repeat its last chunk)
        const int c = min(64 * i + lane, n / 8 - 1);
        a[i] = *reinterpret_cast<const float4*>(x + F::lo(c));
        b[i] = *reinterpret_cast<const float4*>(x + F::hi(c));
    }
#pragma unroll
    for (int i = 0; i < NC; i++) {
        m = fmaxf(fmaxf(m, fmaxf(fabsf(a[i].x), fabsf(a[i].y))), fmaxf(fabsf(a[i].z), fabsf(a[i].w)));
        m = fmaxf(fmaxf(m, fmaxf(fabsf(b[i].x), fabsf(b[i].y))), fmaxf(fabsf(b[i].z), fabsf(b[i].w)));
    }
    const int e = row_exponent(wave_max(m));
    const float inv = ldexpf(1.0f, -e);
    if (lane == 0) scale[row] = ldexpf(1.0f, e);
    uint4* out = reinterpret_cast<uint4*>(dst + row * n);
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const int c = 64 * i + lane;
        if (c < n / 8) out[c] = chunk_to_f16<F>(a[i], b[i], inv, c, sums + row * (n / 32));
    }
}

template <class F>
__global__ __launch_bounds__(256) void rows_to_f16_kernel(const float* __restrict__ src, int n,
                                                          _Float16* __restrict__ dst, float* __restrict__ scale, uint32_t* __restrict__ sums) {
    __shared__ float s_max[4];
    row_to_f16<F>(src, n, dst, scale, blockIdx.x, threadIdx.x, s_max, sums);
}

// --------------------------------------------------------------------------------------------
// The size class of an expert's bucket, by which the tile table is ordered.
__device__ __forceinline__ int size_class(uint32_t pairs) { return pairs <= 16 ? 0 : pairs > 256 ? 5 : 32 - __clz((pairs - 1) >> 4); }

// Up to NT * J pairs: one block of NT / 64 wavefronts per expert e in 0..n_expert; the extra one marks pairs whose id is out of
// range.  A thread holds the ids of pairs tid, tid + NT, ... in registers; the block counts every expert's pairs (those of the
// experts below e give the bucket's offset and its tiles' places in the tile table; consecutive lanes hold consecutive pairs, and
// the ids of one token differ, so few lanes meet on one counter), and then scatters the pairs equal to e: a ballot per 64 pairs
// gives the places among them, the ballots' counts in flat (row, rank) order the rest, so buckets come out rows ascending.
// A chain of latencies: the launch, the ids, the counters, two barriers.  What it takes, us a launch against the ids staged in LDS and scanned twice from there, 128 experts, top-8: 16 rows
// 5.04 and 4.95, 64 rows 5.47 and 5.09, 2048 rows 14.7 and 14.3; us a pass: 3 layers of 16 rows in Q8_0 358.5 and 354.5, two of 64 in
// Q4_K / Q6_K 241.8 and 239.5, 333 rows in Q5_K 126.5 and 125.2, 512 in Q8_0 166.1 and 164.7.
constexpr int kBucketFew = 2048, kBucketMany = 16384;
template <class F, int NT, int J>
__global__ __launch_bounds__(NT) void bucket_once_kernel(const int32_t* __restrict__ ids, int n_pairs, int n_expert, int n_used,
                                                         int32_t* __restrict__ offsets, int32_t* __restrict__ pair_src,
                                                         int32_t* __restrict__ slot_pair, int32_t* __restrict__ pair_row,
                                                         int4* __restrict__ tiles, int tile, int by_size, int always_rows, RowsToF16 conv) {
    if ((int)blockIdx.x > n_expert) {
        rows_beside<F, NT>(conv, blockIdx.x - n_expert - 1);
        return;
    }
    constexpr int NW = NT / 64;
    static_assert(NW % 4 == 0 && J * NW <= 256, "");
    __shared__ uint32_t s_hist[2048];                                  // n_expert <= 2048
    __shared__ __attribute__((aligned(16))) uint32_t s_hits[256];      // pairs of e among 64 j NW + 64 wave ...
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t e = blockIdx.x;
    uint32_t id[J];
#pragma unroll
    for (int j = 0; j < J; j++) {
        id[j] = ~0u;
        if (j * NT < n_pairs) id[j] = (uint32_t)ids[min(j * NT + tid, n_pairs - 1)];
    }
    for (int i = tid; i < n_expert; i += NT) s_hist[i] = 0;
    if (tid < 256) s_hits[tid] = 0;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < J; j++) {
        if (j * NT >= n_pairs) break;
        if (j * NT + tid >= n_pairs || id[j] >= (uint32_t)n_expert) id[j] = ~0u;
        else atomicAdd(&s_hist[id[j]], 1u);
        const uint32_t hits = __builtin_popcountll(__ballot(id[j] == e));
        if (lane == 0) s_hits[j * NW + wave] = hits;
    }
    __syncthreads();
    // every wavefront for itself: the bucket's offset and its tiles' places, and where its own pairs of e go
    const uint32_t own = e < (uint32_t)n_expert ? s_hist[e] : (uint32_t)always_rows;
    uint32_t below = 0, tiles_below = 0, tiles_all = 0;
    for (int i = lane; i <= n_expert; i += 64) {
        const uint32_t c = i < n_expert ? s_hist[i] : (uint32_t)always_rows, nt = (c + tile - 1) / tile;
        if (i < (int)e) below += c;
        tiles_all += nt;
        if (by_size && size_class(c) != size_class(own) ? c > own : i < (int)e) tiles_below += nt;
    }
    const uint4 h = *reinterpret_cast<const uint4*>(&s_hits[4 * lane]);
    uint32_t incl = h.x + h.y + h.z + h.w;
    const uint32_t quad = incl;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        below += __shfl_xor(below, d, 64);
        tiles_below += __shfl_xor(tiles_below, d, 64);
        tiles_all += __shfl_xor(tiles_all, d, 64);
        const uint32_t o = __shfl_up(incl, d, 64);
        if (lane >= d) incl += o;
    }
    if (tid == 0) offsets[e] = (int32_t)below;
    if (tiles) {   // slot 0: the number of tiles; then the tiles
        if (e == (uint32_t)n_expert && tid == 0) tiles[0] = make_int4((int)tiles_all, 0, 0, 0);
        const int cnt = (int)own, first = e == (uint32_t)n_expert ? n_pairs : (int)below;
        for (int i = tid; i * tile < cnt; i += NT)
            tiles[1 + tiles_below + i] = by_size ? make_int4((int)e, first + i * tile, min(tile, cnt - i * tile), 0)
                                                 : make_int4((int)e, first, cnt, (int)tiles_below);
        if (e == (uint32_t)n_expert)
            for (int i = tid; i < always_rows; i += NT) pair_row[n_pairs + i] = i;
    }
    if (e == (uint32_t)n_expert) {
#pragma unroll
        for (int j = 0; j < J; j++)
            if (j * NT + tid < n_pairs && id[j] == ~0u) slot_pair[j * NT + tid] = -1;
        return;
    }
    const int sub = wave & 3;
    const uint32_t before = below + incl - quad + (sub > 0 ? h.x : 0u) + (sub > 1 ? h.y : 0u) + (sub > 2 ? h.z : 0u);
#pragma unroll
    for (int j = 0; j < J; j++) {
        if (j * NT >= n_pairs) break;
        const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)before, j * (NW / 4) + (wave >> 2));
        const uint64_t hits = __ballot(id[j] == e);
        if (id[j] == e) {
            const int i = j * NT + tid;
            const uint32_t pos = base + __builtin_popcountll(hits & ((1ull << lane) - 1));
            pair_src[pos] = i;
            slot_pair[i] = (int32_t)pos;
            if (pair_row) pair_row[pos] = i / n_used;
        }
    }
}

// More pairs: one block of sixteen wavefronts per expert e in 0..n_expert as above.  The block stages the pair ids in LDS (16-bit, in
// chunks), counts every expert's pairs, and then scatters the pairs equal to e: each wavefront takes a
// contiguous part of the chunk, the parts' hit counts give every wavefront its base, and inside a part a wave-wide prefix keeps the
// flat (row, rank) order.
template <class F, int NT>
__global__ __launch_bounds__(NT) void bucket_kernel(const int32_t* __restrict__ ids, int n_pairs, int n_expert,
                                                     int n_used, int32_t* __restrict__ offsets, int32_t* __restrict__ pair_src,
                                                     int32_t* __restrict__ slot_pair, int32_t* __restrict__ pair_row,
                                                     int4* __restrict__ tiles, int tile, int by_size, int always_rows, RowsToF16 conv) {
    if ((int)blockIdx.x > n_expert) {
        rows_beside<F, NT>(conv, blockIdx.x - n_expert - 1);
        return;
    }
    constexpr int kBucketChunk = kBucketMany;
    constexpr int NW = NT / 64, NL = kBucketChunk / 4 / NT;
    __shared__ __attribute__((aligned(16))) uint16_t s_ids[kBucketChunk];
    __shared__ uint32_t s_hist[2048];
    __shared__ uint32_t s_cnt[3 * NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t e = blockIdx.x;
    auto narrow = [&](int32_t v) { return (uint32_t)v < (uint32_t)n_expert ? (uint32_t)v : 0xFFFFu; };  // n_expert <= 2048
    auto stage = [&](int c0, int cn) {
        __syncthreads();  // orders the LDS reads of the previous chunk before these writes
        // full groups of four ids: all of a thread's unconditional (index-clamped) 16-byte loads in flight
        const int full = cn & ~3;
        if (full) {
            int4 v[NL];
#pragma unroll
            for (int j = 0; j < NL; j++) {
                const int i = min((j * NT + tid) * 4, full - 4);
                v[j] = *reinterpret_cast<const int4*>(ids + c0 + i);
            }
#pragma unroll
            for (int j = 0; j < NL; j++) {
                const int i = (j * NT + tid) * 4;
                if (i < full) {
                    const uint32_t lo = narrow(v[j].x) | (narrow(v[j].y) << 16), hi = narrow(v[j].z) | (narrow(v[j].w) << 16);
                    *reinterpret_cast<uint2*>(&s_ids[i]) = make_uint2(lo, hi);
                }
            }
        }
        // the last one to three ids, padded to a group of four with 0xFFFF
        if (tid < 4 && full < cn) s_ids[full + tid] = full + tid < cn ? (uint16_t)narrow(ids[c0 + full + tid]) : (uint16_t)0xFFFF;
        __syncthreads();
    };
    // eight ids of group g (one 128-bit LDS read); the staging filled the chunk's last partial group
    // of four with 0xFFFF, the tail of a partial group of eight is masked here
    auto ids8 = [&](int g, int cn, uint32_t (&id)[8]) {
        const uint4 v = *reinterpret_cast<const uint4*>(&s_ids[8 * g]);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 8; c++) {
            id[c] = (w[c >> 1] >> (16 * (c & 1))) & 0xFFFFu;
            if (8 * g + c >= ((cn + 3) & ~3)) id[c] = 0xFFFFu;
        }
    };
    auto wave_total = [&](uint32_t v) {
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
        return v;
    };

    // ---- pass 0: how many pairs each expert has; from that the bucket's offset and its tiles' places in the tile table
    for (int i = tid; i < n_expert; i += NT) s_hist[i] = 0;
    for (int c0 = 0; c0 < n_pairs; c0 += kBucketChunk) {
        const int cn = min(kBucketChunk, n_pairs - c0);
        stage(c0, cn);   // (its barriers also order the clearing above)
        // consecutive lanes take consecutive pairs: the ids of one token differ, so few lanes meet on one counter
        for (int i0 = 0; i0 < cn; i0 += NT * 8) {
            uint32_t id[8];
#pragma unroll
            for (int j = 0; j < 8; j++) id[j] = s_ids[min(i0 + NT * j + tid, cn - 1)];
#pragma unroll
            for (int j = 0; j < 8; j++)
                if (i0 + NT * j + tid < cn && id[j] != 0xFFFFu) atomicAdd(&s_hist[id[j]], 1u);
        }
    }
    __syncthreads();
    const uint32_t own = e < (uint32_t)n_expert ? s_hist[e] : (uint32_t)always_rows;
    uint32_t below = 0, tiles_below = 0, tiles_all = 0;
    for (int i = tid; i <= n_expert; i += NT) {
        const uint32_t c = i < n_expert ? s_hist[i] : (uint32_t)always_rows, nt = (c + tile - 1) / tile;
        if (i < (int)e) below += c;
        tiles_all += nt;
        if (by_size && size_class(c) != size_class(own) ? c > own : i < (int)e) tiles_below += nt;
    }
    below = wave_total(below);
    tiles_below = wave_total(tiles_below);
    tiles_all = wave_total(tiles_all);
    if (lane == 0) { s_cnt[wave] = below; s_cnt[NW + wave] = tiles_below; s_cnt[2 * NW + wave] = tiles_all; }
    __syncthreads();
    below = tiles_below = tiles_all = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) below += s_cnt[w], tiles_below += s_cnt[NW + w], tiles_all += s_cnt[2 * NW + w];
    if (tid == 0) offsets[e] = (int32_t)below;
    if (tiles) {   // slot 0: the number of tiles; then the tiles
        if (e == (uint32_t)n_expert && tid == 0) tiles[0] = make_int4((int)tiles_all, 0, 0, 0);
        const int cnt = (int)own, first = e == (uint32_t)n_expert ? n_pairs : (int)below;
        for (int i = tid; i * tile < cnt; i += NT)
            tiles[1 + tiles_below + i] = by_size ? make_int4((int)e, first + i * tile, min(tile, cnt - i * tile), 0)
                                                 : make_int4((int)e, first, cnt, (int)tiles_below);
        if (e == (uint32_t)n_expert)
            for (int i = tid; i < always_rows; i += NT) pair_row[n_pairs + i] = i;
    }

    // ---- pass 1: scatter the pairs with id e (the extra block: mark the ids out of range)
    uint32_t run = below;
    for (int c0 = 0; c0 < n_pairs; c0 += kBucketChunk) {
        const int cn = min(kBucketChunk, n_pairs - c0);
        stage(c0, cn);
        if (e == (uint32_t)n_expert) {
            for (int i = tid; i < cn; i += NT)
                if (s_ids[i] == 0xFFFFu) slot_pair[c0 + i] = -1;
            continue;
        }
        const int n8 = (cn + 7) >> 3;
        const int per_wave = (n8 + NT - 1) / NT * 64;   // whole steps of 64 groups
        const int g_lo = wave * per_wave, g_hi = min(n8, g_lo + per_wave);
        // hits of this wavefront's part
        uint32_t hits = 0;
        for (int g = g_lo + lane; g < g_hi; g += 64) {
            uint32_t id[8];
            ids8(g, cn, id);
#pragma unroll
            for (int c = 0; c < 8; c++) hits += id[c] == e;
        }
        hits = wave_total(hits);
        __syncthreads();   // the previous chunk's readers of s_cnt are done
        if (lane == 0) s_cnt[wave] = hits;
        __syncthreads();
        uint32_t base = run;
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const uint32_t h = s_cnt[w];
            base += w < wave ? h : 0;
            run += h;
        }
        for (int g0 = g_lo; g0 < g_hi; g0 += 64) {
            const int g = g0 + lane;
            uint32_t id[8];
#pragma unroll
            for (int c = 0; c < 8; c++) id[c] = 0xFFFFu;
            if (g < g_hi) ids8(g, cn, id);
            uint32_t mine = 0;
#pragma unroll
            for (int c = 0; c < 8; c++) mine += id[c] == e;
            // inclusive prefix of the per-lane hit counts (a lane's eight pairs are consecutive)
            uint32_t incl = mine;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(incl, d, 64);
                if (lane >= d) incl += o;
            }
            uint32_t pos = base + incl - mine;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                if (id[c] == e) {
                    pair_src[pos] = c0 + 8 * g + c;
                    slot_pair[c0 + 8 * g + c] = (int32_t)pos;
                    if (pair_row) pair_row[pos] = (c0 + 8 * g + c) / n_used;
                    pos++;
                }
            }
            base += __shfl(incl, 63, 64);
        }
    }
}

// Routing and bucketing of a few rows that choose among few experts, in one launch of one block: wavefront r routes row r, and the
// block then counts, scans and scatters the pairs in LDS (same order as bucket_kernel: a pair's place in its bucket is the number of
// earlier pairs of that expert).  Either alone is mostly its launch and a few dependent loads.  8 experts, top-2, 16 rows: two
// launches 11.4 us, this one 6.4.  More pairs or experts stay with two launches: the rows' serial sums and selection rounds then
// share four SIMDs, and the ranks below cost a pass over the pairs (16 rows of 128 experts, top-8: 11.4 us, in one launch 11.1 to 12.7).
constexpr int kRouteBucketRows = 16, kRouteBucketPairs = 32, kRouteBucketExperts = 64;
__global__ __launch_bounds__(64 * kRouteBucketRows) void route_bucket_kernel(RouteParams rp, int32_t* __restrict__ offsets,
                                                                            int32_t* __restrict__ pair_src, int32_t* __restrict__ slot_pair,
                                                                            int32_t* __restrict__ pair_row, int4* __restrict__ tiles) {
    extern __shared__ float lds[];
    __shared__ __attribute__((aligned(16))) uint16_t s_ids[kRouteBucketPairs];
    __shared__ uint32_t s_hist[kRouteBucketExperts];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n_expert = rp.n_expert, n_pairs = rp.rows * rp.n_used;
    uint64_t* tab = reinterpret_cast<uint64_t*>(lds);
    if (tid < 32) tab[tid] = kExp2Table[tid];
    if (tid < kRouteBucketExperts) s_hist[tid] = 0;
    __syncthreads();
    if (wave < rp.rows)
        route_row<kRouteBucketExperts / 64>(rp, wave, lane, lds + 64 + wave * route_scratch_floats(n_expert, rp.n_groups), tab, nullptr, nullptr, true, nullptr);
    __syncthreads();
    uint32_t id = 0xFFFFu;   // a pair's id, or "none": ids out of range are in no bucket
    if (tid < kRouteBucketPairs) {
        const uint32_t raw = tid < n_pairs ? (uint32_t)rp.ids[tid] : ~0u;
        if (raw < (uint32_t)n_expert) id = raw;
        s_ids[tid] = (uint16_t)id;
        if (id != 0xFFFFu) atomicAdd(&s_hist[id], 1u);
    }
    __syncthreads();
    if (wave == 0) {   // expert = lane: pairs and tiles below it, as two 16-bit sums
        const uint32_t cnt = s_hist[lane], own = cnt | (cnt + kIntTok - 1) / kIntTok << 16;
        uint32_t incl = own;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        const uint32_t first = (incl - own) & 0xFFFFu, tile0 = (incl - own) >> 16;
        s_hist[lane] = first;
        if (lane < n_expert) {
            offsets[lane] = (int32_t)first;
            if (tiles)
                for (uint32_t t = 0; t * kIntTok < cnt; t++) tiles[1 + tile0 + t] = make_int4(lane, (int)first, (int)cnt, (int)tile0);
        }
        if (lane == 63) {
            offsets[n_expert] = (int32_t)(incl & 0xFFFFu);
            if (tiles) tiles[0] = make_int4((int)(incl >> 16), 0, 0, 0);
        }
    }
    __syncthreads();
    if (tid >= n_pairs) return;
    if (id == 0xFFFFu) {
        slot_pair[tid] = -1;
        return;
    }
    uint32_t pos = s_hist[id];
    for (int g = 0; 8 * g < tid; g++) {
        const uint4 v = *reinterpret_cast<const uint4*>(&s_ids[8 * g]);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 8; c++) pos += 8 * g + c < tid && ((w[c >> 1] >> (16 * (c & 1))) & 0xFFFFu) == id;
    }
    pair_src[pos] = tid;
    slot_pair[tid] = (int32_t)pos;
    if (pair_row) pair_row[pos] = tid / rp.n_used;
}

// dst[row, :] = sum over ranks of w * y[slot_pair[row, rank], :], rank order, separate mul/add.
// Y = _Float16: y rows carry no row scale, pair_scale[pair] multiplies it back in.
template <class Y>
__global__ __launch_bounds__(256) void unbucket_combine_kernel(const Y* __restrict__ y, const int32_t* __restrict__ slot_pair,
                                                               const float* __restrict__ weights, int ne, int n_used,
                                                               int weight_before, float* dst, int identity,
                                                               const float* __restrict__ pair_scale, const float* addend,
                                                               int skip_zero_w, const float* __restrict__ shared, int parts, size_t part_stride) {
    const size_t row = blockIdx.y;
    const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= ne) return;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int k = 0; k < n_used; k++) {
        int pr = slot_pair ? slot_pair[row * n_used + k] : 0;
        if (pr < 0) continue;
        if (identity || !slot_pair) pr = (int)(row * n_used + k);
        if (skip_zero_w && weights[row * n_used + k] == 0.0f) continue;
        const float w = weight_before ? 1.0f : weights[row * n_used + k];
        const float sc = pair_scale ? pair_scale[pr] : 1.0f;
        const Y* yr = y + (size_t)pr * ne + i;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        if (i + 3 < ne) {
            if (sizeof(Y) == 2) {
                const uint2 raw = *reinterpret_cast<const uint2*>(yr);
                const half2v a = as_h2(raw.x), b = as_h2(raw.y);
                v[0] = (float)a[0]; v[1] = (float)a[1]; v[2] = (float)b[0]; v[3] = (float)b[1];
            } else {
                const float4 f = *reinterpret_cast<const float4*>(yr);
                v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
            }
        } else {
            for (int q = 0; i + q < ne; q++) v[q] = (float)yr[q];
        }
        for (int part = 1; part < parts; part++)
            for (int q = 0; q < 4 && i + q < ne; q++) v[q] += (float)yr[part * part_stride + q];
        if (pair_scale) {
#pragma unroll
            for (int q = 0; q < 4; q++) v[q] *= sc;
        }
        acc.x = __fadd_rn(acc.x, __fmul_rn(w, v[0]));
        acc.y = __fadd_rn(acc.y, __fmul_rn(w, v[1]));
        acc.z = __fadd_rn(acc.z, __fmul_rn(w, v[2]));
        acc.w = __fadd_rn(acc.w, __fmul_rn(w, v[3]));
    }
    if (shared) {   // the always-on expert's row, the Add that closes its ops
        float* a = &acc.x;
        for (int q = 0; q < 4 && i + q < ne; q++) a[q] = __fadd_rn(a[q], shared[row * ne + i + q]);
    }
    float* o = dst + row * ne + i;
    if (addend) {   // a following Op::Add folded in: the finished sum is added to the other operand
        const float* ad = addend + row * ne + i;
        if (i + 3 < ne) {
            const float4 f = *reinterpret_cast<const float4*>(ad);
            acc.x = __fadd_rn(f.x, acc.x); acc.y = __fadd_rn(f.y, acc.y);
            acc.z = __fadd_rn(f.z, acc.z); acc.w = __fadd_rn(f.w, acc.w);
        } else {
            float* a = &acc.x;
            for (int q = 0; i + q < ne; q++) a[q] = __fadd_rn(ad[q], a[q]);
        }
    }
    if (i + 3 < ne) *reinterpret_cast<float4*>(o) = acc;
    else {
        const float* a = &acc.x;
        for (int q = 0; i + q < ne; q++) o[q] = a[q];
    }
}

// A row's slots: pair row (0 for a dropped slot: a row that is read and not used), weight, whether it counts.  No load waits for another's
// answer, and none is behind a branch: with a branch per slot the eight slots' scalar loads waited for one another (us a pass, with and
// now: two layers of 64 rows of 128 experts, top-8, 236.1 and 232.3, 333 rows 137.5 and 136.6, 2048 rows 338.1 and 337.8).
template <int K>
__device__ __forceinline__ void combine_slots(const int32_t* __restrict__ slot_pair, const float* __restrict__ weights, size_t row, int identity,
                                              int skip_zero_w, int weight_before, int (&pr)[K], float (&w)[K], bool (&live)[K]) {
#pragma unroll
    for (int k = 0; k < K; k++) {
        w[k] = weights[row * K + k];
        pr[k] = (int)(row * K + k);
    }
    int slot[K];
#pragma unroll
    for (int k = 0; k < K; k++) slot[k] = pr[k];
    if (slot_pair) {
#pragma unroll
        for (int k = 0; k < K; k++) slot[k] = slot_pair[row * K + k];
    }
#pragma unroll
    for (int k = 0; k < K; k++) {   // (bits, not conditions: the compiler branches around those)
        const int drop = (slot[k] < 0) | ((skip_zero_w != 0) & ((__float_as_uint(w[k]) << 1) == 0u));
        live[k] = drop == 0;
        const int same = identity != 0 ? -1 : 0;
        pr[k] = ((pr[k] & same) | (slot[k] & ~same)) & (drop - 1);
        w[k] = weight_before ? 1.0f : w[k];
    }
}

// The same sum for f16 pair rows whose length is a multiple of 8: eight elements (16 bytes) per lane and slot, all
// slots of the row requested before the first is used.  Same operations per element as the kernel above.
template <int K>
__global__ __launch_bounds__(256) void unbucket_combine_h8_kernel(const _Float16* __restrict__ y, const int32_t* __restrict__ slot_pair,
                                                                  const float* __restrict__ weights, int ne, int weight_before,
                                                                  float* dst, int identity, const float* __restrict__ pair_scale,
                                                                  const float* addend, int skip_zero_w, const float* __restrict__ shared) {
    const size_t row = blockIdx.y;
    const int i = (blockIdx.x * 256 + threadIdx.x) * 8;
    if (i >= ne) return;
    float4 s0, s1, a0, a1;   // what is added behind the sum, requested ahead of it
    if (shared) s0 = *reinterpret_cast<const float4*>(shared + row * ne + i), s1 = *reinterpret_cast<const float4*>(shared + row * ne + i + 4);
    if (addend) a0 = *reinterpret_cast<const float4*>(addend + row * ne + i), a1 = *reinterpret_cast<const float4*>(addend + row * ne + i + 4);
    uint4 raw[K];
    float w[K], sc[K];
    bool live[K];
    int pr[K];
    combine_slots<K>(slot_pair, weights, row, identity, skip_zero_w, weight_before, pr, w, live);
#pragma unroll
    for (int k = 0; k < K; k++) {
        sc[k] = pair_scale[pr[k]];
        raw[k] = *reinterpret_cast<const uint4*>(y + (size_t)pr[k] * ne + i);
    }
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < K; k++) {
        const uint32_t d[4] = {raw[k].x, raw[k].y, raw[k].z, raw[k].w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const half2v h = as_h2(d[q]);
            const float t0 = __fadd_rn(acc[2 * q], __fmul_rn(w[k], (float)h[0] * sc[k]));
            const float t1 = __fadd_rn(acc[2 * q + 1], __fmul_rn(w[k], (float)h[1] * sc[k]));
            acc[2 * q] = live[k] ? t0 : acc[2 * q];
            acc[2 * q + 1] = live[k] ? t1 : acc[2 * q + 1];
        }
    }
    if (shared) {   // the always-on expert's row, the Add that closes its ops
        const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
        for (int q = 0; q < 8; q++) acc[q] = __fadd_rn(acc[q], sv[q]);
    }
    float* o = dst + row * ne + i;
    if (addend) {
        const float ad[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
        for (int q = 0; q < 8; q++) acc[q] = __fadd_rn(ad[q], acc[q]);
    }
    *reinterpret_cast<float4*>(o) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    *reinterpret_cast<float4*>(o + 4) = make_float4(acc[4], acc[5], acc[6], acc[7]);
}

// The same for f32 pair rows whose length is a multiple of 4: four elements per lane and slot, a wavefront per block, every
// slot requested before the first is used (a decode batch has few rows: 20 rows of 2048, top-8, 8.8 us in the kernel above, whose
// slots wait for one another on 40 blocks, 5 here).
template <int K>
__global__ __launch_bounds__(64) void unbucket_combine_f4_kernel(const float* __restrict__ y, const int32_t* __restrict__ slot_pair,
                                                                 const float* __restrict__ weights, int ne, int weight_before,
                                                                 float* dst, int identity, const float* addend, int skip_zero_w,
                                                                 int parts, size_t part_stride) {
    const size_t row = blockIdx.y;
    const int i = (blockIdx.x * 64 + threadIdx.x) * 4;
    if (i >= ne) return;
    float4 a0;   // what is added behind the sum, requested ahead of it
    if (addend) a0 = *reinterpret_cast<const float4*>(addend + row * ne + i);
    float4 v[K];
    float w[K];
    size_t at[K];
    bool live[K];
    int pr[K];
    combine_slots<K>(slot_pair, weights, row, identity, skip_zero_w, weight_before, pr, w, live);
#pragma unroll
    for (int k = 0; k < K; k++) at[k] = (size_t)pr[k] * ne + i;
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = *reinterpret_cast<const float4*>(y + at[k]);
    for (int part = 1; part < parts; part++) {
        float4 f[K];
#pragma unroll
        for (int k = 0; k < K; k++) f[k] = *reinterpret_cast<const float4*>(y + part * part_stride + at[k]);
        __builtin_amdgcn_sched_barrier(0);   // all of a part's loads in flight
#pragma unroll
        for (int k = 0; k < K; k++) { v[k].x += f[k].x; v[k].y += f[k].y; v[k].z += f[k].z; v[k].w += f[k].w; }
    }
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const float4 t = make_float4(__fadd_rn(acc.x, __fmul_rn(w[k], v[k].x)), __fadd_rn(acc.y, __fmul_rn(w[k], v[k].y)),
                                     __fadd_rn(acc.z, __fmul_rn(w[k], v[k].z)), __fadd_rn(acc.w, __fmul_rn(w[k], v[k].w)));
        acc.x = live[k] ? t.x : acc.x; acc.y = live[k] ? t.y : acc.y; acc.z = live[k] ? t.z : acc.z; acc.w = live[k] ? t.w : acc.w;
    }
    if (addend) {
        acc.x = __fadd_rn(a0.x, acc.x); acc.y = __fadd_rn(a0.y, acc.y);
        acc.z = __fadd_rn(a0.z, acc.z); acc.w = __fadd_rn(a0.w, acc.w);
    }
    *reinterpret_cast<float4*>(dst + row * ne + i) = acc;
}

// calls f with the k order of a weight format
template <class Fn>
void with_order(int dt, Fn&& f) {
    switch (dt) {
        case INFR_Q4K: case INFR_Q5K: f(Order4K{}); break;
        case INFR_Q6K: f(Order6K{}); break;
        case INFR_Q4_0: f(OrderNibbles<kSwapped>{}); break;
        case INFR_IQ4_XS: f(OrderNibbles<kPlain>{}); break;
        case INFR_MXFP4: f(OrderNibbles<kPairs>{}); break;
        default: f(OrderPlain{}); break;
    }
}

}  // namespace

void launch_rows_to_f16(hipStream_t s, int weight_dt, const float* src, int rows, int n, void* dst, float* scale, uint32_t* sums) {
    if (rows <= 0) return;
    _Float16* d = reinterpret_cast<_Float16*>(dst);
    const int nc = rows < 1024 ? 0 : (n / 8 + 63) / 64;   // few rows: a block each reaches more CUs
    with_order(weight_dt, [&](auto order) {
        typedef decltype(order) F;
        const dim3 quads((rows + 3) / 4);
        if (nc == 1) INFR_LAUNCH((rows_to_f16_wave_kernel<F, 1>), quads, dim3(256), 0, s, src, rows, n, d, scale, sums);
        else if (nc == 2) INFR_LAUNCH((rows_to_f16_wave_kernel<F, 2>), quads, dim3(256), 0, s, src, rows, n, d, scale, sums);
        else if (nc == 3) INFR_LAUNCH((rows_to_f16_wave_kernel<F, 3>), quads, dim3(256), 0, s, src, rows, n, d, scale, sums);
        else if (nc == 4) INFR_LAUNCH((rows_to_f16_wave_kernel<F, 4>), quads, dim3(256), 0, s, src, rows, n, d, scale, sums);
        else INFR_LAUNCH(rows_to_f16_kernel<F>, dim3(rows), dim3(256), 0, s, src, n, d, scale, sums);
    });
}

void launch_bucket(hipStream_t s, const int32_t* ids, int n_pairs, int n_expert, int n_used, int32_t* offsets, int32_t* pair_src,
                   int32_t* slot_pair, int32_t* pair_row, int4* tiles, int tile, int by_size, int always_rows, const RowsToF16* conv) {
    const int nt = n_pairs <= kBucketFew ? 256 : 1024;
    const RowsToF16 c = conv ? *conv : RowsToF16{};
    const dim3 grid(n_expert + 1 + (c.rows + nt / 256 - 1) / (nt / 256)), block(nt);
#define INFR_BUCKET(...)                                                                                                             \
    INFR_LAUNCH((__VA_ARGS__), grid, block, 0, s, ids, n_pairs, n_expert, n_used, offsets, pair_src, slot_pair, pair_row, tiles, tile, \
                by_size, always_rows, c)
    with_order(conv ? conv->weight_dt : INFR_F32, [&](auto order) {
        typedef decltype(order) F;
        if (n_pairs <= kBucketFew) INFR_BUCKET(bucket_once_kernel<F, 256, kBucketFew / 256>);
        else if (n_pairs <= kBucketMany) INFR_BUCKET(bucket_once_kernel<F, 1024, kBucketMany / 1024>);
        else INFR_BUCKET(bucket_kernel<F, 1024>);
    });
#undef INFR_BUCKET
}

bool launch_route_bucket(hipStream_t s, const RouteParams& rp, int32_t* offsets, int32_t* pair_src, int32_t* slot_pair, int32_t* pair_row,
                         int4* tiles) {
    const size_t lds = (64 + rp.rows * route_scratch_floats(rp.n_expert, rp.n_groups)) * sizeof(float);
    if (rp.rows < 1 || rp.rows > kRouteBucketRows || rp.rows * rp.n_used > kRouteBucketPairs || rp.n_expert > kRouteBucketExperts || lds > 48 * 1024)
        return false;
    INFR_LAUNCH(route_bucket_kernel, dim3(1), dim3(64 * kRouteBucketRows), lds, s, rp, offsets, pair_src, slot_pair, pair_row, tiles);
    return true;
}

void launch_unbucket_combine(hipStream_t s, const void* y, const int32_t* slot_pair, const float* weights, int rows,
                             int ne, int n_used, int weight_before, float* dst, int identity, const float* pair_scale,
                             const float* addend, int skip_zero_w, const float* shared, int parts, size_t part_stride) {
    if (rows <= 0) return;
    const dim3 grid((ne + 1023) / 1024, rows), block(256);
    if (pair_scale && ne % 8 == 0 && (((uintptr_t)y | (uintptr_t)dst | (uintptr_t)addend) & 15) == 0 &&
        (n_used == 8 || n_used == 4 || n_used == 6 || n_used == 2)) {
        const dim3 g8((ne + 2047) / 2048, rows);
#define INFR_H8(KK)                                                                                                       \
    INFR_LAUNCH(unbucket_combine_h8_kernel<KK>, g8, block, 0, s, (const _Float16*)y, slot_pair, weights, ne, weight_before, \
                dst, identity, pair_scale, addend, skip_zero_w, shared)
        if (n_used == 8) INFR_H8(8);
        else if (n_used == 6) INFR_H8(6);
        else if (n_used == 4) INFR_H8(4);
        else INFR_H8(2);
#undef INFR_H8
        return;
    }
    if (!pair_scale && ne % 4 == 0 && (((uintptr_t)y | (uintptr_t)dst | (uintptr_t)addend) & 15) == 0 && part_stride % 4 == 0 &&
        (n_used == 8 || n_used == 4 || n_used == 6 || n_used == 2)) {
        const dim3 g4((ne + 255) / 256, rows);
#define INFR_F4(KK)                                                                                                       \
    INFR_LAUNCH(unbucket_combine_f4_kernel<KK>, g4, dim3(64), 0, s, (const float*)y, slot_pair, weights, ne, weight_before, dst,  \
                identity, addend, skip_zero_w, parts, part_stride)
        if (n_used == 8) INFR_F4(8);
        else if (n_used == 6) INFR_F4(6);
        else if (n_used == 4) INFR_F4(4);
        else INFR_F4(2);
#undef INFR_F4
        return;
    }
    if (pair_scale)
        INFR_LAUNCH(unbucket_combine_kernel<_Float16>, grid, block, 0, s, (const _Float16*)y, slot_pair, weights, ne, n_used,
                    weight_before, dst, identity, pair_scale, addend, skip_zero_w, shared, 1, (size_t)0);
    else
        INFR_LAUNCH(unbucket_combine_kernel<float>, grid, block, 0, s, (const float*)y, slot_pair, weights, ne, n_used,
                    weight_before, dst, identity, pair_scale, addend, skip_zero_w, shared, parts, part_stride);
}

}  // namespace infr