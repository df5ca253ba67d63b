// A stable radix sort of up to RS_SINGLE keys inside one workgroup, for kernels that sort and
// go on with the result.
#pragma once
#include "pgx_internal.h"

namespace pgx {

constexpr int RS_BINS = 256;

__device__ __forceinline__ uint32_t rs_digit(uint64_t k, int shift, int dbits) {
    return (uint32_t)(k >> shift) & ((1u << dbits) - 1u);
}

// rank of the lane's element among the wave's elements of the same digit so far; bumps the
// wave's count of the digit (counts: this wave's counters in LDS, one per digit value)
__device__ __forceinline__ int32_t rs_rank(uint32_t d, bool ok, int dbits, uint64_t lt, int32_t* counts) {
    uint64_t same = __ballot(ok);
    for (int b = 0; b < dbits; ++b) {
        const uint64_t bal = __ballot((d >> b) & 1u);
        same &= ((d >> b) & 1u) ? bal : ~bal;
    }
    const int32_t prior = counts[d];
    if (ok && (same & lt) == 0ull) counts[d] = prior + (int32_t)__popcll(same);
    return prior + (int32_t)__popcll(same & lt);
}

// Each pass is ranked and placed as k_rs_scatter places a single tile (no other tile's
// counts). A pass is a chain (rank, scan, place) that costs the more the more keys a wave
// ranks one after the other, so the keys go to as many waves as there are: each takes an
// equal run of whole 64s. 500 keys: 17 us with four waves of 16 items each, 5 us with this.
constexpr int RS_SINGLE_THREADS = 1024, RS_SINGLE_WAVES = RS_SINGLE_THREADS / WAVE;
constexpr int RS_SINGLE_ITEMS = 8;
constexpr int RS_SINGLE = RS_SINGLE_THREADS * RS_SINGLE_ITEMS;
constexpr int NP_ORDER_SMALL = RS_SINGLE;   // pairs that np_run puts in order itself
struct RsBlock {
    uint64_t sk[RS_SINGLE];
    int32_t sv[RS_SINGLE];
    int32_t waveCnt[RS_SINGLE_WAVES][RS_BINS];
    int32_t off[RS_BINS], wsum[RS_BINS / WAVE];
};
// a thread's elements, and the places a pass gives them
struct RsItems {
    uint64_t key[RS_SINGLE_ITEMS];
    int32_t val[RS_SINGLE_ITEMS], pos[RS_SINGLE_ITEMS];
};
// the threads to launch with, and the items of each
inline int rs_threads(int n) { return std::min(RS_SINGLE_THREADS, div_up(std::max(n, 1), RS_BINS) * RS_BINS); }
inline int rs_item_count(int n) { return div_up(std::max(n, 1), rs_threads(n)); }
// where the thread's item k is: the wave's run, 64 at a time
__device__ __forceinline__ int rs_index(int items, int k) {
    return (int)threadIdx.x / WAVE * WAVE * items + k * WAVE + ((int)threadIdx.x & (WAVE - 1));
}
// The places of the elements ordered by one digit. Every thread of the workgroup calls it;
// the counters it leaves are read by no one else before its first barrier.
__device__ __forceinline__ void rs_block_pass(RsBlock& B, RsItems& x, int n, int shift, int dbits, int items) {
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE, waves = blockDim.x / WAVE;
    const uint64_t lt = (1ull << lane) - 1ull;
    for (int d = lane; d < RS_BINS; d += WAVE) B.waveCnt[wv][d] = 0;   // the wave's own counters
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        if (k >= items) break;
        const bool have = rs_index(items, k) < n;
        x.pos[k] = rs_rank(have ? rs_digit(x.key[k], shift, dbits) : 0u, have, dbits, lt, B.waveCnt[wv]);
    }
    __syncthreads();
    // digit tid: the waves' counts to exclusive prefixes across waves, and the digit's
    // offset, the exclusive scan of the totals over the digits
    int32_t total = 0, sum = 0;
    if (tid < RS_BINS) {
#pragma unroll 4
        for (int w = 0; w < waves; ++w) {
            const int32_t c = B.waveCnt[w][tid];
            B.waveCnt[w][tid] = total;
            total += c;
        }
        sum = total;
        for (int o = 1; o < WAVE; o <<= 1) {
            const int32_t y = __shfl_up(sum, o);
            if (lane >= o) sum += y;
        }
        if (lane == WAVE - 1) B.wsum[wv] = sum;
    }
    __syncthreads();
    if (tid < RS_BINS) {
        int32_t before = 0;
        for (int w = 0; w < RS_BINS / WAVE; ++w) before += w < wv ? B.wsum[w] : 0;
        B.off[tid] = before + sum - total;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        if (k >= items) break;
        if (rs_index(items, k) >= n) continue;
        const uint32_t d = rs_digit(x.key[k], shift, dbits);
        x.pos[k] += B.off[d] + B.waveCnt[wv][d];
    }
}
// the elements to their places, and each thread's new ones back
__device__ __forceinline__ void rs_block_exchange(RsBlock& B, RsItems& x, int n, int items) {
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        if (k >= items) break;
        if (rs_index(items, k) >= n) continue;
        B.sk[x.pos[k]] = x.key[k];
        B.sv[x.pos[k]] = x.val[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RS_SINGLE_ITEMS; ++k) {
        if (k >= items) break;
        const int i = rs_index(items, k);
        if (i >= n) continue;
        x.key[k] = B.sk[i];
        x.val[k] = B.sv[i];
    }
}
// the elements ordered by their low bits, all digits but the last exchanged: x.pos is where
// each belongs
__device__ __forceinline__ void rs_block_sort(RsBlock& B, RsItems& x, int n, int bits, int items) {
    const int passes = (bits + 7) / 8;
    for (int p = 0; p < passes; ++p) {
        rs_block_pass(B, x, n, 8 * p, min(8, bits - 8 * p), items);
        if (p + 1 < passes) rs_block_exchange(B, x, n, items);
    }
}

}  // namespace pgx
