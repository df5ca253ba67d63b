// Contact setup, graph colouring and the TGS soft-step substep loop.
//
// Reference semantics (src/Physecs.cpp, src/ContactConstraints.cpp):
//   contact setup (material mix, body indices, body-local anchors, restitution target
//   with the (pair, triangle) cache matched within 0.1 m)      Physecs.cpp:215-315
//   update contact rows each substep                           Physecs.cpp:368-426
//   integrate velocities (gravity, implicit gyroscopic term)   Physecs.cpp:443-468
//   preSolve / solve (normal + one friction row per point)     ContactConstraints.cpp:4-124
//   integrate positions (COM pivot, pseudo velocities)         Physecs.cpp:494-511
//   relaxation (hard contacts, no bias) and write-back         Physecs.cpp:515-530
//
// The reference solves contact constraints sequentially in push order. Here the
// manifolds are graph-coloured on the device so that no two manifolds of one colour share
// a dynamic body; each colour is one kernel launch and is solved fully in parallel with
// the same result as a sequential pass over it in any order. The solve order is
// "colour 0, colour 1, ..." and is exported (pgx_world_get_manifolds) so that a
// sequential solver fed this order reproduces the device result bit for bit.
#include <hip/hip_cooperative_groups.h>
#include <hip/hip_ext.h>
#include "pgx_internal.h"
#include "radix_block.h"

namespace cg = cooperative_groups;

namespace pgx {

// ------------------------------------------------------------------ compaction
// manifolds of pair p: one for a pair with points, meshCount[p] for a triangle-mesh pair
__global__ void k_flag_manifolds(int nPairs, const int32_t* __restrict__ npNum, const int32_t* __restrict__ meshCount,
                                 int32_t* __restrict__ flag, const int32_t* __restrict__ flowErr,
                                 int32_t* __restrict__ counters) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p == 0) counters[3] = *flowErr;
    if (p < nPairs) flag[p] = (npNum[p] > 0 ? 1 : 0) + meshCount[p];
}

__device__ __forceinline__ void pair_colliders(uint64_t key, int localBits, const int32_t* __restrict__ worldColStart,
                                               const int32_t* __restrict__ colOfLocal, int& c0, int& c1, int& wd) {
    uint64_t lmask = (1ull << localBits) - 1;
    wd = (int)(key >> (2 * localBits));
    int base = worldColStart[wd];
    c0 = colOfLocal[base + (int)((key >> localBits) & lmask)];
    c1 = colOfLocal[base + (int)(key & lmask)];
}

// Manifold list in pair order; a triangle-mesh pair contributes its manifolds in the order
// collisionTriangleMesh emitted them. mfSrc is the narrowphase data slot (the pair's own
// slot, or pairCap + the mesh manifold's slot), mfTri the triangle index (-1 otherwise).
struct CompactArgs {
    const int32_t *npNum, *meshFirst, *meshCount, *npTri;
    int pairCap, localBits;
    const uint64_t* pkeys;
    const int32_t *worldColStart, *colOfLocal, *cbody, *cflags;
    int32_t* mfPair;
    uint64_t* mfKey;
    int32_t *mfB0, *mfB1, *mfSrc, *mfTri;
};
// pair p's manifolds, the first of them at m
__device__ __forceinline__ void compact_pair(const CompactArgs& a, int p, int m) {
    const int nm = a.meshCount[p];
    const uint64_t key = a.pkeys[p];
    int c0, c1, wd;
    pair_colliders(key, a.localBits, a.worldColStart, a.colOfLocal, c0, c1, wd);
    const int b0 = (a.cflags[c0] & CF_DYNAMIC) ? a.cbody[c0] : -1;
    const int b1 = (a.cflags[c1] & CF_DYNAMIC) ? a.cbody[c1] : -1;
    if (nm == 0) {
        a.mfPair[m] = p; a.mfKey[m] = key; a.mfB0[m] = b0; a.mfB1[m] = b1; a.mfSrc[m] = p; a.mfTri[m] = -1;
        return;
    }
    const int first = a.meshFirst[p];
    for (int j = 0; j < nm; ++j) {
        a.mfPair[m + j] = p; a.mfKey[m + j] = key; a.mfB0[m + j] = b0; a.mfB1[m + j] = b1;
        a.mfSrc[m + j] = a.pairCap + first + j;
        a.mfTri[m + j] = a.npTri[first + j];
    }
}
__global__ void k_compact(int nPairs, CompactArgs a, const int32_t* __restrict__ npIndex) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= nPairs || (a.npNum[p] == 0 && a.meshCount[p] == 0)) return;
    compact_pair(a, p, npIndex[p]);
}

// k_flag_manifolds, the scan and k_compact of at most MANIFOLDS_SMALL pairs in one workgroup,
// the scan in registers: five launches of a microsecond or two of work each. 585 pairs: 16 us
// of kernels before, 3.5 us now; 4,912 pairs 17 us.
constexpr int MANIFOLDS_THREADS = 1024, MANIFOLDS_ITEMS = 8, MANIFOLDS_SMALL = MANIFOLDS_THREADS * MANIFOLDS_ITEMS;
__global__ __launch_bounds__(MANIFOLDS_THREADS) void k_manifolds_small(int nPairs, int items, CompactArgs a,
                                                                       int32_t* __restrict__ npIndex,
                                                                       const int32_t* __restrict__ flowErr,
                                                                       int32_t* __restrict__ counters) {
    __shared__ int32_t waveSum[MANIFOLDS_THREADS / WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE, base = threadIdx.x * items;
    int n[MANIFOLDS_ITEMS], sum = 0;
#pragma unroll
    for (int k = 0; k < MANIFOLDS_ITEMS; ++k) {
        const int p = base + k;
        n[k] = k < items && p < nPairs ? (a.npNum[p] > 0 ? 1 : 0) + a.meshCount[p] : 0;
        sum += n[k];
    }
    int x = sum;
    for (int o = 1; o < WAVE; o <<= 1) {
        const int y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == WAVE - 1) waveSum[wv] = x;
    __syncthreads();
    int m = x - sum;
    for (int w = 0; w < wv; ++w) m += waveSum[w];
    if (threadIdx.x == MANIFOLDS_THREADS - 1) {
        counters[1] = m + sum;
        counters[3] = *flowErr;
    }
#pragma unroll
    for (int k = 0; k < MANIFOLDS_ITEMS; ++k) {
        const int p = base + k;
        if (k >= items || p >= nPairs) continue;
        npIndex[p] = m;
        if (n[k]) compact_pair(a, p, m);
        m += n[k];
    }
}

// ------------------------------------------------------------------ colouring
// Jones-Plassmann with largest-priority-first selection and smallest-available colour.
// Priorities are a bijective hash of the manifold's index within its world, so a world's
// colouring does not depend on the other worlds sharing the buffers.
__device__ __forceinline__ uint32_t mix32(uint32_t x) {
    x ^= x >> 16; x *= 0x7feb352du;
    x ^= x >> 15; x *= 0x846ca68bu;
    x ^= x >> 16;
    return x;
}

// The colouring's start in one launch: each world's first manifold, and the colours, body
// claims, colour masks, per-round counts and flags cleared.
__global__ void k_color_begin(int M, int D, int rounds, const uint64_t* __restrict__ mfKey, int worldShift,
                              int32_t* __restrict__ wstart, int32_t* __restrict__ color,
                              uint64_t* __restrict__ claim, uint64_t* __restrict__ claim2, uint64_t* __restrict__ used,
                              int32_t* __restrict__ uncol, int32_t* __restrict__ overflow, int32_t* __restrict__ flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) {
        const int wd = (int)(mfKey[i] >> worldShift);
        if (i == 0 || (int)(mfKey[i - 1] >> worldShift) != wd) wstart[wd] = i;
        color[i] = -1;
    }
    if (i < D) { claim[i] = 0ull; claim2[i] = 0ull; }
    if (i < 2 * D) used[i] = 0ull;
    if (i < rounds) uncol[i] = 0;
    if (i == 0) { *overflow = 0; *flag = 0; }
}

__global__ void k_color_claim(int M, int round, const uint64_t* __restrict__ mfKey, int worldShift,
                              const int32_t* __restrict__ wstart, const int32_t* __restrict__ color,
                              const int32_t* __restrict__ b0, const int32_t* __restrict__ b1,
                              unsigned long long* __restrict__ claim) {
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M || color[m] >= 0) return;
    int wd = (int)(mfKey[m] >> worldShift);
    unsigned long long v = ((unsigned long long)round << 32) | mix32((uint32_t)(m - wstart[wd]));
    int a = b0[m], b = b1[m];
    if (a >= 0) atomicMax(&claim[a], v);
    if (b >= 0) atomicMax(&claim[b], v);
}

// One Jones-Plassmann round r: a manifold whose round-r claim (priority tagged with r)
// holds on both its dynamic bodies takes the smallest colour free on both; every other
// uncoloured manifold claims its bodies for round r+1 in the other claim buffer and is
// marked in uncol[r]. Rounds after the last one that left manifolds uncoloured exit at
// once, so a batch of rounds can be queued without asking the host in between.
__global__ void k_color_round(int M, int round, const uint64_t* __restrict__ mfKey, int worldShift,
                              const int32_t* __restrict__ wstart, int32_t* __restrict__ color,
                              const int32_t* __restrict__ b0, const int32_t* __restrict__ b1,
                              const unsigned long long* __restrict__ claimIn, unsigned long long* __restrict__ claimOut,
                              uint64_t* __restrict__ used, int32_t* __restrict__ uncol, int32_t* __restrict__ counters) {
    if (round > 1 && uncol[round - 1] == 0) return;
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M || color[m] >= 0) return;
    int wd = (int)(mfKey[m] >> worldShift);
    uint32_t prio = mix32((uint32_t)(m - wstart[wd]));
    unsigned long long v = ((unsigned long long)round << 32) | prio;
    int a = b0[m], b = b1[m];
    bool won = (a < 0 || claimIn[a] == v) && (b < 0 || claimIn[b] == v);
    if (!won) {
        unsigned long long vn = ((unsigned long long)(round + 1) << 32) | prio;
        if (a >= 0) atomicMax(&claimOut[a], vn);
        if (b >= 0) atomicMax(&claimOut[b], vn);
        uncol[round] = 1;   // any writer writes 1: no atomic needed
        return;
    }
    uint64_t lo = 0, hi = 0;
    if (a >= 0) { lo |= used[2 * a]; hi |= used[2 * a + 1]; }
    if (b >= 0) { lo |= used[2 * b]; hi |= used[2 * b + 1]; }
    int c;
    if (~lo) c = __ffsll((long long)~lo) - 1;
    else if (~hi) c = 64 + __ffsll((long long)~hi) - 1;
    else { c = 127; atomicAdd(&counters[5], 1); }   // overflow: reported as an error by the host
    color[m] = c;
    uint64_t bl = c < 64 ? (1ull << c) : 0ull, bh = c >= 64 ? (1ull << (c - 64)) : 0ull;
    if (a >= 0) { used[2 * a] |= bl; used[2 * a + 1] |= bh; }
    if (b >= 0) { used[2 * b] |= bl; used[2 * b + 1] |= bh; }
}

// The previous step's colour of each manifold that persists (same pair key and triangle,
// found in the previous step's contact cache as k_setup finds it), and its bodies' used
// colours. Persisting manifolds were coloured properly among themselves last step, so
// their colours stay valid unless a body changed from kinematic to dynamic in between: a
// colour set twice on one body raises the clash flag, and k_color_clash then drops every
// inherited colour (the step colours from scratch). Only new manifolds go through the
// claim rounds.
constexpr int CACHE_NUM_MASK = 255, CACHE_COLOR_SHIFT = 8, CACHE_HAS_COLOR = 0x8000;
// the manifold's place in the previous step's cache, or -1
__device__ __forceinline__ int cached_manifold(uint64_t key, int tri, const uint64_t* __restrict__ prevKey,
                                               const int32_t* __restrict__ prevTri, int prevCount) {
    // the cache is in manifold order, so a pair's manifolds are one run of equal keys
    int lo = 0, hi = prevCount;
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (prevKey[mid] < key) lo = mid + 1; else hi = mid;
    }
    for (; lo < prevCount && prevKey[lo] == key; ++lo)
        if (prevTri[lo] == tri) return lo;
    return -1;
}
__global__ void k_color_inherit(int M, const uint64_t* __restrict__ mfKey, const int32_t* __restrict__ mfTri,
                                const uint64_t* __restrict__ prevKey, const int32_t* __restrict__ prevTri,
                                const int32_t* __restrict__ prevNum, int prevCount, const int32_t* __restrict__ b0,
                                const int32_t* __restrict__ b1, int32_t* __restrict__ color,
                                int32_t* __restrict__ mfPrev, unsigned long long* __restrict__ used,
                                int32_t* __restrict__ clash) {
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    const uint64_t key = mfKey[m];
    const int tri = mfTri[m];
    const int prev = cached_manifold(key, tri, prevKey, prevTri, prevCount);
    mfPrev[m] = prev;
    int c = -1;
    if (prev >= 0) {
        const int pn = prevNum[prev];
        if (pn & CACHE_HAS_COLOR) c = (pn >> CACHE_COLOR_SHIFT) & 127;
    }
    color[m] = c;
    if (c < 0) return;
    const unsigned long long bit = 1ull << (c & 63);
    const int word = c >> 6;
    const int a = b0[m], b = b1[m];
    bool twice = false;
    if (a >= 0) twice |= (atomicOr(&used[2 * a + word], bit) & bit) != 0;
    if (b >= 0) twice |= (atomicOr(&used[2 * b + word], bit) & bit) != 0;
    if (twice) *clash = 1;
}

__global__ void k_color_clash(int M, int D, const int32_t* __restrict__ clash, int32_t* __restrict__ color,
                              uint64_t* __restrict__ used) {
    if (!*clash) return;
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < M) color[i] = -1;
    if (i < 2 * D) used[i] = 0;
}

// Solve order: by colour, and within a colour by point count (byPoints), so the lanes of a
// wave solve manifolds of one point count and run the same number of rows. A colour's
// manifolds share no dynamic body, so their order within the colour changes no result. The
// per-world passes keep each world's manifolds of a colour together instead (byPoints 0).
constexpr int COLOR_KEY_SHIFT = 2;
__global__ void k_color_keys(int M, const int32_t* __restrict__ color, const int32_t* __restrict__ npNum,
                             const int32_t* __restrict__ mfSrc, int byPoints, uint64_t* __restrict__ keys,
                             int32_t* __restrict__ vals) {
    int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    const int num = byPoints ? min(max(npNum[mfSrc[m]], 1), 4) : 1;
    keys[m] = ((uint64_t)color[m] << COLOR_KEY_SHIFT) | (uint64_t)(num - 1);
    vals[m] = m;
}

// start[c] = the first solve position with colour >= c, for every c in [0, n): colours with
// no manifold (inherited colours leave gaps) get empty ranges
// One workgroup. Also packs what the host reads back after the colouring rounds into one
// block, so a single copy brings it: [0, n) the starts, [n] the colour-overflow flag,
// [n+1, n+2] the last manifold's key (low, high word), [n+3, n+3+rounds] the count of
// uncoloured manifolds after each round.
__global__ void k_color_start(int M, int n, const uint64_t* __restrict__ keys, int32_t* __restrict__ start,
                              int rounds, const int32_t* __restrict__ uncol, const int32_t* __restrict__ overflow,
                              int32_t* __restrict__ pack) {
    for (int c = threadIdx.x; c < n; c += blockDim.x) {
        int lo = 0, hi = M;
        while (lo < hi) {
            int mid = (lo + hi) >> 1;
            if (keys[mid] < ((uint64_t)c << COLOR_KEY_SHIFT)) lo = mid + 1; else hi = mid;
        }
        start[c] = lo;
        pack[c] = lo;
    }
    for (int r = threadIdx.x; r <= rounds; r += blockDim.x) pack[n + 3 + r] = uncol[r];
    if (threadIdx.x == 0) {
        pack[n] = *overflow;
        const uint64_t last = M > 0 ? keys[M - 1] : 0ull;
        pack[n + 1] = (int32_t)(uint32_t)last;
        pack[n + 2] = (int32_t)(uint32_t)(last >> 32);
    }
}

// The whole colouring of a small scene in one workgroup: k_color_begin, k_color_inherit,
// k_color_clash, k_color_claim, as many k_color_rounds as are needed, the stable sort into
// solve order (k_color_keys and the radix sort, here one counting pass over colour and point
// count), k_color_start and k_color_rank, with the same colours and the same order. The
// bodies' claims and colour masks are in LDS; one claim buffer does, as a round's losers
// claim again only after a barrier. Each of those kernels is a microsecond or two of work
// behind a launch of five, and the host waits for the last: 415 manifolds took thirteen
// launches, 35 us of kernels and about 5 us of launch each, and take one of 11 us now (3,543
// manifolds 37 us). The limit is what fits a
// workgroup's registers and LDS; larger colourings have work for more than one workgroup.
constexpr int COLOR_THREADS = 1024, COLOR_WAVES = COLOR_THREADS / WAVE, COLOR_ITEMS = 4;
constexpr int COLOR_SMALL = COLOR_THREADS * COLOR_ITEMS;
constexpr int COLOR_BINS = 128 << COLOR_KEY_SHIFT, COLOR_STARTS = 130;
__global__ __launch_bounds__(COLOR_THREADS) void k_color_small(
    int M, int D, int items, int maxRounds, const uint64_t* __restrict__ mfKey, int worldShift, int32_t* __restrict__ wstart,
    const int32_t* __restrict__ mfTri, const uint64_t* __restrict__ prevKey, const int32_t* __restrict__ prevTri,
    const int32_t* __restrict__ prevNum, int prevCount, const int32_t* __restrict__ b0, const int32_t* __restrict__ b1,
    const int32_t* __restrict__ npNum, const int32_t* __restrict__ mfSrc, int byPoints, int32_t* __restrict__ mfColor,
    int32_t* __restrict__ mfPrev, uint64_t* __restrict__ usedOut, int32_t* __restrict__ perm, int32_t* __restrict__ rank,
    int32_t* __restrict__ start, int32_t* __restrict__ pack) {
    extern __shared__ unsigned long long bodies[];
    unsigned long long *used = bodies, *claim = bodies + 2 * D;
    __shared__ int32_t waveCnt[COLOR_WAVES][COLOR_BINS];
    __shared__ int32_t off[COLOR_BINS], wsum[COLOR_BINS / WAVE];
    __shared__ int32_t clash, overflow, lastBin;
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wv = tid / WAVE;
    const int run = wv * WAVE * items + lane;   // the wave's manifolds: run + 64 k, in manifold order
    for (int i = tid; i < 3 * D; i += COLOR_THREADS) bodies[i] = 0ull;
    if (tid == 0) { clash = 0; overflow = 0; }
    int color[COLOR_ITEMS], ba[COLOR_ITEMS], bb[COLOR_ITEMS], world[COLOR_ITEMS];
#pragma unroll
    for (int k = 0; k < COLOR_ITEMS; ++k) {
        color[k] = 0;   // no manifold: nothing to colour
        const int m = run + k * WAVE;
        if (k >= items || m >= M) continue;
        const uint64_t key = mfKey[m];
        world[k] = (int)(key >> worldShift);
        if (m == 0 || (int)(mfKey[m - 1] >> worldShift) != world[k]) wstart[world[k]] = m;
        ba[k] = b0[m];
        bb[k] = b1[m];
        const int prev = cached_manifold(key, mfTri[m], prevKey, prevTri, prevCount);
        mfPrev[m] = prev;
        color[k] = -1;
        if (prev >= 0) {
            const int pn = prevNum[prev];
            if (pn & CACHE_HAS_COLOR) color[k] = (pn >> CACHE_COLOR_SHIFT) & 127;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < COLOR_ITEMS; ++k) {
        if (k >= items || run + k * WAVE >= M || color[k] < 0) continue;
        const unsigned long long bit = 1ull << (color[k] & 63);
        const int word = color[k] >> 6;
        bool twice = false;
        if (ba[k] >= 0) twice |= (atomicOr(&used[2 * ba[k] + word], bit) & bit) != 0;
        if (bb[k] >= 0) twice |= (atomicOr(&used[2 * bb[k] + word], bit) & bit) != 0;
        if (twice) clash = 1;
    }
    __syncthreads();
    if (clash) {
        for (int i = tid; i < 2 * D; i += COLOR_THREADS) used[i] = 0ull;
        for (int k = 0; k < COLOR_ITEMS; ++k)
            if (k < items && run + k * WAVE < M) color[k] = -1;
    }
    uint32_t prio[COLOR_ITEMS];
    auto claims = [&](int k, int round) {
        const unsigned long long v = ((unsigned long long)round << 32) | prio[k];
        if (ba[k] >= 0) atomicMax(&claim[ba[k]], v);
        if (bb[k] >= 0) atomicMax(&claim[bb[k]], v);
    };
#pragma unroll
    for (int k = 0; k < COLOR_ITEMS; ++k) {
        prio[k] = 0;
        if (color[k] >= 0) continue;
        prio[k] = mix32((uint32_t)(run + k * WAVE - wstart[world[k]]));
        claims(k, 1);
    }
    int rounds = 0;
    for (int round = 1; round <= maxRounds; ++round) {
        __syncthreads();
        bool lost = false;
#pragma unroll
        for (int k = 0; k < COLOR_ITEMS; ++k) {
            if (color[k] >= 0) continue;
            const unsigned long long v = ((unsigned long long)round << 32) | prio[k];
            const int a = ba[k], b = bb[k];
            if ((a >= 0 && claim[a] != v) || (b >= 0 && claim[b] != v)) { lost = true; continue; }
            uint64_t lo = 0, hi = 0;
            if (a >= 0) { lo |= used[2 * a]; hi |= used[2 * a + 1]; }
            if (b >= 0) { lo |= used[2 * b]; hi |= used[2 * b + 1]; }
            int c;
            if (~lo) c = __ffsll((long long)~lo) - 1;
            else if (~hi) c = 64 + __ffsll((long long)~hi) - 1;
            else { c = 127; overflow = 1; }   // reported as an error by the host
            color[k] = c;
            const uint64_t bl = c < 64 ? (1ull << c) : 0ull, bh = c >= 64 ? (1ull << (c - 64)) : 0ull;
            if (a >= 0) { used[2 * a] |= bl; used[2 * a + 1] |= bh; }
            if (b >= 0) { used[2 * b] |= bl; used[2 * b + 1] |= bh; }
        }
        if (!__syncthreads_or(lost)) { rounds = round; break; }
#pragma unroll
        for (int k = 0; k < COLOR_ITEMS; ++k)
            if (color[k] < 0) claims(k, round + 1);
    }
    for (int i = tid; i < 2 * D; i += COLOR_THREADS) usedOut[i] = used[i];
    // solve order, as k_rs_single ranks and places one digit
    const uint64_t lt = (1ull << lane) - 1ull;
    for (int d = lane; d < COLOR_BINS; d += WAVE) waveCnt[wv][d] = 0;
    uint32_t bin[COLOR_ITEMS];
    int32_t place[COLOR_ITEMS];
#pragma unroll
    for (int k = 0; k < COLOR_ITEMS; ++k) {
        const int m = run + k * WAVE;
        const bool have = k < items && m < M;
        bin[k] = 0;
        if (have) {
            mfColor[m] = color[k];
            const int num = byPoints ? min(max(npNum[mfSrc[m]], 1), 4) : 1;
            bin[k] = (uint32_t)(max(color[k], 0) << COLOR_KEY_SHIFT | (num - 1));
        }
        if (k < items) place[k] = rs_rank(bin[k], have, 7 + COLOR_KEY_SHIFT, lt, waveCnt[wv]);
    }
    __syncthreads();
    int32_t total = 0, x = 0;
    if (tid < COLOR_BINS) {
#pragma unroll
        for (int w = 0; w < COLOR_WAVES; ++w) {
            const int32_t c = waveCnt[w][tid];
            waveCnt[w][tid] = total;
            total += c;
        }
        x = total;
        for (int o = 1; o < WAVE; o <<= 1) {
            const int32_t y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == WAVE - 1) wsum[wv] = x;
    }
    __syncthreads();
    if (tid < COLOR_BINS) {
        int32_t before = 0;
        for (int w = 0; w < COLOR_BINS / WAVE; ++w) before += w < wv ? wsum[w] : 0;
        off[tid] = before + x - total;
        if (total > 0 && before + x == M) lastBin = tid;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < COLOR_ITEMS; ++k) {
        const int m = run + k * WAVE;
        if (k >= items || m >= M) continue;
        const int pos = off[bin[k]] + waveCnt[wv][bin[k]] + place[k];
        perm[pos] = m;
        rank[m] = pos;
    }
    if (tid < COLOR_STARTS) {
        const int at = tid < 128 ? off[tid << COLOR_KEY_SHIFT] : M;
        start[tid] = at;
        pack[tid] = at;
    }
    if (tid == 0) {   // after the starts: the overflow flag, the colours, the rounds (0: too many)
        pack[COLOR_STARTS] = overflow;
        pack[COLOR_STARTS + 1] = (lastBin >> COLOR_KEY_SHIFT) + 1;
        pack[COLOR_STARTS + 2] = rounds;
    }
}

// ------------------------------------------------------------------ setup (solve order)

// each manifold's slot in solve order (the inverse of the colour sort's permutation)
__global__ void k_color_rank(int M, const int32_t* __restrict__ perm, int32_t* __restrict__ rank) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < M) rank[perm[s]] = s;
}

// One thread per manifold in manifold order, so its reads of the manifold arrays are
// coalesced; the solve-order arrays it writes are scattered instead (stores do not stall).
__global__ __launch_bounds__(256) void k_setup(
    int M, int Mcap, const int32_t* __restrict__ rank, const int32_t* __restrict__ mfSrc,
    const int32_t* __restrict__ mfTri, const uint64_t* __restrict__ mfKey, int localBits, const int32_t* __restrict__ worldColStart,
    const int32_t* __restrict__ colOfLocal, const int32_t* __restrict__ cbody, const int32_t* __restrict__ cflags,
    const float4* __restrict__ cmat, const int32_t* __restrict__ npNum, const float4* __restrict__ npNormal,
    const float4* __restrict__ npPts, const int32_t* __restrict__ mfColor, const int32_t* __restrict__ mfB0,
    const int32_t* __restrict__ mfB1, const float4* __restrict__ bpos, const float4* __restrict__ bquat,
    const float4* __restrict__ dvel, const float4* __restrict__ dang, const float4* __restrict__ dcom, int D,
    const int32_t* __restrict__ mfPrev, const int32_t* __restrict__ prevNum,
    const float4* __restrict__ prevLp, int prevCap, uint64_t* __restrict__ curKey,
    int32_t* __restrict__ curTri, int32_t* __restrict__ curNum,
    float4* __restrict__ curLp, int2* __restrict__ sB, int2* __restrict__ sA, int32_t* __restrict__ sFlags,
    int32_t* __restrict__ sCanon, float4* __restrict__ sN, float2* __restrict__ sSoft, float4* __restrict__ sR,
    int32_t* __restrict__ sWorld) {
    const int m = blockIdx.x * blockDim.x + threadIdx.x;
    if (m >= M) return;
    const int s = rank[m];
    int p = mfSrc[m];
    int tri = mfTri[m];
    uint64_t key = mfKey[m];
    int c0, c1, wd;
    pair_colliders(key, localBits, worldColStart, colOfLocal, c0, c1, wd);
    sWorld[s] = wd;
    int a0 = cbody[c0], a1 = cbody[c1];
    int b0 = mfB0[m], b1 = mfB1[m];
    float4 m0 = cmat[c0], m1 = cmat[c1];   // friction, restitution, damping
    float friction = (m0.x + m1.x) * 0.5f;
    bool soft;
    float freq, damp, rest;
    if (m0.z != 0.f || m1.z != 0.f) {
        soft = true;
        if (m0.z != 0.f && m1.z != 0.f) { freq = gmin(m0.y, m1.y); damp = gmin(m0.z, m1.z); }
        else if (m0.z != 0.f) { freq = m0.y; damp = m0.z; }
        else { freq = m1.y; damp = m1.z; }
        rest = 0.f;
    } else {
        soft = false; freq = 0.f; damp = 0.f;
        rest = (m0.y + m1.y) * 0.5f;
    }
    f3 n = xyz(npNormal[p]);
    int num = npNum[p];
    qf q0 = q4(bquat[a0]), q1 = q4(bquat[a1]);
    f3 com0 = s3(0.f), v0 = s3(0.f), w0 = s3(0.f), com1 = s3(0.f), v1 = s3(0.f), w1 = s3(0.f);
    if (b0 >= 0) { com0 = add(xyz(bpos[a0]), qrot(q0, xyz(dcom[b0]))); v0 = xyz(dvel[b0]); w0 = xyz(dang[b0]); }
    if (b1 >= 0) { com1 = add(xyz(bpos[a1]), qrot(q1, xyz(dcom[b1]))); v1 = xyz(dvel[b1]); w1 = xyz(dang[b1]); }
    // previous step's manifold of this (pair, triangle), src/Physecs.cpp:237, as
    // k_color_inherit found it
    const int prev = mfPrev[m];
    qf iq0 = qinverse(q0), iq1 = qinverse(q1);
    for (int k = 0; k < 4; ++k) {
        float4 r0o = make_float4(0.f, 0.f, 0.f, 0.f), r1o = r0o;
        if (k < num) {
            f3 p0 = xyz(npPts[8 * (size_t)p + 2 * k]), p1 = xyz(npPts[8 * (size_t)p + 2 * k + 1]);
            f3 r0 = sub(p0, com0), r1 = sub(p1, com1);
            f3 rel = sub(sub(add(v1, cross(w1, r1)), v0), cross(w0, r0));
            float relN = dot(rel, n);
            r0 = qrot(iq0, r0);
            r1 = qrot(iq1, r1);
            float tv = 0.f;
            bool found = false;
            if (prev >= 0) {
                int pn = prevNum[prev] & CACHE_NUM_MASK;
                for (int i = 0; i < pn; ++i) {
                    float4 lp = prevLp[(size_t)i * prevCap + prev];
                    f3 d = sub(xyz(lp), r0);
                    // glm::distance(...) < 0.1 is a double comparison (Physecs.cpp:294)
                    if ((double)sqrtf(dot(d, d)) < 0.1) { found = true; tv = lp.w; break; }
                }
            }
            if (!found) tv = -rest * relN;
            r0o = f4(r0, tv);
            r1o = f4(r1, tv);   // each side's lane carries the target velocity into its row
            curLp[(size_t)k * Mcap + m] = r0o;
        }
        sR[2 * ((size_t)k * Mcap + s)] = r0o;
        sR[2 * ((size_t)k * Mcap + s) + 1] = r1o;
    }
    curKey[m] = key;
    curTri[m] = tri;
    curNum[m] = num | (mfColor[m] << CACHE_COLOR_SHIFT) | CACHE_HAS_COLOR;
    sB[s] = make_int2(b0, b1);
    sA[s] = make_int2(a0, a1);
    sFlags[s] = num | (soft ? 256 : 0) | (mfColor[m] << 16);
    sCanon[s] = m;
    sN[s] = f4(n, friction);
    sSoft[s] = make_float2(freq, damp);
}

// contact points per colour (statistics). The manifolds are in colour order, so each
// thread sums a run of POINTS_RUN consecutive manifolds and adds to its block's per-colour
// counters in LDS when the colour changes; each block then adds its non-zero counters to
// the output, which starts at zero.
constexpr int POINTS_RUN = 16;
__global__ __launch_bounds__(256) void k_color_points(int M, const int32_t* __restrict__ sFlags,
                                                      int32_t* __restrict__ out) {
    __shared__ int32_t cnt[128];
    if (threadIdx.x < 128) cnt[threadIdx.x] = 0;
    __syncthreads();
    const int first = (blockIdx.x * blockDim.x + threadIdx.x) * POINTS_RUN;
    int colour = -1, sum = 0;
    for (int i = first; i < min(M, first + POINTS_RUN); ++i) {
        const int f = sFlags[i], c = (f >> 16) & 127;
        if (c != colour) {
            if (sum) atomicAdd(&cnt[colour], sum);
            colour = c;
            sum = 0;
        }
        sum += f & 255;
    }
    if (sum) atomicAdd(&cnt[colour], sum);
    __syncthreads();
    if (threadIdx.x < 128 && cnt[threadIdx.x]) atomicAdd(&out[threadIdx.x], cnt[threadIdx.x]);
}

void sv_color_points(World& w, int nColors) {
    if (nColors <= 0) return;
    const int M = w.colorStartHost.back();
    fill_i32(w.stream, w.colorPoints.p, 0, 160);
    hipLaunchKernelGGL(k_color_points, dim3(std::max(1, div_up(M, 256 * POINTS_RUN))), dim3(256), 0, w.stream, M,
                       w.sFlags.p, w.colorPoints.p);
    PGX_LAUNCH_CHECK();
}

// ------------------------------------------------------------------ substep pieces
// Every contact kernel gives a manifold to two adjacent lanes, one per body: lane i works
// on side i & 1 of manifold slot i >> 1. A side's lane loads its own body and its own rows,
// computes its half of each relative velocity and updates its own body; the halves meet
// through DPP lane moves. A launch of one colour of the 32k scene holds about a wave per
// ten SIMDs, so its time is one wave's chain of instructions: k_solve is 718 of them instead
// of 1,076 with a lane per manifold, at 98 registers instead of 208, and took 4.26 us per
// colour launch of the settled 32k scene instead of 5.63 (a run of small colours in
// k_solve_batch 17.1 us instead of 24.8 (before its two teams); a large colour of 1,024 worlds 8.4 instead of 10.4).
//
// Contact rows of point k of side lane i, field f at ((k * RS_NF + f) * Mcap) * 2 + i, so
// a wave's loads are contiguous: r x n (.w = target velocity), the row times the body's
// world inverse inertia, as preSolve keeps it (src/ContactConstraints.cpp:21-24; .w = the
// effective mass 1 / invN, or invN + gamma / h of a soft contact), and I * (r x t) (.w =
// the bias 0.1 c / h, or beta c / h of a soft contact). Side 0's vectors are stored
// negated: both sides then add to the relative velocity and subtract the impulse, and
// negation changes no other bit of a product or a sum's magnitude. Per point also the
// tangent (.w = the friction impulse of one pass). The friction row reads the component
// velocities (src/ContactConstraints.cpp:92-101), which no pass changes, so its impulse
// rv / invT is fixed for the substep like the terms of src/ContactConstraints.cpp:54-68:
// all are computed here, once, with the operations and in the order of the solve. 7 float4
// per point instead of 9, and the solve reads no component velocity.
enum { RS_N = 0, RS_NT, RS_TT, RS_NF };
static_assert(2 * RS_NF + 1 == CONTACT_ROW_FIELDS, "sRow holds CONTACT_ROW_FIELDS float4 per point");
#define ROW(f, k) a.sRow[((size_t)((k) * RS_NF + (f)) * a.Mcap) * 2 + i]
#define ROWT(k) a.sRow[(size_t)(8 * RS_NF + (k)) * a.Mcap + s]
#define LAM(k) a.sLam[(size_t)(k) * a.Mcap + s]
// sMode: what the solve has to know of a slot this substep: points, softness, and the points
// whose normal or friction row has no mass (invN or invT is 0) and is left out
enum { MODE_NUM = 255, MODE_SOFT = 256, MODE_N = 1 << 16, MODE_T = 1 << 20 };
// a pass over the contacts: with the bias; without the soft contacts (relaxation); the
// substep's first (the lambdas are 0) and last (nothing reads them afterwards)
enum { PASS_BIAS = 1, PASS_SKIP_SOFT = 2, PASS_FIRST = 4, PASS_LAST = 8 };

struct SubArgs {
    int M, Mcap, D, nColors, substeps, iterations;
    float h, g;
    const int32_t *sB, *sA;               // 2 per slot: the sides' dynamic bodies (-1) and internal bodies
    const int32_t *sFlags, *colorStart;
    const float4 *sN, *sR;
    const float2* sSoft;
    float4* sRow;
    float2* sLam;
    int32_t* sMode;
    float4 *bpos, *bquat;                 // body poses (dynamic bodies come first)
    float4 *dvel, *dang;                  // component velocity at the start of the substep (dvel.w = invMass)
    float4* bvel;                         // per dynamic body: solver v (.w = invMass), w (velocityTemp)
    float4* brec;                         // per dynamic body: what its contact rows are built from
    const float4 *dcom, *dinvI;
    float4 *pvel, *pang;                  // pseudo velocities (pang.w = constraint count)
    // dependency-driven passes: per body, the colours of its manifolds (2 x 64 bits); a work
    // ticket per pass; a flag set if a wait ran out (never expected)
    const uint64_t* used;
    int32_t* tickets;
    int32_t* flowErr;
    int32_t* qDone;                       // manifolds finished per queue in this step
    int32_t* barrier;                     // arrivals at the pass kernel's grid barriers (this substep)
    int32_t* xctl;                        // control blocks of the one-XCD pass kernel, one per pass
    int xctlWords;                        // words of xctl cleared by k_prepare
};

// the even (side 0) or the odd (side 1) lane's value in both lanes of a pair
__device__ __forceinline__ float side0(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xA0, 0xf, 0xf, true));   // quad_perm 0,0,2,2
}
__device__ __forceinline__ float side1(float x) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), 0xF5, 0xf, 0xf, true));   // quad_perm 1,1,3,3
}
__device__ __forceinline__ f3 side0(f3 v) { return mk3(side0(v.x), side0(v.y), side0(v.z)); }
__device__ __forceinline__ f3 side1(f3 v) { return mk3(side1(v.x), side1(v.y), side1(v.z)); }
// side 0's half of a relative velocity carries a minus sign
__device__ __forceinline__ f3 signed_of(f3 v, int side) { return side ? v : neg(v); }

__device__ __forceinline__ m3 world_inv_inertia(const SubArgs& a, int b) {
    m3 rot = mat3_cast(q4(a.bquat[b]));
    m3 invI = mk_m3(xyz(a.dinvI[3 * b]), xyz(a.dinvI[3 * b + 1]), xyz(a.dinvI[3 * b + 2]));
    return mulmm(mulmm(rot, invI), transpose(rot));   // rot * invI * invRot, src/Physecs.cpp:467
}

// update contact rows (src/Physecs.cpp:368-426) then preSolve (src/ContactConstraints.cpp:4-31)
// of one side of a manifold. Everything of the body comes from its record (integrate_velocity),
// one 128-byte line per side; gathered from the bodies' six arrays, with the inertia and the
// centre of mass rebuilt per manifold, the kernel was bound by those gathers: 58 us on 295k
// manifolds of 218k bodies instead of 25 (and 10 more for the bodies' records in the write-back).
__device__ void prepare_side(const SubArgs& a, int i) {
    const int s = i >> 1, side = i & 1;
    const int b = a.sB[i], flags = a.sFlags[s], num = flags & 255;
    const f3 n = xyz(a.sN[s]);
    qf q;
    f3 com = s3(0.f), v = s3(0.f), w = s3(0.f), cv = s3(0.f), cw = s3(0.f);
    float im = 0.f;
    m3 I = mzero();
    if (b >= 0) {
        const float4 *r = a.brec + br(b, 0), rc = r[BR_COM], rv = r[BR_V], rw = r[BR_W], i0 = r[BR_I0];
        q = q4(r[BR_Q]);
        com = xyz(rc); im = rc.w;
        v = xyz(rv); w = xyz(rw);
        I = mk_m3(xyz(i0), xyz(r[BR_I1]), xyz(r[BR_I2]));
        cv = add(v, mul(a.h, mk3(0.f, -a.g, 0.f)));   // as integrate_velocity
        cw = mk3(rv.w, rw.w, i0.w);
    } else {
        q = q4(a.bquat[a.sA[i]]);
    }
    const float nn = dot(n, n), imSum = side0(im) + side1(im);
    const bool soft = (flags & 256) != 0;
    const float2 sp = a.sSoft[s];
    const float h = a.h;
    int mode = num | (soft ? MODE_SOFT : 0);
    for (int k = 0; k < num; ++k) {
        const float4 anchor = a.sR[2 * (size_t)k * a.Mcap + i];
        const f3 r = qrot(q, xyz(anchor));
        const f3 cp = add(com, r);
        const float cn = dot(sub(side1(cp), side0(cp)), n);
        const f3 rxn = cross(r, n);
        const f3 wxr = cross(w, r);
        const f3 rel = sub(sub(side1(add(v, wxr)), side0(v)), side0(wxr));
        const float relN = dot(rel, n);
        f3 t = sub(rel, mul(relN, n));
        const float tl = length(t);
        if (tl != 0.f) t = divs(t, tl);
        const f3 rxt = cross(r, t);
        const f3 rxnt = mulmv(I, rxn), rxtt = mulmv(I, rxt);
        const float dn = dot(rxn, rxnt), dt = dot(rxt, rxtt);
        const float invN = nn * imSum + side0(dn) + side1(dn);
        const float invT = dot(t, t) * imSum + side0(dt) + side1(dt);
        // src/ContactConstraints.cpp:54-68 on the substep's fixed values
        const float effMass = 1.f / invN;
        const float bias = 0.1f * cn / h;
        float termA = effMass, termB = bias;
        if (soft) {
            float af = 2.f * 3.14159265358979323846f * sp.x;
            float stiffness = af * af * effMass;
            float damping = 2.f * af * sp.y * effMass;
            float gamma = 1.f / (damping + h * stiffness);
            float beta = h * stiffness / (damping + h * stiffness);
            termA = invN + gamma / h;
            termB = beta * cn / h;
        }
        // the friction impulse of one pass, on the component velocities
        const float ct = dot(signed_of(t, side), cv), cr = dot(signed_of(rxt, side), cw);
        const float rvT = side0(ct + cr) + side1(ct) + side1(cr);
        if (!(invN == 0.f)) mode |= MODE_N << k;
        if (!(invT == 0.f)) mode |= MODE_T << k;
        ROW(RS_N, k) = f4(signed_of(rxn, side), anchor.w);
        ROW(RS_NT, k) = f4(signed_of(rxnt, side), termA);
        ROW(RS_TT, k) = f4(signed_of(rxtt, side), termB);
        if (side == 0) ROWT(k) = f4(t, rvT / invT);
    }
    if (side == 0) a.sMode[s] = mode;
}

// src/MathUtil.h:10-21
__device__ __forceinline__ f3 solve33(const m3& A, f3 b) {
    f3 c12 = cross(A.c1, A.c2);
    float det = dot(A.c0, c12);
    if (det == 0.f) return s3(0.f);
    float id = 1.f / det;
    return mk3(id * dot(b, c12), id * dot(A.c0, cross(b, A.c2)), id * dot(A.c0, cross(A.c1, b)));
}

// integrate velocities of one body, src/Physecs.cpp:443-468, from its component velocities;
// and its record for the substep's contact and joint rows
__device__ void integrate_velocity(const SubArgs& a, int d, float4 vv, f3 ang) {
    const float4 cm = a.dcom[d];
    if (cm.w != 0.f) return;   // kinematic
    const qf q = q4(a.bquat[d]);
    m3 rot = mat3_cast(q);
    m3 invRot = transpose(rot);
    f3 v = add(xyz(vv), mul(a.h, mk3(0.f, -a.g, 0.f)));
    m3 invI = mk_m3(xyz(a.dinvI[3 * d]), xyz(a.dinvI[3 * d + 1]), xyz(a.dinvI[3 * d + 2]));
    f3 wl = mulmv(invRot, ang);
    m3 I = inverse(invI);
    f3 Iw = mulmv(I, wl);
    f3 f = mul(a.h, cross(wl, Iw));
    m3 J = madd(I, mscale(a.h, msub(mulmm(matrixCross3(wl), I), matrixCross3(Iw))));
    wl = sub(wl, solve33(J, f));
    f3 w = mulmv(rot, wl);
    a.bvel[bv(d, BV_V)] = f4(v, vv.w);
    a.bvel[bv(d, BV_W)] = f4(w, 0.f);
    const m3 wI = world_inv_inertia(a, d);   // massTemp of the substep
    float4* r = a.brec + br(d, 0);
    r[BR_COM] = f4(add(xyz(a.bpos[d]), qrot(q, xyz(cm))), vv.w);
    r[BR_Q] = f4q(q);
    r[BR_V] = f4(xyz(vv), w.x);
    r[BR_W] = f4(ang, w.y);
    r[BR_I0] = f4(wI.c0, w.z);
    r[BR_I1] = f4(wI.c1, 0.f);
    r[BR_I2] = f4(wI.c2, 0.f);
    a.pvel[d] = make_float4(0.f, 0.f, 0.f, 0.f);
    a.pang[d] = make_float4(0.f, 0.f, 0.f, 0.f);
}

// Everything one side's solve reads except its body's solver velocities: the manifold's
// mode, normal and friction, and its rows, tangents and lambdas. All
// of it is fixed for the whole pass.
struct SideIn {
    int num, mode, b;
    bool soft;
    float4 n;         // normal, friction
    float4 row[4][RS_NF], t[4];
    float2 lam[4];
};

// EAGER loads point slot 0's rows (every manifold has a first point) with the manifold's
// mode and body index, without waiting for the point count; slots 1-3 wait for the count,
// in the same round of loads as the body's velocities (which wait for the body index
// anyway), so unused slots cost no traffic and the solve still takes two dependent rounds.
// the rest of a side whose mode and body index are known
template <bool EAGER = false>
__device__ __forceinline__ void load_rows(const SubArgs& a, int i, int pass, SideIn& in) {
    const int s = i >> 1;
    in.soft = (in.mode & MODE_SOFT) != 0;
    in.num = in.mode & MODE_NUM;
    in.n = a.sN[s];
    // all rows of the side are loaded before any dependent arithmetic (memory-level
    // parallelism); unused point slots are never read back
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if ((EAGER && k == 0) || k < in.num) {
#pragma unroll
            for (int f = 0; f < RS_NF; ++f) in.row[k][f] = ROW(f, k);
            in.t[k] = ROWT(k);
            in.lam[k] = (pass & PASS_FIRST) ? make_float2(0.f, 0.f) : LAM(k);
        }
    }
}
template <bool EAGER = false>
__device__ __forceinline__ void load_side(const SubArgs& a, int i, int pass, SideIn& in) {
    in.mode = a.sMode[i >> 1];
    in.b = a.sB[i];
    load_rows<EAGER>(a, i, pass, in);
}

// ContactConstraints::solve (src/ContactConstraints.cpp:33-124) of one side of a manifold,
// normal then friction rows, on its body's solver velocities (v.w = invMass; updated in
// place); the even lane stores the accumulated lambdas. Manifolds of one colour touch
// disjoint dynamic bodies, so a colour is solved in parallel exactly as a sequential pass
// over it would be. Both lanes of the pair run it together.
//
// A pass is a chain of these, each a chain of points on its body's velocities, so what counts
// is the instructions a wave issues one after the other: one branch per point and row (soft
// rows, rare, have theirs only in waves that hold one), selects for the rest. With a branch
// for each condition a colour of four-point manifolds took 1.7 us of a run's workgroup.
__device__ __forceinline__ void solve_side(int i, SideIn& in, int pass, float4& v4, f3& w) {
    const bool moves = in.b >= 0;
    const float im = (i & 1) ? v4.w : -v4.w;
    const f3 n = xyz(in.n), sn = signed_of(n, i & 1);
    const bool anySoft = __ballot(in.soft) != 0;
    f3 v = xyz(v4);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!(in.mode & (MODE_N << k))) continue;
        const float4* r = in.row[k];
        const float p = dot(sn, v), q = dot(xyz(r[RS_N]), w);
        const float rv = side0(p + q) + side1(p) + side1(q);
        float lambda = (rv - r[RS_N].w + ((pass & PASS_BIAS) ? r[RS_TT].w : 0.f)) * r[RS_NT].w;
        if (anySoft) {
            if (in.soft) lambda = (rv + r[RS_TT].w) / r[RS_NT].w;
        }
        const float prev = in.lam[k].x;
        in.lam[k].x = gmin(prev + lambda, 0.f);
        // a side that does not move has zero velocities, which a zero push leaves as they are
        lambda = moves ? in.lam[k].x - prev : 0.f;
        v = sub(v, mul(lambda * im, n));   // the normal with side 1's sign times -im or im: the side's own sign
        w = sub(w, mul(lambda, xyz(r[RS_NT])));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (!(in.mode & (MODE_T << k))) continue;
        const float limit = in.n.w * in.lam[k].x;
        const float prev = in.lam[k].y;
        in.lam[k].y = gclamp(prev + in.t[k].w, limit, -limit);
        const float lambda = moves ? in.lam[k].y - prev : 0.f;
        v = sub(v, mul(lambda * im, xyz(in.t[k])));
        w = sub(w, mul(lambda, xyz(in.row[k][RS_TT])));
    }
    v4 = f4(v, v4.w);
}
// the manifold's accumulated lambdas, by its even lane, once the velocities are handed on
__device__ __forceinline__ void store_lambdas(const SubArgs& a, int i, const SideIn& in, int pass) {
    if ((i & 1) || (pass & PASS_LAST)) return;
    const int s = i >> 1;
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (k < in.num) LAM(k) = in.lam[k];
}

// one side of a manifold of a colour launch: every other manifold touching its body is in
// another launch, so plain accesses see the previous colours' results
template <bool EAGER = false>
__device__ void solve_lane(const SubArgs& a, int i, int pass) {
    SideIn in;
    load_side<EAGER>(a, i, pass, in);
    if ((pass & PASS_SKIP_SOFT) && in.soft) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    f3 w = s3(0.f);
    if (in.b >= 0) { v = a.bvel[bv(in.b, BV_V)]; w = xyz(a.bvel[bv(in.b, BV_W)]); }
    solve_side(i, in, pass, v, w);
    if (in.b >= 0) { a.bvel[bv(in.b, BV_V)] = v; a.bvel[bv(in.b, BV_W)] = f4(w, 0.f); }
    store_lambdas(a, i, in, pass);
}

// integrate positions of one body, src/Physecs.cpp:494-511
__device__ void integrate_position(const SubArgs& a, int d) {
    float4 cm = a.dcom[d];
    if (cm.w != 0.f) return;
    float4 pa = a.pang[d];
    float cnt = pa.w;
    float sc = cnt != 0.f ? 1.f / cnt : 1.f;
    f3 com = xyz(cm);
    f3 pos = xyz(a.bpos[d]);
    qf q = q4(a.bquat[d]);
    pos = add(pos, add(mul(a.h, xyz(a.bvel[bv(d, BV_V)])), mul(sc, xyz(a.pvel[d]))));
    f3 prevCom = qrot(q, com);
    f3 hv = mul(0.5f, add(mul(a.h, xyz(a.bvel[bv(d, BV_W)])), mul(sc, xyz(pa))));
    qf dq = qmul(mkq(0.f, hv.x, hv.y, hv.z), q);
    q = mkq(q.w + dq.w, q.x + dq.x, q.y + dq.y, q.z + dq.z);
    q = qnormalize(q);
    pos = add(pos, sub(prevCom, qrot(q, com)));
    a.bpos[d] = f4(pos, 0.f);
    a.bquat[d] = f4q(q);
}

// write back, src/Physecs.cpp:523-530, and, when another substep follows (next), its
// velocity integration: one launch over the bodies between two substeps
__device__ void write_back(const SubArgs& a, int d, bool next) {
    if (a.dcom[d].w != 0.f) return;
    const float4 v = a.bvel[bv(d, BV_V)], w = a.bvel[bv(d, BV_W)];
    a.dvel[d] = v;
    a.dang[d] = w;
    if (next) integrate_velocity(a, d, v, xyz(w));
}

// ------------------------------------------------------------------ discrete kernels
// the first substep's velocity integration
__global__ __launch_bounds__(256) void k_integrate_velocities(SubArgs a) {
    const int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d < a.D) integrate_velocity(a, d, a.dvel[d], xyz(a.dang[d]));
}

__global__ __launch_bounds__(256) void k_prepare(SubArgs a, int sub) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x, nth = gridDim.x * blockDim.x;
    for (int j = i; j < (a.iterations + 1) * FLOW_QUEUES; j += nth) a.tickets[j] = 0;
    if (i == 0) a.barrier[0] = 0;
    for (int j = i; j < a.xctlWords; j += nth) a.xctl[j] = 0;
    if (sub == 0 && i < FLOW_QUEUES) a.qDone[i] = 0;
    if (i < 2 * a.M) prepare_side(a, i);
}
// XCD-homed lanes. Workgroups are dispatched round-robin to the 8 XCDs (workgroup b on XCD
// b % 8), each with its own L2. k_prepare writes side lane i's rows from workgroup i / 256, so
// from XCD (i / 256) % 8, the lane's home; the colour launches give each workgroup a chunk
// of BLOCK lanes homed on its own XCD, so the rows (and the lambdas, rewritten in place every
// pass) are read from that XCD's L2 rather than from memory. Chunk k holds lanes
// [k * BLOCK, (k + 1) * BLOCK); its home is (k / q) % 8 with q = 256 / BLOCK chunks per
// prepare workgroup, so home-x chunks come in runs of q, one run every 8q chunks. Workgroup
// b (XCD x = b % 8) takes the (b / 8)-th home-x chunk at or after chunk k0.
__device__ __forceinline__ int homed_chunk(int b, int k0, int q) {
    const int x = b & 7, i = b >> 3, period = 8 * q;
    const int g = k0 / period, r = k0 - g * period;
    const int m = q * g + min(max(r - q * x, 0), q) + i;   // home-x chunks below k0, plus i
    return period * (m / q) + q * x + (m % q);
}

// side lanes [begin, end) of one colour (both even)
template <int BLOCK, bool EAGER>
__global__ __launch_bounds__(BLOCK) void k_solve(SubArgs a, int begin, int end, int pass) {
    const int k = homed_chunk(blockIdx.x, begin / BLOCK, 256 / BLOCK);
    const int i = k * BLOCK + threadIdx.x;
    if (i >= begin && i < end) solve_lane<EAGER>(a, i, pass);
}

// ------------------------------------------------------------------ one launch per pass
// k_solve_pass runs every colour of one contact pass in one launch, a grid barrier between
// colours. Within it, the only data that passes from one colour to the next across CUs (and
// XCDs, whose L2 caches are not coherent with each other) is the bodies' solver velocities:
// they are read and written with relaxed agent-scope atomic accesses, which go to the
// device's coherence point, so the barrier needs no cache writeback. Each thread's
// accesses are complete (s_waitcnt 0) before its workgroup arrives; one lane per workgroup
// adds the arrival and polls the count with agent-scope loads. Every other input of a
// manifold is fixed for the pass and read with plain loads: a thread loads the next colour's
// manifold before it waits at the barrier. Lambdas are read and written by the same thread
// within the launch.
constexpr int PASS_THREADS = 256;
constexpr int PASS_SPIN_LIMIT = 1 << 22;   // ~seconds; never expected with co-resident blocks

__device__ __forceinline__ f3 ld_agent3(const float4* p) {
    uint32_t* q = reinterpret_cast<uint32_t*>(const_cast<float4*>(p));
    const uint32_t x = __hip_atomic_load(q + 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t y = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const uint32_t z = __hip_atomic_load(q + 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return mk3(__uint_as_float(x), __uint_as_float(y), __uint_as_float(z));
}
__device__ __forceinline__ void st_agent3(float4* p, f3 v) {
    uint32_t* q = reinterpret_cast<uint32_t*>(p);
    __hip_atomic_store(q + 0, __float_as_uint(v.x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 1, __float_as_uint(v.y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 2, __float_as_uint(v.z), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// the solve of one side whose fixed inputs are loaded, on velocities at the coherence point
// (the inverse mass beside them never changes)
__device__ __forceinline__ void solve_coherent(const SubArgs& a, int i, SideIn& in, int pass) {
    if ((pass & PASS_SKIP_SOFT) && in.soft) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    f3 w = s3(0.f);
    if (in.b >= 0) {
        v = f4(ld_agent3(&a.bvel[bv(in.b, BV_V)]), a.bvel[bv(in.b, BV_V)].w);
        w = ld_agent3(&a.bvel[bv(in.b, BV_W)]);
    }
    solve_side(i, in, pass, v, w);
    if (in.b >= 0) { st_agent3(&a.bvel[bv(in.b, BV_V)], xyz(v)); st_agent3(&a.bvel[bv(in.b, BV_W)], w); }
    store_lambdas(a, i, in, pass);
}

// grid barrier number `target` / gridDim.x of the substep: every workgroup has arrived
// `target` times in all. A wait that runs out (or that finds another one ran out) sets the
// error flag and lets the grid go on, so every wave still reaches the end of the kernel.
__device__ __forceinline__ void pass_barrier(int32_t* count, int target, int32_t* err) {
    __builtin_amdgcn_s_waitcnt(0);   // this thread's velocity stores are at the coherence point
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_fetch_add(count, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int spins = 0;
        while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            __builtin_amdgcn_s_sleep(1);
            if (++spins > PASS_SPIN_LIMIT || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
    }
    __syncthreads();
}

__global__ __launch_bounds__(PASS_THREADS) void k_solve_pass(SubArgs a, int nColors, int pass, int barrierBase) {
    const int tid = blockIdx.x * PASS_THREADS + threadIdx.x;
    const int nth = gridDim.x * PASS_THREADS;
    int i = 2 * a.colorStart[0] + tid, e = 2 * a.colorStart[1];
    SideIn in;
    bool have = i < e;
    if (have) load_side<true>(a, i, pass, in);
    for (int c = 0; c < nColors; ++c) {
        if (have) solve_coherent(a, i, in, pass);
        for (int i2 = i + nth; i2 < e; i2 += nth) {
            SideIn in2;
            load_side<true>(a, i2, pass, in2);
            solve_coherent(a, i2, in2, pass);
        }
        if (c + 1 == nColors) break;
        i = e + tid;                 // the next colour starts where this one ends
        e = 2 * a.colorStart[c + 2];
        have = i < e;
        if (have) load_side<true>(a, i, pass, in);
        pass_barrier(a.barrier, barrierBase + (c + 1) * (int)gridDim.x, a.flowErr);
    }
}

// ------------------------------------------------------------------ one launch per pass, on one XCD
// k_solve_xpass runs every colour of one contact pass in one launch, like k_solve_pass, but
// only on the CUs of one XCD, so the solver velocities handed from one colour to the next
// stay in that XCD's L2 instead of crossing to the device's coherence point:
// - every workgroup registers the XCD it runs on (hardware register XCC_ID) with one
//   agent-scope atomic add on a 64-bit word holding one byte per XCD; the byte's old value
//   is the workgroup's rank on its XCD. When all gridDim.x have registered, every workgroup
//   reads the word and the XCD with the most workgroups (the lowest on a tie) is chosen;
//   the workgroups of the other XCDs leave;
// - the participants solve the colours in order, a barrier between colours: velocities are
//   loaded with agent-scope loads, which skip the CU's L1 and are served by the XCD's L2,
//   where the other participants' plain stores land; stores are plain and complete
//   (s_waitcnt 0) before a workgroup arrives at the barrier (pass_barrier's count);
// - every wait is bounded and reports through flowErr.
// ctl (per launch, cleared by k_prepare): [0..1] the registration word, [2] the barrier count.
constexpr int XPASS_THREADS = 256;
constexpr int XPASS_CTL = 4;        // int32 words of one launch's control block
constexpr int XPASS_MAX_GRID = 248; // at most 31 workgroups per XCD: a byte never overflows

__device__ __forceinline__ f3 ld_l2_3(const float4* p) { return ld_agent3(p); }

__device__ __forceinline__ void solve_xcd(const SubArgs& a, int i, SideIn& in, int pass) {
    if ((pass & PASS_SKIP_SOFT) && in.soft) return;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    f3 w = s3(0.f);
    if (in.b >= 0) {
        v = f4(ld_l2_3(&a.bvel[bv(in.b, BV_V)]), a.bvel[bv(in.b, BV_V)].w);
        w = ld_l2_3(&a.bvel[bv(in.b, BV_W)]);
    }
    solve_side(i, in, pass, v, w);
    if (in.b >= 0) { a.bvel[bv(in.b, BV_V)] = v; a.bvel[bv(in.b, BV_W)] = f4(w, 0.f); }
    store_lambdas(a, i, in, pass);
}

__global__ __launch_bounds__(XPASS_THREADS) void k_solve_xpass(SubArgs a, int nColors, int pass, int32_t* ctl) {
    __shared__ int sRank, sP;
    unsigned long long* reg = reinterpret_cast<unsigned long long*>(ctl);
    if (threadIdx.x == 0) {
        const int x = (int)(__builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 7);   // hwreg(HW_REG_XCC_ID)
        const unsigned long long old =
            __hip_atomic_fetch_add(reg, 1ull << (8 * x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        int spins = 0;
        unsigned long long v = 0;
        for (;;) {
            v = __hip_atomic_load(reg, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            int total = 0;
            for (int k = 0; k < 8; ++k) total += (int)((v >> (8 * k)) & 255);
            if (total >= (int)gridDim.x) break;
            __builtin_amdgcn_s_sleep(1);
            if (++spins > PASS_SPIN_LIMIT || __hip_atomic_load(a.flowErr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                __hip_atomic_store(a.flowErr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v = 0;
                break;
            }
        }
        int best = 0, bestN = 0;
        for (int k = 0; k < 8; ++k) {
            const int c = (int)((v >> (8 * k)) & 255);
            if (c > bestN) { best = k; bestN = c; }
        }
        sRank = (int)((old >> (8 * x)) & 255);
        sP = (x == best) ? bestN : 0;
    }
    __syncthreads();
    const int P = sP;
    if (P == 0) return;            // another XCD's workgroup (or registration failed)
    const int tid = sRank * XPASS_THREADS + threadIdx.x;
    const int nth = P * XPASS_THREADS;
    int i = 2 * a.colorStart[0] + tid, e = 2 * a.colorStart[1];
    SideIn in;
    bool have = i < e;
    if (have) load_side<true>(a, i, pass, in);
    for (int c = 0; c < nColors; ++c) {
        if (have) solve_xcd(a, i, in, pass);
        for (int i2 = i + nth; i2 < e; i2 += nth) {
            SideIn in2;
            load_side<true>(a, i2, pass, in2);
            solve_xcd(a, i2, in2, pass);
        }
        if (c + 1 == nColors) break;
        i = e + tid;
        e = 2 * a.colorStart[c + 2];
        have = i < e;
        if (have) load_side<true>(a, i, pass, in);
        pass_barrier(ctl + 2, (c + 1) * P, a.flowErr);
    }
}

// Consecutive small colours c0..c1-1 (solve slots [S, E)) in one launch of one workgroup:
// the colours are solved in order with a workgroup barrier between them, so the solve order
// is the colour order, exactly as with one launch per colour. The solver velocities of the
// run's bodies stay in LDS for the whole run: one gather before the first colour, one
// scatter after the last, and between colours only the manifolds' fixed inputs come from
// global memory. k_batch_map gives each run its bodies (batchList, from 2S on) and each
// manifold side its LDS slot (batchLoc, 2 per solve slot; -1 for a static side), once per
// step: a run's slots never change within the step.
constexpr int BATCH_THREADS = 1024;     // two lanes per manifold; 4 waves per SIMD at 128 registers
constexpr int BATCH_MAP_THREADS = 1024;
constexpr int BATCH_HASH = 8192;        // LDS hash of body -> slot, at most 59% full
constexpr int BATCH_MAX_GROUPS = 16;
constexpr int BATCH_MAX_MANIFOLDS = 2400;   // 2 x 2400 bodies x 32 B of velocities in LDS
static_assert(10 * 2 * BATCH_MAX_MANIFOLDS <= 6 * BATCH_HASH, "a run's bodies fill at most six tenths of the hash");
constexpr int BATCH_MAX_COLOURS = 128;
constexpr int BATCH_LANES = BATCH_THREADS / 2;   // a team's
constexpr int BATCH_MAX_TURNS = BATCH_MAX_COLOURS + 2 * BATCH_MAX_MANIFOLDS / BATCH_LANES + 1;

struct BatchGroups {
    int n;
    int S[BATCH_MAX_GROUPS], E[BATCH_MAX_GROUPS];
    int c0[BATCH_MAX_GROUPS], c1[BATCH_MAX_GROUPS];   // colours
    int turns[BATCH_MAX_GROUPS];
};

__device__ __forceinline__ uint32_t batch_hash(int b) { return ((uint32_t)b * 2654435761u) >> (32 - 13); }

// One workgroup, every run in turn: the run's bodies get slots 0..n-1 in first-claim order
// (the order does not reach the arithmetic) through an LDS hash table with linear probing.
__global__ __launch_bounds__(BATCH_MAP_THREADS) void k_batch_map(BatchGroups g, const int32_t* __restrict__ sB,
                                                                 int32_t* __restrict__ batchLoc,
                                                                 int32_t* __restrict__ batchList,
                                                                 const int32_t* __restrict__ colorStart,
                                                                 int2* __restrict__ batchTurns) {
    static_assert(BATCH_HASH == 1 << 13, "batch_hash gives 13 bits");
    __shared__ int32_t hk[BATCH_HASH], hv[BATCH_HASH];
    __shared__ int32_t count;
    const int q = blockIdx.x;
    const int S = g.S[q], E = g.E[q], sides = 2 * (E - S);
    for (int i = threadIdx.x; i < BATCH_HASH; i += BATCH_MAP_THREADS) hk[i] = -1;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < sides; i += BATCH_MAP_THREADS) {
        const int b = sB[2 * S + i];
        if (b < 0) continue;
        uint32_t h = batch_hash(b);
        for (int probe = 0; probe < BATCH_HASH; ++probe) {   // the table is never full
            const int prev = atomicCAS(&hk[h], -1, b);
            if (prev == -1) {
                const int slot = atomicAdd(&count, 1);
                hv[h] = slot;
                batchList[2 * S + slot] = b;
                break;
            }
            if (prev == b) break;
            h = (h + 1) & (BATCH_HASH - 1);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < sides; i += BATCH_MAP_THREADS) {
        const int b = sB[2 * S + i];
        int slot = -1;
        if (b >= 0) {
            uint32_t h = batch_hash(b);
            for (int probe = 0; probe < BATCH_HASH && hk[h] != b; ++probe) h = (h + 1) & (BATCH_HASH - 1);
            slot = hv[h];
        }
        batchLoc[2 * S + i] = slot;
    }
    for (int i = count + threadIdx.x; i < sides; i += BATCH_MAP_THREADS) batchList[2 * S + i] = -1;
    if (threadIdx.x < WAVE) {   // the turns, in colour order
        int2* turns = batchTurns + (size_t)BATCH_MAX_TURNS * q;
        int at = 0;
        for (int c = g.c0[q]; c < g.c1[q]; c += WAVE) {
            const int k = c + (int)threadIdx.x;
            int b = 0, e = 0;
            if (k < g.c1[q]) { b = 2 * colorStart[k]; e = 2 * colorStart[k + 1]; }
            const int mine = (e - b + BATCH_LANES - 1) / BATCH_LANES;
            int x = mine;
            for (int o = 1; o < WAVE; o <<= 1) {
                const int y = __shfl_up(x, o);
                if ((int)threadIdx.x >= o) x += y;
            }
            for (int j = 0; j < mine; ++j) turns[at + x - mine + j] = make_int2(b + j * BATCH_LANES, min(b + (j + 1) * BATCH_LANES, e));
            at += __shfl(x, WAVE - 1);
        }
    }
}

// A workgroup barrier that orders LDS only: the global loads a thread has in flight stay in
// flight across it (s_waitcnt lgkmcnt(0); s_barrier).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The run's bodies' velocities (solver v with the inverse mass, and w) are gathered into
// LDS once per launch, so a manifold's solve needs only its own rows from global memory.
// Those are two dependent rounds of loads (the mode, then as many slots as the mode has
// points), longer than the solve itself, so the workgroup's waves form two teams that take
// turns: while one team solves a turn (a colour, or 512 lanes of a larger one), the other
// stores its lambdas and loads the rows of its next turn (their modes were loaded a turn
// earlier). A barrier between turns orders LDS only. The first rows and the bodies' velocities
// are fetched together. 415 manifolds in eight colours: 11.5 us, 18.5 with one team that loads
// a colour after the one before it; four teams of 256 lanes take 12.2 and eight of 128 15.4
// (more turns), two of 256 11.6 there and 13.0 for 11.9 on 789 manifolds.
// FIRST: the substep's first pass, whose lambdas are not read (a branch on the pass would wait
// for the loads).
template <bool FIRST>
__global__ __launch_bounds__(BATCH_THREADS) void k_solve_batch(SubArgs a, int S, int E, int total,
                                                               const int2* __restrict__ turnsIn,
                                                               const int32_t* __restrict__ batchLoc,
                                                               const int32_t* __restrict__ batchList, int flags) {
    const int pass = FIRST ? flags | PASS_FIRST : flags & ~PASS_FIRST;
    extern __shared__ float4 rec[];       // [n] solver v, then [n] solver w of the run's bodies
    __shared__ int2 turns[BATCH_MAX_TURNS];   // side lanes [x, y), in colour order
    const int n = 2 * (E - S);
    const int team = __builtin_amdgcn_readfirstlane((int)threadIdx.x / BATCH_LANES), t = (int)threadIdx.x - team * BATCH_LANES;
    constexpr int GATHER = (2 * BATCH_MAX_MANIFOLDS + BATCH_THREADS - 1) / BATCH_THREADS;
    int body[GATHER];   // the bodies this thread gathers and writes back: slots threadIdx.x + 1024 j
#pragma unroll
    for (int j = 0; j < GATHER; ++j) {
        const int i = threadIdx.x + j * BATCH_THREADS;
        body[j] = i < n ? batchList[2 * S + i] : -1;
    }
    if ((int)threadIdx.x < total) turns[threadIdx.x] = turnsIn[threadIdx.x];
    lds_barrier();
    // a side's turn: its place, and what is loaded a turn ahead of its rows
    struct Turn { int i, mode, b, l; };
    auto turn = [&](int k, Turn& h) {
        h.i = -1;
        if (k >= total) return;
        const int2 range = turns[k];
        if (range.x + t >= range.y) return;
        h.i = range.x + t;
        h.mode = a.sMode[h.i >> 1];
        h.b = a.sB[h.i];
        h.l = batchLoc[h.i];
    };
    auto rows = [&](const Turn& h, SideIn& in) {
        SideIn x;   // slots that are not loaded hold nothing, not the last turn's rows
        x.mode = h.mode;
        x.b = h.b;
        if (h.i >= 0) load_rows(a, h.i, pass, x);
        in = x;
    };
    Turn now, next;
    SideIn in;
    turn(team, now);
#pragma unroll
    for (int j = 0; j < GATHER; ++j) {
        if (body[j] < 0) continue;
        const int i = threadIdx.x + j * BATCH_THREADS;
        rec[i] = a.bvel[bv(body[j], BV_V)];
        rec[n + i] = a.bvel[bv(body[j], BV_W)];
    }
    rows(now, in);
    turn(team + 2, next);
    for (int k = 0; k <= total; ++k) {
        lds_barrier();   // the previous turn's velocities are in LDS
        if (k < total && (k & 1) == team && now.i >= 0 && !((pass & PASS_SKIP_SOFT) && in.soft)) {
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            f3 w = s3(0.f);
            if (in.b >= 0) { v = rec[now.l]; w = xyz(rec[n + now.l]); }
            solve_side(now.i, in, pass, v, w);
            if (in.b >= 0) { rec[now.l] = v; rec[n + now.l] = f4(w, 0.f); }
        }
        // after its turn, while the next team solves
        if (k > 0 && ((k - 1) & 1) == team) {
            if (now.i >= 0 && !((pass & PASS_SKIP_SOFT) && in.soft)) store_lambdas(a, now.i, in, pass);
            now = next;
            // arrived a turn ago: taken before the rows' loads, which a later wait for them
            // would wait for too
            asm volatile("" : "+v"(now.i), "+v"(now.mode), "+v"(now.b), "+v"(now.l));
            rows(now, in);
            turn(k + 3, next);
        }
    }
    lds_barrier();
#pragma unroll
    for (int j = 0; j < GATHER; ++j) {
        if (body[j] < 0) continue;
        const int i = threadIdx.x + j * BATCH_THREADS;
        a.bvel[bv(body[j], BV_V)] = rec[i];
        a.bvel[bv(body[j], BV_W)] = rec[n + i];
    }
}

// ------------------------------------------------------------------ per-world passes
// Worlds never share a body, and a world's dynamic bodies are a contiguous index range, so
// one workgroup can run a whole contact pass of one world: the solver velocities of its
// bodies in LDS, its manifolds colour by colour with a workgroup barrier between colours.
// Every body sees its manifolds in colour order, as with one launch per colour, so the
// floats are the same. No launch per colour and no global body gathers inside the pass.
struct WorldPassArgs {
    int W, nColors;
    const int32_t* wDyn;                  // W + 1: first dynamic body of each world
    const int32_t *wcS, *wcE;             // per colour and world: its solve slots [S, E)
    const int32_t* list;                  // the worlds of this launch (one workgroup each)
};

// the solve slots of every (colour, world) run; slots are in colour order and, within a
// colour, in world order. Absent runs stay [0, 0).
__global__ void k_world_ranges(int M, int W, const int32_t* __restrict__ sFlags, const int32_t* __restrict__ sWorld,
                               int32_t* __restrict__ wcS, int32_t* __restrict__ wcE) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= M) return;
    const int c = (sFlags[s] >> 16) & 127, wd = sWorld[s];
    if (s == 0 || ((sFlags[s - 1] >> 16) & 127) != c || sWorld[s - 1] != wd) wcS[c * W + wd] = s;
    if (s == M - 1 || ((sFlags[s + 1] >> 16) & 127) != c || sWorld[s + 1] != wd) wcE[c * W + wd] = s + 1;
}

// One wave per world: a world's colour holds a few dozen manifolds, two lanes each, and
// one-wave workgroups keep many worlds resident per CU (when their LDS fits). Rows are
// loaded eagerly: these colours are latency-bound.
constexpr int WORLD_THREADS = 64;
__global__ __launch_bounds__(WORLD_THREADS) void k_world_pass(SubArgs a, WorldPassArgs p, int pass) {
    extern __shared__ float4 wv[];        // [n] solver v, then [n] solver w of the world's bodies
    const int wd = p.list[blockIdx.x];
    const int d0 = p.wDyn[wd], n = p.wDyn[wd + 1] - d0;
    if (n == 0) return;
    for (int i = threadIdx.x; i < n; i += WORLD_THREADS) {
        wv[i] = a.bvel[bv(d0 + i, BV_V)];
        wv[n + i] = a.bvel[bv(d0 + i, BV_W)];
    }
    __syncthreads();
    for (int c = 0; c < p.nColors; ++c) {
        const int S = 2 * p.wcS[c * p.W + wd], E = 2 * p.wcE[c * p.W + wd];
        for (int i = S + (int)threadIdx.x; i < E; i += WORLD_THREADS) {
            SideIn in;
            load_side<true>(a, i, pass, in);
            if ((pass & PASS_SKIP_SOFT) && in.soft) continue;
            const int l = in.b - d0;
            float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
            f3 w = s3(0.f);
            if (in.b >= 0) { v = wv[l]; w = xyz(wv[n + l]); }
            solve_side(i, in, pass, v, w);
            if (in.b >= 0) { wv[l] = v; wv[n + l] = f4(w, 0.f); }
            store_lambdas(a, i, in, pass);
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < n; i += WORLD_THREADS) {
        a.bvel[bv(d0 + i, BV_V)] = wv[i];
        a.bvel[bv(d0 + i, BV_W)] = wv[n + i];
    }
}

// colours of body b, and its colours below colour c
__device__ __forceinline__ int colours_of(const uint64_t* used, int b) {
    return __popcll(used[2 * b]) + __popcll(used[2 * b + 1]);
}
__device__ __forceinline__ int colours_below(const uint64_t* used, int b, int c) {
    uint64_t lo = used[2 * b], hi = used[2 * b + 1];
    if (c < 64) return __popcll(lo & ((1ull << c) - 1ull));
    return __popcll(lo) + __popcll(hi & ((1ull << (c - 64)) - 1ull));
}

// ------------------------------------------------------------------ dependency-driven pass
// A pass (one of the substep's biased iterations, or the relaxation) over every colour in
// ONE launch. A manifold of colour c needs the velocities its bodies hold after their
// manifolds of lower colours in this pass; with r = (colours of body b below c) such
// manifolds before it, the r-th of them publishes body b's velocities under version
// (epoch, r). The first manifold of a body (r = 0) reads the plain solver velocities, which
// are complete when the launch starts (previous pass, joints); its last manifold of the
// pass writes them, their only writer in the launch.
//
// Published velocities: 6 words of {value, version} per body, each word readable on its
// own, so a reader accepts a record only when all six carry the version it waits for and
// needs no ordering between the words' stores. Records are agent-scope atomic accesses (a
// load that hits the CU's own cache may never see another CU's store within a launch).
// Queues: one device-wide queue, or one per XCD (world w on XCD w % XCDs; waves take
// manifolds only from their own XCD's queue, read from the hardware register XCC_ID), so
// that a world's hand-offs stay inside one XCD: a few hundred nanoseconds each, against
// microseconds between XCDs.
//
// The solve order is the colour order's, so the arithmetic is exactly that of one launch
// per colour. Waves take manifolds in solve order from the pass's ticket, 32, or 64 that they
// solve in two turns (more than FLOW_RESIDENT in all): a
// manifold waits only on manifolds of lower solve positions, which are solved, or held by waves
// already running that solve lower ones first, so the waits resolve in order. Every wait is bounded; one that runs out sets flowErr and
// gives up (the host reports the error) rather than hang.
constexpr int FLOW_SPIN_LIMIT = 1 << 18;   // ~0.5 s of polling: a wait this long is a bug

constexpr int FLOW_RESIDENT = 131072;      // 32 manifolds each of the waves that fit the chip, four a SIMD (128 registers)

struct FlowArgs {
    int index;                             // the pass within its substep
    int take;                              // manifolds per ticket, a multiple of 32
    int pass;                              // PASS_* flags
    uint32_t epoch;                        // unique per launch (24 bits used)
    uint64_t* pub;                         // 6 words per body
    int xcdScope;                          // 1: a queue per XCD, 0: one queue
    int nQueues;
    const int32_t* qStart;                 // nQueues + 1 offsets into qList
    const int32_t* qList;                  // solve positions by queue (nullptr: identity)
};

__device__ __forceinline__ uint64_t pub_word(float v, uint32_t ver) {
    return (uint64_t)__float_as_uint(v) | ((uint64_t)ver << 32);
}

// body b's published velocities under version ver, if all six words carry it
__device__ __forceinline__ bool read_pub(const FlowArgs& f, int b, uint32_t ver, f3& v, f3& w) {
    uint64_t q[6];
    uint64_t* p = f.pub + 6 * (size_t)b;
#pragma unroll
    for (int k = 0; k < 6; ++k) q[k] = __hip_atomic_load(p + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    bool ok = true;
#pragma unroll
    for (int k = 0; k < 6; ++k) ok = ok && (uint32_t)(q[k] >> 32) == ver;
    v = mk3(__uint_as_float((uint32_t)q[0]), __uint_as_float((uint32_t)q[1]), __uint_as_float((uint32_t)q[2]));
    w = mk3(__uint_as_float((uint32_t)q[3]), __uint_as_float((uint32_t)q[4]), __uint_as_float((uint32_t)q[5]));
    return ok;
}

// Hands body b's velocities on after one of its manifolds: to the next manifold of the
// pass (published under version ver), or, after its last manifold of the pass, to the
// kernels after the pass (the plain solver velocities, written back at the launch's end).
__device__ __forceinline__ void hand_on(const SubArgs& a, const FlowArgs& f, int b, bool last, uint32_t ver, float4 v,
                                        f3 w) {
    if (last) {
        a.bvel[bv(b, BV_V)] = v;
        a.bvel[bv(b, BV_W)] = f4(w, 0.f);
        return;
    }
    uint64_t* p = f.pub + 6 * (size_t)b;
    __hip_atomic_store(p + 0, pub_word(v.x, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 1, pub_word(v.y, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 2, pub_word(v.z, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 3, pub_word(w.x, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 4, pub_word(w.y, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(p + 5, pub_word(w.z, ver), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ __launch_bounds__(256, 4) void k_solve_flow(SubArgs a, FlowArgs f) {
    const int lane = threadIdx.x & (WAVE - 1);
    int queue = 0;
    if (f.xcdScope) {
        queue = (int)(__builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) & 15);   // hwreg(HW_REG_XCC_ID, 0, 4)
        if (queue >= f.nQueues) return;
    }
    const int qb = f.qStart[queue], qn = f.qStart[queue + 1] - qb;
    const uint32_t vbase = (f.epoch & 0xffffffu) << 8;
    int done = 0, base = -WAVE / 2, taken = 0;
    for (;;) {
        if ((base += WAVE / 2) == taken) {   // the next manifolds of the pass
            if (lane == 0) base = atomicAdd(a.tickets + f.index * FLOW_QUEUES + queue, f.take);
            base = __shfl(base, 0);
            taken = base + f.take;
        }
        if (base >= qn) break;
        const int idx = base + (lane >> 1);
        bool pending = idx < qn;           // the same in both lanes of a pair
        const int i = 2 * (pending ? (f.qList ? f.qList[qb + idx] : qb + idx) : 0) + (lane & 1);
        SideIn in;
        int r = 0;
        bool last = false, have = true;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        f3 w = s3(0.f);
        if (pending) {
            // everything but the bodies' solver velocities is fixed for the pass: loaded
            // before the wait, off the critical path
            load_side(a, i, f.pass, in);
            const int c = a.sFlags[i >> 1] >> 16;
            if (in.b >= 0) {
                r = colours_below(a.used, in.b, c);
                last = r == colours_of(a.used, in.b) - 1;
                have = r == 0;
                v = a.bvel[bv(in.b, BV_V)];   // the velocities only when have; the inverse mass always
                w = xyz(a.bvel[bv(in.b, BV_W)]);
            }
        }
        int spins = 0;
        while (__ballot(pending)) {
            if (pending) {
                if (!have) {
                    f3 pv;
                    have = read_pub(f, in.b, vbase | (uint32_t)r, pv, w);
                    v = f4(pv, v.w);
                }
                const bool both = __builtin_amdgcn_mov_dpp((int)have, 0xB1, 0xf, 0xf, true) != 0 && have;   // quad_perm 1,0,3,2
                if (both) {
                    // a soft manifold in the relaxation passes its bodies' velocities on
                    const bool solved = !((f.pass & PASS_SKIP_SOFT) && in.soft);
                    if (solved) solve_side(i, in, f.pass, v, w);
                    if (in.b >= 0) hand_on(a, f, in.b, last, vbase | (uint32_t)(r + 1), v, w);
                    if (solved) store_lambdas(a, i, in, f.pass);
                    pending = false;
                    done += lane & 1;
                } else if (++spins > FLOW_SPIN_LIMIT) {
                    atomicOr(a.flowErr, 1);
                    pending = false;
                }
            }
            if (__ballot(pending)) __builtin_amdgcn_s_sleep(1);
        }
    }
    // manifolds finished per queue: the host checks that every queue was served
    for (int o = WAVE / 2; o > 0; o >>= 1) done += __shfl_xor(done, o);
    if (lane == 0 && done) atomicAdd(a.qDone + queue, done);
}

// The queues of the dependency-driven pass. One world, or one device-wide queue: queue 0
// is the whole solve order. Several worlds on XCD queues: world w goes to queue w % nq,
// keeping solve order inside each queue (a stable sort by queue).
__global__ void k_flow_identity(int M, int nq, int32_t* qStart) {
    int i = threadIdx.x;
    if (i <= nq) qStart[i] = i == 0 ? 0 : M;
}
__global__ void k_flow_keys(int M, const int32_t* __restrict__ sCanon, const uint64_t* __restrict__ mfKey,
                            int worldShift, int nq, uint64_t* __restrict__ keys, int32_t* __restrict__ vals) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= M) return;
    keys[s] = (mfKey[sCanon[s]] >> worldShift) % (uint64_t)nq;
    vals[s] = s;
}
__global__ void k_flow_starts(int M, int nq, const uint64_t* __restrict__ keys, int32_t* __restrict__ qStart) {
    int q = threadIdx.x;
    if (q > nq) return;
    int lo = 0, hi = M;   // first position with key >= q
    while (lo < hi) {
        int mid = (lo + hi) >> 1;
        if (keys[mid] < (uint64_t)q) lo = mid + 1;
        else hi = mid;
    }
    qStart[q] = lo;
}

__global__ __launch_bounds__(256) void k_integrate_positions(SubArgs a) {
    int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d < a.D) integrate_position(a, d);
}
__global__ __launch_bounds__(256) void k_writeback(SubArgs a, int next) {
    int d = blockIdx.x * blockDim.x + threadIdx.x;
    if (d < a.D) write_back(a, d, next != 0);
}

// ------------------------------------------------------------------ persistent kernel
// Every substep of one step in a single cooperative launch; grid-wide barriers separate the
// phases and the colours. Blocks are co-resident (cooperative launch), every block reaches
// every barrier the same number of times, and the kernel ends after the last substep.
__global__ __launch_bounds__(256) void k_step_persistent(SubArgs a) {
    cg::grid_group grid = cg::this_grid();
    const int tid = blockIdx.x * blockDim.x + threadIdx.x;
    const int nth = gridDim.x * blockDim.x;
    for (int d = tid; d < a.D; d += nth) integrate_velocity(a, d, a.dvel[d], xyz(a.dang[d]));
    grid.sync();
    for (int sub = 0; sub < a.substeps; ++sub) {
        for (int i = tid; i < 2 * a.M; i += nth) prepare_side(a, i);
        grid.sync();
        for (int it = 0; it < a.iterations; ++it) {
            for (int c = 0; c < a.nColors; ++c) {
                const int b = 2 * a.colorStart[c], e = 2 * a.colorStart[c + 1];
                for (int i = b + tid; i < e; i += nth) solve_lane(a, i, PASS_BIAS | (it == 0 ? PASS_FIRST : 0));
                grid.sync();
            }
        }
        for (int d = tid; d < a.D; d += nth) integrate_position(a, d);
        grid.sync();
        for (int c = 0; c < a.nColors; ++c) {
            const int b = 2 * a.colorStart[c], e = 2 * a.colorStart[c + 1];
            for (int i = b + tid; i < e; i += nth)
                solve_lane(a, i, PASS_SKIP_SOFT | PASS_LAST | (a.iterations == 0 ? PASS_FIRST : 0));
            grid.sync();
        }
        for (int d = tid; d < a.D; d += nth) write_back(a, d, sub + 1 < a.substeps);
        grid.sync();
    }
}

// ------------------------------------------------------------------ host orchestration
int sv_setup_manifolds(World& w, int nPairs) {
    hipStream_t s = w.stream;
    if (nPairs == 0) return 0;
    // manifold index of every pair with points: exclusive scan of the hit flags (the pair
    // sort's value buffer is free at this point and holds the flags)
    const CompactArgs ca{w.npNum.p, w.meshFirst.p, w.meshCount.p, w.npTri.p, w.pairCap, w.localBits, w.pkeys.p,
                         w.worldColStart.p, w.colOfLocal.p, w.cbody.p, w.cflags.p, w.mfPair.p, w.mfKey.p, w.mfB0.p,
                         w.mfB1.p, w.mfSrc.p, w.mfTri.p};
    const bool small = nPairs <= MANIFOLDS_SMALL;
    if (small) {
        hipLaunchKernelGGL(k_manifolds_small, dim3(1), dim3(MANIFOLDS_THREADS), 0, s, nPairs,
                           div_up(nPairs, MANIFOLDS_THREADS), ca, w.npIndex.p, w.flowErr.p, w.counters.p);
    } else {
        hipLaunchKernelGGL(k_flag_manifolds, dim3(div_up(nPairs, 256)), dim3(256), 0, s, nPairs, w.npNum.p,
                           w.meshCount.p, w.pvals.p, w.flowErr.p, w.counters.p);
        exclusive_scan_i32(s, w.pvals.p, w.npIndex.p, nPairs, w.counters.p + 1, w.scanT);
    }
    int M = 0, epaErrors = 0, flowErr = 0;
    int meshInfo[3] = {0, 0, 0};   // mesh pairs, mesh manifold slots, mesh capacity errors
    // the counters (manifold total, EPA and mesh counts) and the previous step's
    // dependency-driven passes: a wait that ran out, and every queue served by waves of its
    // XCD; to pinned host memory
    int qDone[FLOW_QUEUES] = {}, qStart[FLOW_QUEUES + 1] = {};
    const int lastQueues = w.lastQueues, lastPasses = w.lastFlowPasses;
    w.readHost.alloc(READ_HOST_INTS);
    int32_t* rb = w.readHost.p;
    PGX_HIP(hipMemcpyAsync(rb, w.counters.p, 16 * sizeof(int32_t), hipMemcpyDeviceToHost, s));
    if (lastQueues) {
        PGX_HIP(hipMemcpyAsync(qDone, w.qDone.p, sizeof(qDone), hipMemcpyDeviceToHost, s));
        PGX_HIP(hipMemcpyAsync(qStart, w.qStart.p, sizeof(int) * (lastQueues + 1), hipMemcpyDeviceToHost, s));
    }
    if (!small)
        hipLaunchKernelGGL(k_compact, dim3(div_up(nPairs, 256)), dim3(256), 0, s, nPairs, ca, w.npIndex.p);
    PGX_LAUNCH_CHECK();
    PGX_HIP(hipStreamSynchronize(s));
    M = rb[1];
    flowErr = rb[3];
    if (w.nConvex) epaErrors = rb[9];
    if (w.nTriMesh) std::copy(rb + 10, rb + 13, meshInfo);
    if (flowErr)
        throw PgxError{PGX_ERR_HIP, "contact solve: a wait of the previous step ran out (dependency-driven pass or "
                                    "grid barrier of the one-launch pass)"};
    for (int q = 0; q < lastQueues; ++q)
        if (qDone[q] != lastPasses * (qStart[q + 1] - qStart[q]))
            throw PgxError{PGX_ERR_HIP, "contact solve: queue " + std::to_string(q) + " of the previous step finished " +
                                            std::to_string(qDone[q]) + " of " +
                                            std::to_string(lastPasses * (qStart[q + 1] - qStart[q])) +
                                            " manifold solves (no wave ran on its XCD)"};
    if (epaErrors)
        throw PgxError{PGX_ERR_CAPACITY, "EPA polytope capacity exceeded in " + std::to_string(epaErrors) + " pairs"};
    if (meshInfo[2])
        throw PgxError{PGX_ERR_CAPACITY, "triangle-mesh narrowphase capacity exceeded in " +
                                             std::to_string(meshInfo[2]) + " pairs (candidates, stack or slots)"};
    w.lastMeshSlots = meshInfo[1];
    return M;
}

constexpr int MAX_ROUNDS = 1024;

// The colouring of at most COLOR_SMALL manifolds and bodies: one launch and the read-back.
static int color_small(World& w, int M, std::vector<int32_t>& starts, int& nColors) {
    hipStream_t s = w.stream;
    w.colorPack.alloc(133 + MAX_ROUNDS + 1);
    w.readHost.alloc(READ_HOST_INTS);
    w.mfPrev.alloc(w.manifoldCap);
    if (!w.colorLdsSet) {
        PGX_HIP(hipFuncSetAttribute((const void*)k_color_small, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)(3 * sizeof(uint64_t) * COLOR_SMALL)));
        w.colorLdsSet = true;
    }
    const int prv = w.cacheCur;
    hipLaunchKernelGGL(k_color_small, dim3(1), dim3(COLOR_THREADS), 3 * sizeof(uint64_t) * (size_t)w.D, s, M, w.D,
                       div_up(M, COLOR_THREADS), MAX_ROUNDS, w.mfKey.p, 2 * w.localBits, w.worldMStart.p, w.mfTri.p,
                       w.cacheKey[prv].p, w.cacheTri[prv].p, w.cacheNum[prv].p, w.cacheCount[prv], w.mfB0.p, w.mfB1.p,
                       w.npNum.p, w.mfSrc.p, w.execMode == EXEC_WORLDS ? 0 : 1, w.mfColor.p, w.mfPrev.p, w.usedMask.p,
                       w.colorPerm.p, w.colorRank.p, w.colorCount.p, w.colorPack.p);
    PGX_LAUNCH_CHECK();
    PGX_HIP(hipMemcpyAsync(w.readHost.p, w.colorPack.p, sizeof(int32_t) * 133, hipMemcpyDeviceToHost, s));
    PGX_HIP(hipStreamSynchronize(s));
    const int32_t* rb = w.readHost.p;
    if (rb[130]) throw PgxError{PGX_ERR_CAPACITY, "a body touches more than 127 contact colours"};
    if (rb[132] == 0) throw PgxError{PGX_ERR_INVALID, "graph colouring did not converge"};
    std::copy(rb, rb + 130, starts.begin());
    nColors = rb[131];
    return rb[132];
}

int sv_color(World& w, int M) {
    hipStream_t s = w.stream;
    const int prevRounds = w.lastRounds;
    w.lastRounds = 0;
    if (M == 0) {
        w.colorStartHost.assign(1, 0);
        return 0;
    }
    int worldShift = 2 * w.localBits;
    int nb = div_up(M, 256);
    std::vector<int32_t> starts(130, 0);
    int nColors = 0;
    if (M <= COLOR_SMALL && w.D <= COLOR_SMALL) {
        w.lastRounds = color_small(w, M, starts, nColors);
    } else {
        static_assert(133 + MAX_ROUNDS + 1 <= READ_HOST_INTS, "the colouring's read-back fits the pinned buffer");
        w.colorUncol.alloc(MAX_ROUNDS + 1);
        w.colorPack.alloc(133 + MAX_ROUNDS + 1);
        w.readHost.alloc(READ_HOST_INTS);
        w.claim2.alloc(std::max(w.D, 1));
        w.mfPrev.alloc(w.manifoldCap);
        w.colorFlag.alloc(1);
        hipLaunchKernelGGL(k_color_begin, dim3(div_up(std::max({M, 2 * w.D, MAX_ROUNDS + 1}), 256)), dim3(256), 0, s, M,
                           w.D, MAX_ROUNDS + 1, w.mfKey.p, worldShift, w.worldMStart.p, w.mfColor.p, w.claim.p,
                           w.claim2.p, w.usedMask.p, w.colorUncol.p, w.counters.p + 5, w.colorFlag.p);
        unsigned long long* claims[2] = {(unsigned long long*)w.claim.p, (unsigned long long*)w.claim2.p};
        // colours of the manifolds that persist from the previous step; only new ones are
        // coloured in the rounds below
        const int prevCache = w.cacheCur;
        hipLaunchKernelGGL(k_color_inherit, dim3(nb), dim3(256), 0, s, M, w.mfKey.p, w.mfTri.p, w.cacheKey[prevCache].p,
                           w.cacheTri[prevCache].p, w.cacheNum[prevCache].p, w.cacheCount[prevCache], w.mfB0.p, w.mfB1.p,
                           w.mfColor.p,
                           w.mfPrev.p, (unsigned long long*)w.usedMask.p, w.colorFlag.p);
        hipLaunchKernelGGL(k_color_clash, dim3(div_up(std::max(M, 2 * w.D), 256)), dim3(256), 0, s, M, w.D, w.colorFlag.p,
                           w.mfColor.p, w.usedMask.p);
        // round-1 claims
        hipLaunchKernelGGL(k_color_claim, dim3(nb), dim3(256), 0, s, M, 1, w.mfKey.p, worldShift, w.worldMStart.p,
                           w.mfColor.p, w.mfB0.p, w.mfB1.p, claims[1]);
        // Rounds are queued in batches sized from the last step's count (a round after the last
        // one needed exits at once); the sort into colour order and the colour starts follow,
        // and one read-back tells whether the batch finished, with the counts and starts. Only
        // a batch that ran short is followed by another (and the sort is redone).
        int round = 0;
        int batch = std::min(MAX_ROUNDS, std::max(w.tune.colorRounds, prevRounds + 4));
        std::vector<int32_t> uc;
        uint64_t lastKey = 0;
        while (true) {
            for (int r = 0; r < batch && round < MAX_ROUNDS; ++r) {
                ++round;
                hipLaunchKernelGGL(k_color_round, dim3(nb), dim3(256), 0, s, M, round, w.mfKey.p, worldShift,
                                   w.worldMStart.p, w.mfColor.p, w.mfB0.p, w.mfB1.p,
                                   (const unsigned long long*)claims[round & 1], claims[(round + 1) & 1], w.usedMask.p,
                                   w.colorUncol.p, w.counters.p);
            }
            // stable sort by colour and point count -> solve order
            hipLaunchKernelGGL(k_color_keys, dim3(nb), dim3(256), 0, s, M, w.mfColor.p, w.npNum.p, w.mfSrc.p,
                               w.execMode == EXEC_WORLDS ? 0 : 1, w.colorKeys.p, w.colorPerm.p);
            radix_sort_u64(s, w.colorKeys.p, w.colorPerm.p, M, 7 + COLOR_KEY_SHIFT, w.sortT);
            hipLaunchKernelGGL(k_color_start, dim3(1), dim3(256), 0, s, M, 130, w.colorKeys.p, w.colorCount.p, round,
                               w.colorUncol.p, w.counters.p + 5, w.colorPack.p);
            PGX_LAUNCH_CHECK();
            // one copy to pinned host memory brings the starts, the overflow flag, the last key
            // and the per-round counts
            const size_t packed = 133 + (size_t)round + 1;
            PGX_HIP(hipMemcpyAsync(w.readHost.p, w.colorPack.p, sizeof(int32_t) * packed, hipMemcpyDeviceToHost, s));
            PGX_HIP(hipStreamSynchronize(s));
            const int32_t* rb = w.readHost.p;
            const int ovf = rb[130];
            lastKey = (uint64_t)(uint32_t)rb[131] | ((uint64_t)(uint32_t)rb[132] << 32);
            std::copy(rb, rb + 130, starts.begin());
            uc.assign(rb + 133, rb + 133 + round + 1);
            if (ovf) throw PgxError{PGX_ERR_CAPACITY, "a body touches more than 127 contact colours"};
            if (uc[round] == 0) break;
            if (round >= MAX_ROUNDS) throw PgxError{PGX_ERR_INVALID, "graph colouring did not converge"};
            batch = 16;
        }
        // rounds actually used: the first whose count of uncoloured manifolds is zero
        int used = round;
        for (int r = 1; r <= round; ++r)
            if (uc[r] == 0) { used = r; break; }
        nColors = (int)(lastKey >> COLOR_KEY_SHIFT) + 1;
        w.lastRounds = used;
        hipLaunchKernelGGL(k_color_rank, dim3(nb), dim3(256), 0, s, M, w.colorPerm.p, w.colorRank.p);
    }
    w.colorStartHost.assign(starts.begin(), starts.begin() + nColors + 1);
    // contact setup, written in solve order
    int cur = w.cacheCur ^ 1, prv = w.cacheCur;
    hipLaunchKernelGGL(k_setup, dim3(nb), dim3(256), 0, s, M, w.manifoldCap, w.colorRank.p, w.mfSrc.p, w.mfTri.p,
                       w.mfKey.p,
                       w.localBits, w.worldColStart.p, w.colOfLocal.p, w.cbody.p, w.cflags.p, w.cmat.p, w.npNum.p,
                       w.npNormal.p, w.npPts.p, w.mfColor.p, w.mfB0.p, w.mfB1.p, w.bpos.p, w.bquat.p, w.dvel.p,
                       w.dang.p, w.dcom.p, w.D, w.mfPrev.p, w.cacheNum[prv].p, w.cacheLp[prv].p, w.manifoldCap,
                       w.cacheKey[cur].p, w.cacheTri[cur].p,
                       w.cacheNum[cur].p, w.cacheLp[cur].p,
                       w.sB.p, w.sA.p, w.sFlags.p, w.sCanon.p, w.sN.p, w.sSoft.p, w.sR.p, w.sWorld.p);
    PGX_LAUNCH_CHECK();
    return nColors;
}

static SubArgs make_args(World& w, int M, float dt) {
    SubArgs a;
    a.M = M; a.Mcap = w.manifoldCap; a.D = w.D;
    a.nColors = (int)w.colorStartHost.size() - 1;
    a.substeps = w.substeps; a.iterations = w.iterations;
    a.h = dt / w.substeps; a.g = w.g;
    a.sB = (const int32_t*)w.sB.p; a.sA = (const int32_t*)w.sA.p; a.sFlags = w.sFlags.p;
    a.colorStart = w.colorCount.p;
    a.sN = w.sN.p; a.sR = w.sR.p; a.sSoft = w.sSoft.p; a.sRow = w.sRow.p; a.sLam = w.sLam.p; a.sMode = w.sMode.p;
    a.bpos = w.bpos.p; a.bquat = w.bquat.p; a.dvel = w.dvel.p; a.dang = w.dang.p;
    a.bvel = w.bvel.p; a.brec = w.brec.p; a.dcom = w.dcom.p; a.dinvI = w.dinvI.p;
    a.pvel = w.pvel.p; a.pang = w.pang.p;
    a.used = w.usedMask.p; a.tickets = w.tickets.p; a.flowErr = w.flowErr.p; a.qDone = w.qDone.p;
    a.barrier = w.passBarrier.p;
    if (w.execMode == EXEC_XPASS) w.xpassCtl.alloc(XPASS_CTL * (size_t)(w.iterations + 1));
    a.xctl = w.xpassCtl.p;
    a.xctlWords = w.execMode == EXEC_XPASS ? XPASS_CTL * (w.iterations + 1) : 0;
    return a;
}

// Largest co-resident grid for the persistent kernel (cached per world).
static int persistent_blocks(World& w) {
    if (w.persistentBlocks > 0) return w.persistentBlocks;
    int perCU = 0, cus = 0;
    PGX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, (const void*)k_step_persistent, 256, 0));
    PGX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, w.device));
    int target = w.persistentBlocksWanted > 0 ? w.persistentBlocksWanted : cus;   // one block per CU by default
    w.persistentBlocks = std::max(1, std::min(target, perCU * cus));
    return w.persistentBlocks;
}

// Grid of the one-launch-per-pass kernel: enough threads for the largest colour in one
// round, at most one workgroup per CU, and never more than can be co-resident.
static int pass_blocks(World& w, int maxColour) {
    if (w.passBlocksMax == 0) {
        int perCU = 0, cus = 0;
        PGX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, (const void*)k_solve_pass, PASS_THREADS, 0));
        PGX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, w.device));
        w.passBlocksMax = std::max(1, std::min(cus, perCU * cus));
    }
    const int want = w.persistentBlocksWanted > 0 ? w.persistentBlocksWanted
                                                  : div_up(2 * std::max(maxColour, 1), PASS_THREADS);
    return std::max(1, std::min(want, w.passBlocksMax));
}

// Grid of the one-XCD pass kernel: about an eighth of it lands on each XCD, so 8 x enough
// workgroups for the largest colour in one round on one XCD, never more than can be
// co-resident, and at most XPASS_MAX_GRID so no XCD's registration byte can overflow.
static int xpass_blocks(World& w, int maxColour) {
    if (w.xpassBlocksMax == 0) {
        int perCU = 0, cus = 0;
        PGX_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, (const void*)k_solve_xpass, XPASS_THREADS, 0));
        PGX_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, w.device));
        w.xpassBlocksMax = std::max(8, std::min(XPASS_MAX_GRID, perCU * cus));
    }
    const int perXcd = w.persistentBlocksWanted > 0 ? div_up(w.persistentBlocksWanted, 8)
                                                    : div_up(2 * std::max(maxColour, 1), XPASS_THREADS);
    return std::max(8, std::min(8 * perXcd, w.xpassBlocksMax));
}

// The start/stop events of one timed k_solve launch (timing mode, first substep of the
// step). They go to hipExtLaunchKernelGGL, which stamps them from the kernel's own dispatch
// packet: the kernel's execution time, without the launch latency an event recorded on the
// stream before and after the launch would add.
static void solve_events(World& w, int color, hipEvent_t* start, hipEvent_t* stop, int colorEnd = 0) {
    int idx = 2 * w.solveEvUsed;
    while ((int)w.solveEv.size() <= idx + 1) {
        hipEvent_t e;
        PGX_HIP(hipEventCreate(&e));
        w.solveEv.push_back(e);
    }
    *start = w.solveEv[idx];
    *stop = w.solveEv[idx + 1];
    if ((int)w.solveEvColor.size() <= w.solveEvUsed) {
        w.solveEvColor.resize(w.solveEvUsed + 1);
        w.solveEvColorEnd.resize(w.solveEvUsed + 1);
    }
    w.solveEvColor[w.solveEvUsed] = color;
    w.solveEvColorEnd[w.solveEvUsed] = colorEnd;
    ++w.solveEvUsed;
}

// per-world passes need every world's dynamic bodies contiguous and their solver
// velocities within one workgroup's LDS
bool sv_world_pass_fits(World& w) {
    if (!w.worldsContiguous) return false;
    if (w.ldsMax == 0) PGX_HIP(hipDeviceGetAttribute(&w.ldsMax, hipDeviceAttributeMaxSharedMemoryPerBlock, w.device));
    return 2 * sizeof(float4) * (size_t)std::max(1, w.maxWorldDyn) <= (size_t)w.ldsMax;
}

// Workgroups of a colour launch over side lanes [b, e) in chunks of bs homed on their XCD
// (homed_chunk): 8 per round, as many rounds as the XCD with the most chunks needs.
static int homed_blocks(int b, int e, int bs) {
    const int q = 256 / bs, period = 8 * q, k0 = b / bs, k1 = (e - 1) / bs + 1;   // chunks [k0, k1)
    auto below = [&](int k, int x) {   // home-x chunks below chunk k
        const int g = k / period, r = k - g * period;
        return q * g + std::min(std::max(r - q * x, 0), q);
    };
    int most = 0;
    for (int x = 0; x < 8; ++x) most = std::max(most, below(k1, x) - below(k0, x));
    return 8 * most;
}

// one colour [b, e) in workgroups of `block` threads; with events, stamped from the
// launch's own dispatch packet
static void launch_solve(int block, bool eager, hipStream_t s, hipEvent_t e0, hipEvent_t e1, const SubArgs& a, int b,
                         int e, int pass) {
    auto go = [&](auto kernel, int bs) {
        const int nb = homed_blocks(2 * b, 2 * e, bs);
        if (e0) hipExtLaunchKernelGGL(kernel, dim3(nb), dim3(bs), 0, s, e0, e1, 0, a, 2 * b, 2 * e, pass);
        else hipLaunchKernelGGL(kernel, dim3(nb), dim3(bs), 0, s, a, 2 * b, 2 * e, pass);
    };
    if (eager) {
        if (block == 256) go(k_solve<256, true>, 256);
        else if (block == 128) go(k_solve<128, true>, 128);
        else go(k_solve<64, true>, 64);
    } else {
        if (block == 256) go(k_solve<256, false>, 256);
        else if (block == 128) go(k_solve<128, false>, 128);
        else go(k_solve<64, false>, 64);
    }
}

// Buffers and launch attributes of the substep loop, set before a graph capture of it (no
// allocation under capture); idempotent.
void sv_presize(World& w) {
    w.tickets.alloc((size_t)(w.iterations + 1) * FLOW_QUEUES);   // k_prepare clears them
    if (w.tune.colorBatch > 0) {
        w.batchLoc.alloc(2 * (size_t)w.manifoldCap);
        w.batchList.alloc(2 * (size_t)w.manifoldCap);
        w.batchTurns.alloc((size_t)BATCH_MAX_GROUPS * BATCH_MAX_TURNS);
        if (!w.batchLdsSet) {
            for (const void* k : {(const void*)k_solve_batch<true>, (const void*)k_solve_batch<false>})
                PGX_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)(4 * sizeof(float4) * BATCH_MAX_MANIFOLDS)));
            w.batchLdsSet = true;
        }
    }
}

void sv_substeps(World& w, int M, float dt) {
    hipStream_t s = w.stream;
    w.solveEvUsed = 0;
    sv_presize(w);
    SubArgs a = make_args(w, M, dt);
    if (w.execMode == EXEC_COOPERATIVE && w.J == 0) {
        int blocks = persistent_blocks(w);
        void* args[] = {&a};
        if (w.timing) PGX_HIP(hipEventRecord(w.ev[6], s));
        PGX_HIP(hipLaunchCooperativeKernel((const void*)k_step_persistent, dim3(blocks), dim3(256), args, 0, s));
        if (w.timing) PGX_HIP(hipEventRecord(w.ev[7], s));
        return;
    }
    int nbP = div_up(2 * (long)std::max(M, 1), 256), nbD = div_up(std::max(w.D, 1), 256);
    int nColors = a.nColors;
    const bool flow = w.execMode == EXEC_FLOW || w.execMode == EXEC_FLOW_XCD;
    FlowArgs f{};
    f.pub = w.flowPub.p;
    if (flow && M > 0) {
        f.xcdScope = w.execMode == EXEC_FLOW_XCD;
        f.nQueues = f.xcdScope ? std::min(w.W, w.nXcd) : 1;
        f.qStart = w.qStart.p;
        f.qList = nullptr;
        if (f.nQueues > 1) {
            // several worlds: a stable partition of the solve order by world % queues
            hipLaunchKernelGGL(k_flow_keys, dim3(div_up(M, 256)), dim3(256), 0, s, M, w.sCanon.p, w.mfKey.p,
                               2 * w.localBits, f.nQueues, w.colorKeys.p, w.qList.p);
            radix_sort_u64(s, w.colorKeys.p, w.qList.p, M, 4, w.sortT);
            hipLaunchKernelGGL(k_flow_starts, dim3(1), dim3(64), 0, s, M, f.nQueues, w.colorKeys.p, w.qStart.p);
            f.qList = w.qList.p;
        } else {
            hipLaunchKernelGGL(k_flow_identity, dim3(1), dim3(64), 0, s, M, f.nQueues, w.qStart.p);
        }
        PGX_LAUNCH_CHECK();
    }
    // per-world passes: the (colour, world) runs once per step
    const bool worlds = w.execMode == EXEC_WORLDS && sv_world_pass_fits(w) && M > 0;
    WorldPassArgs wp{};
    if (worlds) {
        wp.W = w.W; wp.nColors = nColors; wp.wDyn = w.wDyn.p;
        const size_t cells = (size_t)std::max(nColors, 1) * w.W;
        w.wcS.alloc(cells); w.wcE.alloc(cells);
        fill_i32(s, w.wcS.p, 0, (int)cells);
        fill_i32(s, w.wcE.p, 0, (int)cells);
        hipLaunchKernelGGL(k_world_ranges, dim3(div_up(M, 256)), dim3(256), 0, s, M, w.W, w.sFlags.p, w.sWorld.p,
                           w.wcS.p, w.wcE.p);
        PGX_LAUNCH_CHECK();
        wp.wcS = w.wcS.p; wp.wcE = w.wcE.p;
    }
    // worlds by size: each size class in its own launch, with LDS for its largest world
    const size_t worldLds[2] = {2 * sizeof(float4) * (size_t)WORLD_SMALL,
                                2 * sizeof(float4) * (size_t)std::max(1, w.maxWorldDyn)};
    if (worlds && worldLds[1] > 65536)
        PGX_HIP(hipFuncSetAttribute((const void*)k_world_pass, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)worldLds[1]));
    w.lastQueues = flow && M > 0 ? f.nQueues : 0;
    w.lastFlowPasses = flow && M > 0 ? w.substeps * (w.iterations + 1) : 0;
    // Waves of the dependency-driven pass: all manifolds at once while they fit the chip; of more,
    // two waves a SIMD with 64 manifolds each in turn, since what more waves would solve next
    // waits for what these hold, and their polling is in its way. 4,096 worlds, 1.4 M manifolds:
    // 405 M body-substeps/s; 317 with 8,192 waves of 32 manifolds, 305 of 64, 343 with 2,048 of 32.
    // On XCD queues, 64 workgroups per XCD: 348, and 321 with 32 manifolds a wave.
    const bool resident = M <= FLOW_RESIDENT;
    f.take = resident ? WAVE / 2 : WAVE;
    const int flowBlocks = f.xcdScope ? 64 * w.nXcd : resident ? div_up(2 * (long)std::max(M, 1), 256) : 512;
    // launch groups of the colour passes: (first colour, end colour, batched run index + 1);
    // a run holds consecutive colours of at most colorBatch manifolds each, at most
    // BATCH_MAX_MANIFOLDS in all (its bodies' velocities fit in LDS), two colours or more
    std::vector<int3> groups;
    BatchGroups bg{};
    for (int c = 0; c < nColors;) {
        const int n = w.colorStartHost[c + 1] - w.colorStartHost[c];
        if (w.tune.colorBatch > 0 && n <= w.tune.colorBatch && bg.n < BATCH_MAX_GROUPS) {
            int c1 = c + 1;
            while (c1 < nColors && w.colorStartHost[c1 + 1] - w.colorStartHost[c1] <= w.tune.colorBatch &&
                   w.colorStartHost[c1 + 1] - w.colorStartHost[c] <= BATCH_MAX_MANIFOLDS)
                ++c1;
            if (c1 - c >= 2) {
                bg.S[bg.n] = w.colorStartHost[c];
                bg.E[bg.n] = w.colorStartHost[c1];
                bg.c0[bg.n] = c;
                bg.c1[bg.n] = c1;
                bg.turns[bg.n] = 0;
                for (int k = c; k < c1; ++k)
                    bg.turns[bg.n] += div_up(2 * (w.colorStartHost[k + 1] - w.colorStartHost[k]), BATCH_LANES);
                groups.push_back(make_int3(c, c1, ++bg.n));
                c = c1;
                continue;
            }
        }
        if (n > 0) groups.push_back(make_int3(c, c + 1, 0));
        ++c;
    }
    if (bg.n > 0) {   // the runs' body slots, fixed for the step
        sv_presize(w);
        hipLaunchKernelGGL(k_batch_map, dim3(bg.n), dim3(BATCH_MAP_THREADS), 0, s, bg, a.sB, w.batchLoc.p,
                           w.batchList.p, a.colorStart, w.batchTurns.p);
        PGX_LAUNCH_CHECK();
    }
    int passIndex = 0;
    const bool onePass = w.execMode == EXEC_PASS && M > 0 && nColors > 0;
    const bool xcdPass = w.execMode == EXEC_XPASS && M > 0 && nColors > 0;
    int passGrid = 0;
    if (onePass || xcdPass) {
        int maxColour = 0;
        for (int c = 0; c < nColors; ++c) maxColour = std::max(maxColour, w.colorStartHost[c + 1] - w.colorStartHost[c]);
        passGrid = onePass ? pass_blocks(w, maxColour) : xpass_blocks(w, maxColour);
    }
    auto pass = [&](bool rec, int flags) {
        const int p = passIndex++;
        if (p == 0) flags |= PASS_FIRST;
        if (M == 0) return;
        if (xcdPass) {
            int nc = nColors;
            int32_t* ctl = w.xpassCtl.p + XPASS_CTL * p;
            void* args[] = {&a, &nc, &flags, &ctl};
            hipEvent_t e0 = nullptr, e1 = nullptr;
            if (rec) {
                solve_events(w, -1, &e0, &e1);
                PGX_HIP(hipEventRecord(e0, s));
            }
            PGX_HIP(hipLaunchCooperativeKernel((const void*)k_solve_xpass, dim3(passGrid), dim3(XPASS_THREADS), args,
                                               0, s));
            if (rec) PGX_HIP(hipEventRecord(e1, s));
            return;
        }
        if (onePass) {
            // barriers of this substep so far: (nColors - 1) per earlier pass, each counted
            // once per workgroup; the count is cleared by k_prepare
            int base = p * (nColors - 1) * passGrid;
            int nc = nColors;
            void* args[] = {&a, &nc, &flags, &base};
            hipEvent_t e0 = nullptr, e1 = nullptr;
            if (rec) {
                solve_events(w, -1, &e0, &e1);
                PGX_HIP(hipEventRecord(e0, s));
            }
            PGX_HIP(hipLaunchCooperativeKernel((const void*)k_solve_pass, dim3(passGrid), dim3(PASS_THREADS), args, 0,
                                               s));
            if (rec) PGX_HIP(hipEventRecord(e1, s));
            return;
        }
        if (flow) {
            f.index = p; f.pass = flags;
            f.epoch = ++w.flowEpoch;
            if (rec) {
                hipEvent_t e0, e1;
                solve_events(w, -1, &e0, &e1);
                hipExtLaunchKernelGGL(k_solve_flow, dim3(flowBlocks), dim3(256), 0, s, e0, e1, 0, a, f);
            } else {
                hipLaunchKernelGGL(k_solve_flow, dim3(flowBlocks), dim3(256), 0, s, a, f);
            }
            return;
        }
        if (worlds) {
            hipEvent_t e0 = nullptr, e1 = nullptr;
            if (rec) solve_events(w, -1, &e0, &e1);
            for (int k = 0; k < 2; ++k) {
                const int nw = (int)w.worldListHost[k].size();
                if (!nw) continue;
                WorldPassArgs q = wp;
                q.list = w.worldList[k].p;
                // the events bracket both launches: the first stamps the start, the last the end
                const bool first = k == 0 || w.worldListHost[0].empty(), last = k == 1 || w.worldListHost[1].empty();
                if (rec && (first || last))
                    hipExtLaunchKernelGGL(k_world_pass, dim3(nw), dim3(WORLD_THREADS), worldLds[k], s,
                                          first ? e0 : nullptr, last ? e1 : nullptr, 0, a, q, flags);
                else
                    hipLaunchKernelGGL(k_world_pass, dim3(nw), dim3(WORLD_THREADS), worldLds[k], s, a, q, flags);
            }
            return;
        }
        // one launch per colour (a colour's manifolds share no dynamic body), runs of small
        // colours in one single-workgroup launch
        for (const int3& g : groups) {
            if (g.z) {
                const int q = g.z - 1;
                // 2 bodies per manifold at most
                const size_t lds = 4 * sizeof(float4) * (size_t)(bg.E[q] - bg.S[q]);
                const int2* turns = w.batchTurns.p + (size_t)BATCH_MAX_TURNS * q;
                auto* kernel = (flags & PASS_FIRST) ? k_solve_batch<true> : k_solve_batch<false>;
                if (rec) {   // a run of colours [g.x, g.y), stamped from its dispatch packet
                    hipEvent_t e0, e1;
                    solve_events(w, g.x, &e0, &e1, g.y);
                    hipExtLaunchKernelGGL(kernel, dim3(1), dim3(BATCH_THREADS), lds, s, e0, e1, 0, a, bg.S[q],
                                          bg.E[q], bg.turns[q], turns, w.batchLoc.p, w.batchList.p, flags);
                } else {
                    hipLaunchKernelGGL(kernel, dim3(1), dim3(BATCH_THREADS), lds, s, a, bg.S[q], bg.E[q],
                                       bg.turns[q], turns, w.batchLoc.p, w.batchList.p, flags);
                }
                continue;
            }
            const int c = g.x, b = w.colorStartHost[c], e = w.colorStartHost[c + 1];
            hipEvent_t e0 = nullptr, e1 = nullptr;
            if (rec) solve_events(w, c, &e0, &e1);
            launch_solve(w.tune.solveBlock, e - b <= w.tune.eagerMax, s, e0, e1, a, b, e, flags);
        }
    };
    jt_step_setup(w);
    hipLaunchKernelGGL(k_integrate_velocities, dim3(nbD), dim3(256), 0, s, a);
    for (int sub = 0; sub < w.substeps; ++sub) {
        const bool rec = w.timing && sub == 0;
        passIndex = 0;
        // rows + preSolve of the contacts (the velocities were integrated before the first
        // substep and by the write-back before each other one); then the joint rows, whose
        // preSolve follows the contacts' (src/Physecs.cpp:430-479)
        if (M > 0) hipLaunchKernelGGL(k_prepare, dim3(nbP), dim3(256), 0, s, a, sub);
        jt_update(w, a.h);
        jt_colors(w, a.h, 0, false);
        for (int it = 0; it < w.iterations; ++it) {
            pass(rec, PASS_BIAS);
            jt_colors(w, a.h, 1, it == 0);   // joint colours after the contacts (Physecs.cpp:482-490)
        }
        hipLaunchKernelGGL(k_integrate_positions, dim3(nbD), dim3(256), 0, s, a);
        pass(rec, PASS_SKIP_SOFT | PASS_LAST);
        hipLaunchKernelGGL(k_writeback, dim3(nbD), dim3(256), 0, s, a, sub + 1 < w.substeps ? 1 : 0);
        PGX_LAUNCH_CHECK();
    }
}

// Algorithmic bytes of a contact pass over so many points and manifolds, both sides dynamic,
// averaged over a substep's passes. Per point 7 rows of 16 B, and the lambdas, 8 B read but in
// the first pass and written but in the last; per manifold its mode, normal, friction and
// bodies (28 B) and both bodies' solver v and w, read and written (128 B).
double sv_pass_bytes(const World& w, double points, double manifolds) {
    return (112.0 + 16.0 * w.iterations / (w.iterations + 1)) * points + 156.0 * manifolds;
}

// Algorithmic bytes of one step's substep loop. Rows: per manifold both bodies' records (7
// fields of 16 B each), bodies, flags, normal and softness read, the mode written; per point
// two anchors of 16 B read, 7 rows of 16 B written. Per body: velocity integration with the
// write-back before it (336 B), position integration (144 B).
double sv_step_bytes(const World& w, int M, long points) {
    const double N = w.D, C = (double)points;
    return w.substeps * (264.0 * M + 144.0 * C + (w.iterations + 1) * sv_pass_bytes(w, C, M) + 480.0 * N);
}

void sv_finish_step(World& w, int M) {
    // contact cache of this step becomes the previous one (Physecs.cpp:553)
    w.cacheCur ^= 1;
    w.cacheCount[w.cacheCur] = M;
    bp_compute_bounds(w, true);
}

}  // namespace pgx
