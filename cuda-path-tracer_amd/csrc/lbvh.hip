// LBVH construction on gfx950 (reference: CUDA::BVHBuilder::build,
// BVHBuilder.cu:207-269, after Karras 2012), for one scene or for a batch of
// scenes at once.  Scenes are contiguous segments [off[s], off[s+1]) of the
// triangle array; every array below is indexed by global leaf slot.  The
// parity dump derives the reference's node numbers, child and parent words.
//
//   k_morton        30-bit Morton key (the scene's box) + index + scene id,
//                   and the first sort pass's per-tile digit counts
//   k_sort_hist     \
//   k_sort_rowscan   } LSD radix sort, 10-bit digits, stable: 3 passes over
//   k_sort_scatter  /  the 30-bit key, each scene of a batch on its own or,
//                      with many small ones, all together and then 1-2
//                      passes over the scene id (wave64 ballot match + LDS
//                      staging per 4096-key tile)
//   k_tree_leaves   sorted triangle records, then the radix tree and its boxes
//                   bottom-up inside each 1024-leaf block (LDS, workgroup
//                   scope); each node's traversal record is written whole by
//                   the thread that completes it
//   k_tree_merge    the same over the subtrees that 16 blocks left open, level
//                   by level until none is
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>

#include "context.hpp"
#include "devmath.hpp"
#include "traverse.hpp"

namespace pt {
namespace {

constexpr int kSortTile = 4096;                                // keys per sort tile
constexpr int kDigitBits = 10;                                 // 3 passes over a 30-bit key
constexpr uint32_t kRadix = 1u << kDigitBits;                  // 1024 digits
constexpr int kScatterThreads = 512;                           // scatter: 8 keys per thread, 8 waves per tile
// A segment (see there) of at most this many tiles needs no scan launch: its
// scatter workgroups add up the tiles' counts themselves, all loads in flight
// together.  Soups of 17 / 25 / 32 / 64 tiles build in 87.6 / 91.9 / 94.1 / 111.3
// us so, in 94.1 / 97.9 / 97.4 / 105.3 with the scan.
constexpr uint32_t kFewTiles = 32;
// Scenes of a batch are sorted as segments of their own, which saves the passes
// over the scene id, unless that takes too many half-empty tiles: at most
// kSpareTiles + 4 per tile of an unsegmented sort.  64 scenes of 100 triangles
// build in 54 us (78 by scene passes), 1,000 in 91 (109), 2,000 in 137 (138),
// 4,000 in 237 (160); 2,000 scenes of 500 in 192 (209), 1,000 of 2,500 in 280
// (463), 64 of 1,024 .. 262,144 in 345 (447).
constexpr uint32_t kSpareTiles = 1536;
// The tree is built bottom-up, boxes included, in levels: one workgroup per
// block of kLeafBlock sorted leaves, then one per kFanIn blocks' open subtrees,
// and so on (see the tree section).
constexpr uint32_t kLeafBlock = 1024;
constexpr uint32_t kFanIn = 16;
// Open subtrees of a block: each hangs off a node whose leaf range crosses the
// block's first or last boundary, and a boundary is crossed only by the <= 62
// ancestors of its two leaves' lowest common ancestor.  (About 20 in practice.)
constexpr uint32_t kOpenCap = 128;
constexpr uint32_t kMergeCap = kFanIn * kOpenCap;
constexpr uint32_t kMergeThreads = 512;

// ---- Morton keys ------------------------------------------------------------

__device__ __forceinline__ uint32_t spread10(uint32_t a) {
    a &= 0x3FFu;
    a = (a | (a << 16)) & 0x030000FFu;
    a = (a | (a << 8)) & 0x0300F00Fu;
    a = (a | (a << 4)) & 0x030C30C3u;
    a = (a | (a << 2)) & 0x09249249u;
    return a;
}

// quantize (math_util.h:10-13) with CUDA's saturating float->int conversion.
__device__ __forceinline__ uint32_t quantize1024(float x) {
    float s = x * 1024.0f;
    if (!(s == s)) return 0u;
    if (s >= 1023.0f) return 1023u;
    if (s < 1.0f) return 0u;
    return static_cast<uint32_t>(static_cast<int32_t>(s));
}

// Sort tiles.  A segment is a range of slots sorted on its own: each scene
// (table: an entry for every tile), or all slots (no table).
struct Segment {
    uint32_t start, end;  // slots
    uint32_t id;          // scene
    uint32_t first_tile;
};
__device__ __forceinline__ Segment segment_of_tile(const uint4* __restrict__ table, uint32_t n, uint32_t tile) {
    if (table == nullptr) return Segment{0u, n, 0u, 0u};
    const uint4 t = table[tile];
    return Segment{t.x, t.y, t.z, t.w};
}
__device__ __forceinline__ uint32_t tile_base(const Segment& s, uint32_t tile) {
    return s.start + (tile - s.first_tile) * kSortTile;
}
__device__ __forceinline__ uint32_t tile_count(const Segment& s) {
    return (s.end - s.start + kSortTile - 1u) / kSortTile;
}

// Scene of leaf slot i: the last s with off[s] <= i (off has nscenes + 1 entries).
__device__ __forceinline__ uint32_t scene_of_slot(const uint32_t* __restrict__ off, uint32_t nscenes,
                                                  uint32_t i) {
    uint32_t lo = 0, hi = nscenes - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (off[mid] <= i) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// morton_encoder (BVHBuilder.cu:12-32): centroid ((v0 + v1) + v2) / 3, mapped
// into the scene's enclosing box with invScale computed on the host
// (box[6*s..] = min.xyz, invScale.xyz).  One workgroup per sort tile, which also
// counts the tile's first-pass digits (key bits 0-9) into its row of tile_hist --
// the first sort pass then starts at the scan.  Also sets every scene's root word
// to kInvalid, for the scenes whose tree writes none, and clears `strict`.
constexpr int kMortonThreads = 1024;

__global__ __launch_bounds__(kMortonThreads) void k_morton(const pt_triangle* __restrict__ tris, uint32_t n,
                                                           const uint32_t* __restrict__ off, uint32_t nscenes,
                                                           const float* __restrict__ box,
                                                           const uint4* __restrict__ table,
                                                           uint2* __restrict__ pairs,
                                                           uint32_t* __restrict__ scene_of,
                                                           uint32_t* __restrict__ tile_hist,
                                                           uint32_t* __restrict__ root_word,
                                                           uint32_t* __restrict__ strict) {
    __shared__ uint32_t h[kRadix];
    const uint32_t tid = threadIdx.x;
    if (blockIdx.x == 0 && tid == 0) *strict = 0u;
    for (uint32_t s = blockIdx.x * kMortonThreads + tid; s < nscenes; s += gridDim.x * kMortonThreads) root_word[s] = kInvalid;
    for (uint32_t d = tid; d < kRadix; d += kMortonThreads) h[d] = 0u;
    __syncthreads();
    const Segment seg = segment_of_tile(table, n, blockIdx.x);
    const uint32_t base = tile_base(seg, blockIdx.x);
#pragma unroll
    for (int r = 0; r < kSortTile / kMortonThreads; ++r) {
        const uint32_t i = base + r * kMortonThreads + tid;
        if (i >= seg.end) break;
        const uint32_t sc = table != nullptr ? seg.id : scene_of_slot(off, nscenes, i);
        const float* bx = box + 6 * static_cast<size_t>(sc);
        const float* t = reinterpret_cast<const float*>(tris + i);
        float cx = ((t[0] + t[3]) + t[6]) / 3.0f;
        float cy = ((t[1] + t[4]) + t[7]) / 3.0f;
        float cz = ((t[2] + t[5]) + t[8]) / 3.0f;
        uint32_t qx = quantize1024((cx - bx[0]) * bx[3]);
        uint32_t qy = quantize1024((cy - bx[1]) * bx[4]);
        uint32_t qz = quantize1024((cz - bx[2]) * bx[5]);
        const uint32_t key = spread10(qx) | (spread10(qy) << 1) | (spread10(qz) << 2);
        pairs[i] = make_uint2(key, i);
        scene_of[i] = sc;
        atomicAdd(&h[key & (kRadix - 1u)], 1u);
    }
    __syncthreads();
    for (uint32_t d = tid; d < kRadix; d += kMortonThreads)
        tile_hist[static_cast<size_t>(blockIdx.x) * kRadix + d] = h[d];
}

// ---- radix sort ---------------------------------------------------------------

// Digit of an element: bits [shift, shift+10) of its key, or -- in the
// batched build's last passes -- of the scene id of its original slot.
template <bool BY_SCENE>
__device__ __forceinline__ uint32_t sort_digit(uint32_t k, uint32_t v,
                                               const uint32_t* __restrict__ scene_of, int shift) {
    return ((BY_SCENE ? scene_of[v] : k) >> shift) & (kRadix - 1u);
}

// Per-tile digit histogram: tile_hist[tile * kRadix + digit] (one contiguous
// row per tile).
constexpr int kHistThreads = 1024;

template <bool BY_SCENE>
__global__ __launch_bounds__(kHistThreads) void k_sort_hist(const uint2* __restrict__ pairs,
                                                            const uint32_t* __restrict__ scene_of,
                                                            const uint4* __restrict__ table,
                                                            uint32_t n, int shift,
                                                            uint32_t* __restrict__ tile_hist) {
    __shared__ uint32_t h[kRadix];
    const int tid = threadIdx.x;
    for (int d = tid; d < static_cast<int>(kRadix); d += kHistThreads) h[d] = 0;
    __syncthreads();
    const Segment seg = segment_of_tile(table, n, blockIdx.x);
    const uint32_t base = tile_base(seg, blockIdx.x);
#pragma unroll
    for (int r = 0; r < kSortTile / kHistThreads; ++r) {
        uint32_t i = base + r * kHistThreads + tid;
        if (i < seg.end) {
            const uint2 p = pairs[i];
            atomicAdd(&h[sort_digit<BY_SCENE>(p.x, p.y, scene_of, shift)], 1u);
        }
    }
    __syncthreads();
    for (int d = tid; d < static_cast<int>(kRadix); d += kHistThreads)
        tile_hist[static_cast<size_t>(blockIdx.x) * kRadix + d] = h[d];
}

// Exclusive scan of each digit's counts over a segment's tiles (in place) and
// the digit's total, for segments of more than kFewTiles tiles (scans: first and
// past-last tile of each; none: all tiles).  Their totals' row is first_tile /
// (kFewTiles + 1), which no two of them share.  One workgroup per segment and 64
// digits: lane = digit, so every load
// and store of a tile's 64 counts is one contiguous 256-byte access; the 16
// waves split the tiles into 16 ranges, and each wave's range starts at the
// sum of the earlier ranges.
constexpr int kScanDigits = 64;
constexpr int kScanWaves = 16;

__global__ __launch_bounds__(kScanWaves * 64) void k_sort_rowscan(uint32_t* __restrict__ tile_hist,
                                                                  uint32_t num_tiles,
                                                                  const uint2* __restrict__ scans,
                                                                  uint32_t* __restrict__ digit_total) {
    __shared__ uint32_t s_part[kScanWaves][kScanDigits];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const uint32_t seg = blockIdx.x / (kRadix / kScanDigits);
    const uint32_t d = blockIdx.x % (kRadix / kScanDigits) * kScanDigits + lane;
    const uint32_t first = scans != nullptr ? scans[seg].x : 0u;
    const uint32_t last = scans != nullptr ? scans[seg].y : num_tiles;
    const uint32_t per = (last - first + kScanWaves - 1) / kScanWaves;
    const uint32_t t0 = min(last, first + wave * per), t1 = min(last, t0 + per);
    // Loads in batches of kScanBatch, issued together (the counts come from
    // other XCDs' writes: each load is a far round trip).  The first batch
    // stays in registers for the second sweep (up to 256 tiles, 2^20 keys,
    // that is all of it).
    constexpr uint32_t kScanBatch = 16;
    uint32_t v0[kScanBatch];
#pragma unroll
    for (uint32_t k = 0; k < kScanBatch; ++k)
        v0[k] = t0 + k < t1 ? tile_hist[static_cast<size_t>(t0 + k) * kRadix + d] : 0u;
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanBatch; ++k) sum += v0[k];
    for (uint32_t t = t0 + kScanBatch; t < t1; t += kScanBatch) {
        uint32_t v[kScanBatch];
#pragma unroll
        for (uint32_t k = 0; k < kScanBatch; ++k)
            v[k] = t + k < t1 ? tile_hist[static_cast<size_t>(t + k) * kRadix + d] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kScanBatch; ++k) sum += v[k];
    }
    s_part[wave][lane] = sum;
    __syncthreads();
    uint32_t run = 0;
    for (int w = 0; w < wave; ++w) run += s_part[w][lane];
#pragma unroll
    for (uint32_t k = 0; k < kScanBatch; ++k) {
        if (t0 + k < t1) tile_hist[static_cast<size_t>(t0 + k) * kRadix + d] = run;
        run += v0[k];
    }
    for (uint32_t t = t0 + kScanBatch; t < t1; t += kScanBatch) {
        uint32_t v[kScanBatch];
#pragma unroll
        for (uint32_t k = 0; k < kScanBatch; ++k)
            v[k] = t + k < t1 ? tile_hist[static_cast<size_t>(t + k) * kRadix + d] : 0u;
#pragma unroll
        for (uint32_t k = 0; k < kScanBatch; ++k) {
            if (t + k < t1) tile_hist[static_cast<size_t>(t + k) * kRadix + d] = run;
            run += v[k];
        }
    }
    if (wave == kScanWaves - 1) digit_total[static_cast<size_t>(first / (kFewTiles + 1u)) * kRadix + d] = run;
}

// Block-wide exclusive scan of one value per thread over WAVES waves;
// `total` receives the block sum.  Contains two barriers.
template <int WAVES>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* s_w, uint32_t& total) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        uint32_t y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) s_w[wave] = x;
    __syncthreads();
    uint32_t pre = 0, sum = 0;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) {
        const uint32_t w = s_w[k];
        pre += (k < wave) ? w : 0u;
        sum += w;
    }
    total = sum;
    __syncthreads();
    return pre + x - v;
}

// Stable scatter of one 4096-key tile by THREADS threads.  Each wave ranks
// 64 keys at a time against the keys of its chunk so far: lanes holding the
// same digit are found with ten ballots, their order is the popcount of
// lower peer lanes, and a per-wave LDS counter per digit carries the count
// between rounds.  Keys are then staged in LDS in digit order and written
// out in runs.  Thread t owns digits DPT*t .. DPT*t+DPT-1 in the per-digit
// scans.
template <bool BY_SCENE, int THREADS>
__global__ __launch_bounds__(THREADS) void k_sort_scatter(
    const uint2* __restrict__ pairs_in, uint2* __restrict__ pairs_out,
    const uint32_t* __restrict__ scene_of, const uint4* __restrict__ table, uint32_t n, int shift,
    const uint32_t* __restrict__ tile_hist, const uint32_t* __restrict__ digit_total) {
    constexpr int WAVES = THREADS / 64;
    constexpr int KPT = kSortTile / THREADS;  // keys per thread
    constexpr int DPT = kRadix / THREADS;     // digits per thread
    static_assert(KPT * THREADS == kSortTile && DPT * THREADS == static_cast<int>(kRadix), "tile shape");
    // The waves' digit counters, then (once every key has its place) the keys.
    __shared__ uint2 s_pairs[kSortTile];
    static_assert(WAVES * kRadix <= 2 * kSortTile, "the counters fit the keys' memory");
    uint32_t (*s_wc)[kRadix] = reinterpret_cast<uint32_t (*)[kRadix]>(s_pairs);
    __shared__ uint32_t s_dstart[kRadix];
    __shared__ uint32_t s_gbase[kRadix];
    __shared__ uint32_t s_w[WAVES];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
#pragma unroll
    for (int k = 0; k < WAVES; ++k)
#pragma unroll
        for (int j = 0; j < DPT; ++j) s_wc[k][tid + j * THREADS] = 0;
    __syncthreads();

    const uint32_t tile = blockIdx.x;
    const Segment seg = segment_of_tile(table, n, tile);
    const uint32_t base = tile_base(seg, tile);
    const uint32_t count = min(static_cast<uint32_t>(kSortTile), seg.end - base);
    const uint64_t lt = (1ull << lane) - 1ull;

    uint2 pair[KPT];
    uint32_t rk[KPT];
    uint32_t dig[KPT];
#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t li = wave * (KPT * 64) + r * 64 + lane;
        const bool valid = li < count;
        pair[r] = valid ? pairs_in[base + li] : make_uint2(0u, 0u);
    }
    // This thread's digits: the segment's totals, and those of the tiles before
    // (up to kFewTiles tiles, tile_hist still holds each tile's own counts).
    static_assert(DPT == 2, "a thread's two digits are one load");
    uint32_t gt[DPT], before[DPT];
    const uint32_t tiles = tile_count(seg);
    if (tiles <= kFewTiles) {
        const uint2* row = reinterpret_cast<const uint2*>(tile_hist + static_cast<size_t>(seg.first_tile) * kRadix) + tid;
        const uint32_t mine = tile - seg.first_tile;
        gt[0] = gt[1] = before[0] = before[1] = 0u;
#pragma unroll 4
        for (uint32_t t = 0; t < tiles; ++t) {
            const uint2 c = row[static_cast<size_t>(t) * (kRadix / 2)];
            gt[0] += c.x;
            gt[1] += c.y;
            before[0] += t < mine ? c.x : 0u;
            before[1] += t < mine ? c.y : 0u;
        }
    } else {
        const uint2 g2 = reinterpret_cast<const uint2*>(
            digit_total + static_cast<size_t>(seg.first_tile / (kFewTiles + 1u)) * kRadix)[tid];
        const uint2 b2 = reinterpret_cast<const uint2*>(tile_hist + static_cast<size_t>(tile) * kRadix)[tid];
        gt[0] = g2.x;
        gt[1] = g2.y;
        before[0] = b2.x;
        before[1] = b2.y;
    }
#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t li = wave * (KPT * 64) + r * 64 + lane;
        const bool valid = li < count;
        const uint32_t d = valid ? sort_digit<BY_SCENE>(pair[r].x, pair[r].y, scene_of, shift) : 0u;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < kDigitBits; ++b) {
            const bool bit = (d >> b) & 1u;
            const uint64_t bal = __ballot(bit);
            peers &= bit ? bal : ~bal;
        }
        const uint32_t rank = static_cast<uint32_t>(__popcll(peers & lt));
        uint32_t old = 0;
        if (valid) {
            old = s_wc[wave][d];
            if (rank == 0) s_wc[wave][d] = old + static_cast<uint32_t>(__popcll(peers));
        }
        dig[r] = d;
        rk[r] = old + rank;
    }
    __syncthreads();

    // Digits DPT*t ..: offsets of each wave's run, tile-local start, global base.
    uint32_t tot[DPT];
    uint32_t tsum = 0, gsum = 0;
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = DPT * tid + j;
        uint32_t run = 0;
#pragma unroll
        for (int k = 0; k < WAVES; ++k) {  // each digit's words are read and rewritten by its own thread only
            const uint32_t c = s_wc[k][d];
            s_wc[k][d] = run;
            run += c;
        }
        tot[j] = run;
        tsum += tot[j];
        gsum += gt[j];
    }
    uint32_t tmp;
    uint32_t dstart = block_excl_scan<WAVES>(tsum, s_w, tmp);
    uint32_t gpre = seg.start + block_excl_scan<WAVES>(gsum, s_w, tmp);
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
        const int d = DPT * tid + j;
        s_dstart[d] = dstart;
        s_gbase[d] = gpre + before[j];
        dstart += tot[j];
        gpre += gt[j];
    }
    __syncthreads();

#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t li = wave * (KPT * 64) + r * 64 + lane;
        if (li < count) rk[r] += s_dstart[dig[r]] + s_wc[wave][dig[r]];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < KPT; ++r) {
        const uint32_t li = wave * (KPT * 64) + r * 64 + lane;
        if (li < count) s_pairs[rk[r]] = pair[r];
    }
    __syncthreads();
    for (uint32_t i = tid; i < count; i += THREADS) {
        const uint2 p = s_pairs[i];
        const uint32_t d = sort_digit<BY_SCENE>(p.x, p.y, scene_of, shift);
        const uint32_t g = s_gbase[d] + (i - s_dstart[d]);
        pairs_out[g] = p;
    }
}

// ---- tree and boxes -----------------------------------------------------------
//
// The radix tree (BVHBuilder.cu:107-201) and its boxes (:39-98) in one
// bottom-up pass (Apetrei, "Fast and Simple Agglomerative LBVH Construction",
// 2014).  delta(i) is the length of the common prefix of the adjacent sorted
// keys i and i + 1, extended by the scene-local index when they are equal
// (BVHBuilder.cu:116-133), and -1 across a scene's ends.  A finished subtree
// over leaves [lo, hi] is the left child of its parent, which splits after hi,
// if delta(hi) > delta(lo - 1), and the right child, split after lo - 1,
// otherwise (the two differ unless both are -1: the root).  Of the two
// subtrees meeting at a split the one to arrive second unites them.  So no
// node searches the keys for its range and split, no separate pass refits the
// boxes, and the words of both children are at hand where a record is written.
// The reference's node numbers follow from the splits: a left child split off
// after s is node s, a right child node s + 1 (see the dump).
//
// A workgroup does this in LDS for one block of leaves (hand-offs need only
// workgroup scope).  Subtrees whose sibling reaches outside the block are
// written, in leaf order, to the block's open list; the next level's
// workgroup goes on with the lists of kFanIn blocks as its elements, and so on
// until one workgroup has them all.  2^20 soup triangles: the separate tree
// kernel and the refit of three levels took 34 + 57 + 13 + 10 us (the build 194
// us), these 63 + 13 + 15 + 10 (178 us).

struct Box {
    float mnx, mxx, mny, mxy, mnz, mxz;
};

__device__ __forceinline__ Box unite(const Box& a, const Box& b) {
    // leftBBox.unite(rightBBox) (BVHBuilder.cu:85, BBox.cpp:30-36).
    Box o;
    o.mnx = gmin(a.mnx, b.mnx);
    o.mxx = gmax(a.mxx, b.mxx);
    o.mny = gmin(a.mny, b.mny);
    o.mxy = gmax(a.mxy, b.mxy);
    o.mnz = gmin(a.mnz, b.mnz);
    o.mxz = gmax(a.mxz, b.mxz);
    return o;
}

// The whole traversal record of the node with child word w (slot w >> 2, its
// left child's index): both child boxes and both children's own words
// (kInvalid for a leaf), in one 64-byte line.
__device__ __forceinline__ void store_record(float4* nodes, uint32_t w, const Box& lb, const Box& rb, uint32_t wl,
                                             uint32_t wr) {
    float4* rec = nodes + 4 * static_cast<size_t>(w >> 2);
    rec[0] = make_float4(lb.mnx, lb.mxx, lb.mny, lb.mxy);
    rec[1] = make_float4(lb.mnz, lb.mxz, rb.mnx, rb.mxx);
    rec[2] = make_float4(rb.mny, rb.mxy, rb.mnz, rb.mxz);
    rec[3] = make_float4(__uint_as_float(wl), __uint_as_float(wr), 0.0f, 0.0f);
}

__device__ __forceinline__ void store_root(float* root_box, uint32_t* root_word, uint32_t scene, const Box& b,
                                           uint32_t word) {
    float* o = root_box + 6 * static_cast<size_t>(scene);
    o[0] = b.mnx; o[1] = b.mny; o[2] = b.mnz;
    o[3] = b.mxx; o[4] = b.mxy; o[5] = b.mxz;
    root_word[scene] = word;
}

// A block's open subtrees, in leaf order: last leaf, delta there, child word
// (kInvalid: one leaf) and box of each.
struct OpenList {
    uint32_t count;
    uint32_t hi[kOpenCap];
    int32_t delta[kOpenCap];
    uint32_t word[kOpenCap];
    float box[6][kOpenCap];

    __device__ __forceinline__ void put(uint32_t k, uint32_t last_leaf, int32_t d, uint32_t w, const Box& b) {
        hi[k] = last_leaf;
        delta[k] = d;
        word[k] = w;
        box[0][k] = b.mnx; box[1][k] = b.mxx; box[2][k] = b.mny;
        box[3][k] = b.mxy; box[4][k] = b.mnz; box[5][k] = b.mxz;
    }
};

// The elements of one workgroup (leaves or open subtrees) and the subtrees
// waiting for their siblings.  Boundary x lies before element x (boundary CAP
// at most: after the last).  A subtree over elements [e0, e1] waits in slot e1
// as a left child and in slot e0 as a right child, facing its sibling; before
// that the slot belonged to one of its own parts.  Whole waves issue a step's
// instructions until their last lane stops, and those bound the leaf kernel,
// so a step has no branch but its exits and moves a slot as two 16-byte
// accesses.
template <uint32_t CAP>
struct TreeStage {
    float4 lo[CAP];            // min.x, max.x, min.y, max.y
    float4 hi[CAP];            // min.z, max.z, child word, the far end and the delta beyond it (far_word)
    int32_t delta[CAP + 1];    // across boundary x
    uint32_t at[CAP + 1];      // arrivals at boundary x: 1 from the left, 16 from the right
    uint32_t open[CAP];        // slot of an open subtree: 1 a left child, 2 a right child

    static __device__ __forceinline__ uint32_t far_word(uint32_t far, int32_t d) {
        return far | static_cast<uint32_t>(d + 1) << 16;
    }
    __device__ __forceinline__ void put(uint32_t k, const Box& b, uint32_t word, uint32_t fw) {
        lo[k] = make_float4(b.mnx, b.mxx, b.mny, b.mxy);
        hi[k] = make_float4(b.mnz, b.mxz, __uint_as_float(word), __uint_as_float(fw));
    }
    __device__ __forceinline__ Box get(uint32_t k, uint32_t& word, uint32_t& fw) const {
        const float4 l = lo[k], h = hi[k];
        word = __float_as_uint(h.z);
        fw = __float_as_uint(h.w);
        return Box{l.x, l.y, l.z, l.w, h.x, h.y};
    }
};
static_assert(kMergeCap <= 65536, "a slot's far end takes 16 bits");

// Element e's climb.  last_leaf(e): the last leaf of element e.
template <uint32_t CAP, class LastLeaf>
__device__ __forceinline__ void climb(TreeStage<CAP>& S, uint32_t e, Box b, uint32_t word, float4* __restrict__ nodes,
                                      float* __restrict__ root_box, uint32_t* __restrict__ root_word,
                                      const uint32_t* __restrict__ scene_of, LastLeaf last_leaf) {
    uint32_t e0 = e, e1 = e;
    int32_t dl = S.delta[e], dr = S.delta[e + 1u];
    while ((dl & dr) >= 0) {  // until the subtree is a whole scene (both -1)
        const uint32_t left = dr > dl ? 1u : 0u;
        const uint32_t x = left ? e1 + 1u : e0;  // the boundary its sibling lies beyond
        S.put(x - left, b, word, TreeStage<CAP>::far_word(left ? e0 : e1, left ? dl : dr));
        // A wave's LDS accesses are carried out in order, so the slot is written
        // before the arrival counts and read after it without waiting in
        // between; the fences keep the compiler to that order.  At the outer
        // boundaries nobody else arrives.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        const uint32_t before = __hip_atomic_fetch_add(&S.at[x], left ? 1u : 16u, __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_WORKGROUP);
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (before == 0u) return;
        uint32_t sw, sf;
        const Box sb = S.get(x - 1u + left, sw, sf);
        const uint32_t far = sf & 0xffffu;
        const int32_t fard = static_cast<int32_t>(sf >> 16) - 1;
        e0 = left ? e0 : far;
        e1 = left ? far : e1;
        dl = left ? dl : fard;
        dr = left ? fard : dr;
        const Box lb{left ? b.mnx : sb.mnx, left ? b.mxx : sb.mxx, left ? b.mny : sb.mny,
                     left ? b.mxy : sb.mxy, left ? b.mnz : sb.mnz, left ? b.mxz : sb.mxz};
        const Box rb{left ? sb.mnx : b.mnx, left ? sb.mxx : b.mxx, left ? sb.mny : b.mny,
                     left ? sb.mxy : b.mxy, left ? sb.mnz : b.mnz, left ? sb.mxz : b.mxz};
        const uint32_t wl = left ? word : sw, wr = left ? sw : word;
        word = (last_leaf(x - 1u) << 2) | (wl != kInvalid ? 1u : 0u) | (wr != kInvalid ? 2u : 0u);
        store_record(nodes, word, lb, rb, wl, wr);
        b = unite(lb, rb);
    }
    store_root(root_box, root_word, scene_of ? scene_of[last_leaf(e1)] : 0u, b, word);
}

// After a barrier: the subtrees left waiting for a sibling outside.
template <uint32_t CAP>
__device__ __forceinline__ void mark_open(TreeStage<CAP>& S, uint32_t count) {
    for (uint32_t x = threadIdx.x; x <= count; x += blockDim.x) {
        const uint32_t a = S.at[x];
        if (a == 1u) S.open[x - 1u] = 1u;
        else if (a == 16u) S.open[x] = 2u;
    }
    __syncthreads();
}

// One workgroup per kLeafBlock sorted leaves, one thread per leaf: the leaf's
// triangle is gathered through the sort permutation into its 48-byte record
// (the reference instead permutes the 40-byte triangles inside the sort), then
// climbs.  2^20 soup triangles take 63 us: without the climb (gather, a random
// 40-byte read per leaf, and triangle records) 36, the record stores add 14,
// the climb's steps the rest; with the triangles already in order 50.
__global__ __launch_bounds__(kLeafBlock) void k_tree_leaves(
    const pt_triangle* __restrict__ in_tris, const uint2* __restrict__ pairs,
    const uint32_t* __restrict__ off, const uint32_t* __restrict__ scene_of, uint32_t n,
    float4* __restrict__ nodes, float4* __restrict__ tri_recs, float* __restrict__ root_box,
    uint32_t* __restrict__ root_word, uint32_t* __restrict__ strict, OpenList* __restrict__ lists,
    uint32_t* __restrict__ status) {
    __shared__ TreeStage<kLeafBlock> S;
    __shared__ uint32_t s_w[16];
    const uint32_t tid = threadIdx.x;
    const uint32_t base = blockIdx.x * kLeafBlock;
    const uint32_t count = min(kLeafBlock, n - base);
    const uint32_t k = base + tid;
    S.at[tid] = 0u;
    if (tid == 0u) S.at[kLeafBlock] = 0u;
    S.open[tid] = 0u;
    Box b{0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    // delta between leaves i and i + 1 (scene_of null: one scene).
    auto delta_after = [&](uint32_t i) -> int32_t {
        if (i + 1u >= n) return -1;
        uint32_t first = 0u;
        if (scene_of) {
            const uint32_t sc = scene_of[i];
            if (scene_of[i + 1u] != sc) return -1;
            first = off[sc];
        }
        const uint32_t ka = pairs[i].x, kb = pairs[i + 1u].x;
        if (ka == kb) return 32 + __clz(static_cast<int>((i - first) ^ (i + 1u - first)));
        return __clz(static_cast<int>(ka ^ kb));
    };
    if (tid < count) {
        const pt_triangle* t = in_tris + pairs[k].y;
        const V3 v0 = v3(t->v0[0], t->v0[1], t->v0[2]);
        const V3 v1 = v3(t->v1[0], t->v1[1], t->v1[2]);
        const V3 v2 = v3(t->v2[0], t->v2[1], t->v2[2]);
        const uint32_t id = t->id;
        S.delta[tid + 1u] = delta_after(k);
        if (tid == 0u) S.delta[0] = base > 0u ? delta_after(base - 1u) : -1;
        const V3 e1 = sub(v1, v0), e2 = sub(v2, v0);
        tri_recs[3 * static_cast<size_t>(k) + 0] = make_float4(v0.x, v0.y, v0.z, __uint_as_float(id));
        tri_recs[3 * static_cast<size_t>(k) + 1] = make_float4(e1.x, e1.y, e1.z, 0.0f);
        tri_recs[3 * static_cast<size_t>(k) + 2] = make_float4(e2.x, e2.y, e2.z, 0.0f);
        // BBox() then unite({v0, v1, v2}) (BBox.cpp:4-6, 14-24).
        b.mnx = gmin(gmin(gmin(kFltMax, v0.x), v1.x), v2.x);
        b.mny = gmin(gmin(gmin(kFltMax, v0.y), v1.y), v2.y);
        b.mnz = gmin(gmin(gmin(kFltMax, v0.z), v1.z), v2.z);
        b.mxx = gmax(gmax(gmax(-kFltMax, v0.x), v1.x), v2.x);
        b.mxy = gmax(gmax(gmax(-kFltMax, v0.y), v1.y), v2.y);
        b.mxz = gmax(gmax(gmax(-kFltMax, v0.z), v1.z), v2.z);
        if (__builtin_isunordered(b.mnx, b.mxx) || __builtin_isunordered(b.mny, b.mxy) ||
            __builtin_isunordered(b.mnz, b.mxz))
            atomicOr(strict, 1u);
    }
    __syncthreads();
    if (tid < count)
        climb(S, tid, b, kInvalid, nodes, root_box, root_word, scene_of, [&](uint32_t e) { return base + e; });
    __syncthreads();
    mark_open(S, count);
    const uint32_t o = tid < count ? S.open[tid] : 0u;
    uint32_t total;
    const uint32_t pos = block_excl_scan<kLeafBlock / 64>(o ? 1u : 0u, s_w, total);
    OpenList& L = lists[blockIdx.x];
    if (tid == 0u) {
        L.count = min(total, kOpenCap);
        if (total > kOpenCap) raise_status(status, PT_STATUS_REFIT_OVERFLOW);  // bound argued above
    }
    if (o && pos < kOpenCap) {
        uint32_t word, fw;
        const Box ob = S.get(tid, word, fw);
        const uint32_t end = o == 1u ? tid : fw & 0xffffu;
        L.put(pos, base + end, S.delta[end + 1u], word, ob);
    }
}

// One workgroup per kFanIn lists of the level below: their open subtrees as
// elements, in order, climb on; what is still open goes to this level's list.
// Bound by the longest chain of climb steps (19 in a 16-block part of the
// 2^20-triangle soup), each a few LDS round trips, so the fan-in is of little
// weight: 2^20 triangles build in 183 / 178 / 178 / 179 us at 8 / 16 / 32 / 64,
// 2.88M in 376 / 363 / 372 / 379.
__global__ __launch_bounds__(kMergeThreads) void k_tree_merge(const OpenList* __restrict__ in, uint32_t nlists,
                                                              const uint32_t* __restrict__ scene_of,
                                                              float4* __restrict__ nodes,
                                                              float* __restrict__ root_box,
                                                              uint32_t* __restrict__ root_word,
                                                              OpenList* __restrict__ out,
                                                              uint32_t* __restrict__ status) {
    constexpr uint32_t kPer = kMergeCap / kMergeThreads;
    __shared__ TreeStage<kMergeCap> S;
    __shared__ uint32_t s_last[kMergeCap];  // last leaf of element e
    __shared__ uint32_t s_start[kFanIn + 1];
    __shared__ uint32_t s_w[kMergeThreads / 64];
    const uint32_t tid = threadIdx.x;
    const uint32_t k0 = blockIdx.x * kFanIn;
    if (tid < 64u) {  // the lists' places: an exclusive scan of their counts
        const uint32_t c = tid < kFanIn && k0 + tid < nlists ? in[k0 + tid].count : 0u;
        uint32_t x = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, 64);
            if (tid >= static_cast<uint32_t>(o)) x += y;
        }
        if (tid < kFanIn) s_start[tid + 1u] = x;
        if (tid == 0u) s_start[0] = 0u;
    } else if (tid == 64u) {  // before the first list: the level's previous element, or a scene's start
        const uint32_t c = k0 > 0u ? in[k0 - 1u].count : 0u;
        S.delta[0] = c > 0u ? in[k0 - 1u].delta[c - 1u] : -1;
        S.at[0] = 0u;
    }
    __syncthreads();
    const uint32_t count = s_start[kFanIn];
    Box b[kPer];
    uint32_t w[kPer];
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
        const uint32_t e = tid + q * kMergeThreads;
        if (e >= count) continue;
        uint32_t l = 0u;  // the last list that starts at or before e
#pragma unroll
        for (uint32_t h = kFanIn / 2; h > 0u; h >>= 1)
            if (s_start[l + h] <= e) l += h;
        const OpenList& L = in[k0 + l];
        const uint32_t j = e - s_start[l];
        b[q] = Box{L.box[0][j], L.box[1][j], L.box[2][j], L.box[3][j], L.box[4][j], L.box[5][j]};
        w[q] = L.word[j];
        s_last[e] = L.hi[j];
        S.delta[e + 1u] = L.delta[j];
        S.at[e + 1u] = 0u;
        S.open[e] = 0u;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t q = 0; q < kPer; ++q) {
        const uint32_t e = tid + q * kMergeThreads;
        if (e < count) climb(S, e, b[q], w[q], nodes, root_box, root_word, scene_of, [&](uint32_t x) { return s_last[x]; });
    }
    __syncthreads();
    mark_open(S, count);
    OpenList& L = out[blockIdx.x];
    uint32_t kept = 0u;
    for (uint32_t e0 = 0u; e0 < count; e0 += kMergeThreads) {
        const uint32_t e = e0 + tid;
        const uint32_t o = e < count ? S.open[e] : 0u;
        uint32_t total;
        const uint32_t pos = kept + block_excl_scan<kMergeThreads / 64>(o ? 1u : 0u, s_w, total);
        if (o && pos < kOpenCap) {
            uint32_t word, fw;
            const Box ob = S.get(e, word, fw);
            const uint32_t end = o == 1u ? e : fw & 0xffffu;
            L.put(pos, s_last[end], S.delta[end + 1u], word, ob);
        }
        kept += total;
    }
    if (tid == 0u) {
        L.count = min(kept, kOpenCap);
        if (kept > kOpenCap) raise_status(status, PT_STATUS_REFIT_OVERFLOW);  // bound argued above
    }
}

// Parity dump of scene [base, base + n): the reference's arrays in local
// indices, from the records.  The record of the node that splits after leaf s
// sits in slot s; its left child, if internal, is node s, its right child node
// s + 1, and the root is node 0.  First each node's child word and box (min.xyz,
// max.xyz) from its parent's record, and owner[s]: the number of the node that
// splits after s.
__global__ __launch_bounds__(256) void k_dump_nodes(const float4* __restrict__ nodes,
                                                    const uint32_t* __restrict__ root_word,
                                                    const float* __restrict__ root_box, uint32_t base, uint32_t n,
                                                    float* __restrict__ out_boxes, uint32_t* __restrict__ out_children,
                                                    uint32_t* __restrict__ owner) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s + 1 >= n) return;
    const uint32_t lb = base << 2;
    if (s == 0) {
        const uint32_t w = root_word[0] - lb;
        out_children[0] = w;
        owner[w >> 2] = 0u;
        for (int k = 0; k < 6; ++k) out_boxes[k] = root_box[k];
    }
    const float4* rec = nodes + 4 * static_cast<size_t>(base + s);
    const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2], r3 = rec[3];
    const uint32_t wl = __float_as_uint(r3.x), wr = __float_as_uint(r3.y);
    if (wl != kInvalid) {
        out_children[s] = wl - lb;
        owner[(wl - lb) >> 2] = s;
        float* o = out_boxes + 6 * static_cast<size_t>(s);
        o[0] = r0.x; o[1] = r0.z; o[2] = r1.x; o[3] = r0.y; o[4] = r0.w; o[5] = r1.y;
    }
    if (wr != kInvalid) {
        out_children[s + 1] = wr - lb;
        owner[(wr - lb) >> 2] = s + 1;
        float* o = out_boxes + 6 * static_cast<size_t>(s + 1);
        o[0] = r1.z; o[1] = r2.x; o[2] = r2.z; o[3] = r1.w; o[4] = r2.y; o[5] = r2.w;
    }
}

// Then the parents.
__global__ __launch_bounds__(256) void k_dump_parents(const float4* __restrict__ nodes,
                                                      const uint32_t* __restrict__ owner, uint32_t base, uint32_t n,
                                                      uint32_t* __restrict__ out_pl, uint32_t* __restrict__ out_pi) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0) (n == 1 ? out_pl : out_pi)[0] = kInvalid;  // BVHBuilder.cu:224
    if (s + 1 >= n) return;
    const uint2 w = *reinterpret_cast<const uint2*>(nodes + 4 * static_cast<size_t>(base + s) + 3);
    const uint32_t p = owner[s];
    (w.x != kInvalid ? out_pi : out_pl)[s] = p;
    (w.y != kInvalid ? out_pi : out_pl)[s + 1] = p;
}

// Sorted keys, and the permutation in local indices.
__global__ __launch_bounds__(256) void k_dump_pairs(const uint2* __restrict__ pairs, uint32_t base, uint32_t n,
                                                    uint32_t* __restrict__ out_keys, uint32_t* __restrict__ out_perm) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint2 p = pairs[base + i];
    out_keys[i] = p.x;
    out_perm[i] = p.y - base;
}

inline uint32_t div_up(uint64_t a, uint64_t b) { return static_cast<uint32_t>((a + b - 1) / b); }

}  // namespace

BuildTuning& build_tuning() {
    static BuildTuning t;
    return t;
}

void plan_sort(DeviceScene& s, hipStream_t st) {
    const uint32_t nscenes = s.nscenes();
    const uint32_t plain = div_up(s.n, kSortTile);
    uint64_t tiles = 0;
    for (uint32_t k = 0; k < nscenes; ++k) tiles += div_up(s.off_host[k + 1] - s.off_host[k], kSortTile);
    s.sort_plan_host.clear();
    s.sort_segmented = nscenes > 1 && tiles <= kSpareTiles + 4ull * plain;
    if (!s.sort_segmented) {
        s.sort_tiles = plain;
        s.sort_scans = plain > kFewTiles ? 1u : 0u;
        return;
    }
    // An entry per tile, then first and past-last tile of each segment to scan.
    s.sort_tiles = static_cast<uint32_t>(tiles);
    s.sort_scans = 0;
    std::vector<uint32_t>& plan = s.sort_plan_host;
    plan.reserve(4 * tiles);
    std::vector<uint32_t> scans;
    uint32_t t = 0;
    for (uint32_t k = 0; k < nscenes; ++k) {
        const uint32_t a = s.off_host[k], b = s.off_host[k + 1], first = t;
        for (const uint32_t last = first + div_up(b - a, kSortTile); t < last; ++t) plan.insert(plan.end(), {a, b, k, first});
        if (t - first > kFewTiles) {
            scans.insert(scans.end(), {first, t});
            ++s.sort_scans;
        }
    }
    plan.insert(plan.end(), scans.begin(), scans.end());
    s.sort_plan.reserve(plan.size() * 4);
    PT_HIP(hipMemcpyAsync(s.sort_plan.as<void>(), plan.data(), plan.size() * 4, hipMemcpyHostToDevice, st));
}

void build_lbvh(DeviceScene& s, hipStream_t st) {
    DeviceBvh& b = s.bvh;
    const uint32_t n = s.n;
    const uint32_t nscenes = static_cast<uint32_t>(s.off_host.size()) - 1;
    b.n = n;
    b.strict.reserve(sizeof(uint32_t));
    if (n == 0) {
        PT_HIP(hipMemsetAsync(b.strict.as<void>(), 0, sizeof(uint32_t), st));
        return;
    }
    if (n >= (1u << 30)) throw Error(PT_E_INVALID_ARG, "LBVH supports fewer than 2^30 triangles");
    const size_t n4 = static_cast<size_t>(n) * 4;
    b.pairs.reserve(2 * n4);
    b.pairs_alt.reserve(2 * n4);
    b.scene_of.reserve(n4);
    b.nodes.reserve(static_cast<size_t>(n) * 64);
    b.tris.reserve(static_cast<size_t>(n) * 48);
    b.root_box.reserve(static_cast<size_t>(nscenes) * 6 * sizeof(float));
    b.root_word.reserve(static_cast<size_t>(nscenes) * 4);
    const uint32_t num_tiles = s.sort_tiles;
    const uint4* table = s.sort_segmented ? s.sort_plan.as<uint4>() : nullptr;
    const uint2* scans = table ? reinterpret_cast<const uint2*>(table + num_tiles) : nullptr;
    b.tile_hist.reserve(static_cast<size_t>(num_tiles) * kRadix * 4);
    b.digit_total.reserve(static_cast<size_t>(num_tiles / (kFewTiles + 1) + 1) * kRadix * 4);
    // Open lists of every level, one after the other.
    const uint32_t blocks = div_up(n, kLeafBlock);
    size_t nlists = blocks;
    for (uint32_t m = blocks; m > 1; m = div_up(m, kFanIn)) nlists += div_up(m, kFanIn);
    b.open_lists.reserve(nlists * sizeof(OpenList));

    uint2* in = b.pairs.as<uint2>();
    hipLaunchKernelGGL(k_morton, dim3(num_tiles), dim3(kMortonThreads), 0, st, s.tris.as<pt_triangle>(), n,
                       s.off.as<uint32_t>(), nscenes, s.morton_box.as<float>(), table, in,
                       b.scene_of.as<uint32_t>(), b.tile_hist.as<uint32_t>(), b.root_word.as<uint32_t>(),
                       b.strict.as<uint32_t>());
    PT_HIP(hipGetLastError());

    if (n >= 2) {
        uint2* out = b.pairs_alt.as<uint2>();
        // 3 passes over the 30-bit keys; unless the scenes are segments, then the
        // scene id's 10-bit digits (stable: each scene keeps its key order, ties
        // in input order).
        constexpr int kKeyPasses = (30 + kDigitBits - 1) / kDigitBits;
        int scene_passes = 0;
        if (!s.sort_segmented)
            for (uint32_t v = nscenes - 1; v != 0; v >>= kDigitBits) ++scene_passes;
        const int passes = kKeyPasses + scene_passes;
        const uint32_t* sc = b.scene_of.as<uint32_t>();
        uint32_t* hist = b.tile_hist.as<uint32_t>();
        uint32_t* totals = b.digit_total.as<uint32_t>();
        for (int pass = 0; pass < passes; ++pass) {
            const bool by_scene = pass >= kKeyPasses;
            const int shift = kDigitBits * (by_scene ? pass - kKeyPasses : pass);
            // The first pass's counts come from k_morton.
            if (pass > 0) {
                hipLaunchKernelGGL(by_scene ? k_sort_hist<true> : k_sort_hist<false>, dim3(num_tiles), dim3(kHistThreads),
                                   0, st, in, sc, table, n, shift, hist);
            }
            if (s.sort_scans > 0) {
                hipLaunchKernelGGL(k_sort_rowscan, dim3(s.sort_scans * (kRadix / kScanDigits)), dim3(kScanWaves * 64), 0, st,
                                   hist, num_tiles, scans, totals);
            }
            const auto scatter = by_scene ? k_sort_scatter<true, kScatterThreads> : k_sort_scatter<false, kScatterThreads>;
            hipLaunchKernelGGL(scatter, dim3(num_tiles), dim3(kScatterThreads), 0, st, in, out, sc, table, n,
                               shift, hist, totals);
            std::swap(in, out);
        }
        if (passes % 2) {
            // Odd pass count: the result sits in the alternate buffers.
            swap(b.pairs, b.pairs_alt);
        }
        PT_HIP(hipGetLastError());
    }
    const uint32_t* scene_of = nscenes > 1 ? b.scene_of.as<uint32_t>() : nullptr;
    OpenList* lists = b.open_lists.as<OpenList>();
    hipLaunchKernelGGL(k_tree_leaves, dim3(blocks), dim3(kLeafBlock), 0, st, s.tris.as<pt_triangle>(),
                       b.pairs.as<uint2>(), s.off.as<uint32_t>(), scene_of, n,
                       b.nodes.as<float4>(), b.tris.as<float4>(), b.root_box.as<float>(), b.root_word.as<uint32_t>(),
                       b.strict.as<uint32_t>(), lists, s.status.as<uint32_t>());
    for (uint32_t m = blocks; m > 1;) {
        const uint32_t next = div_up(m, kFanIn);
        hipLaunchKernelGGL(k_tree_merge, dim3(next), dim3(kMergeThreads), 0, st, lists, m, scene_of, b.nodes.as<float4>(),
                           b.root_box.as<float>(), b.root_word.as<uint32_t>(), lists + m, s.status.as<uint32_t>());
        lists += m;
        m = next;
    }
    PT_HIP(hipGetLastError());
}

void dump_bvh(DeviceScene& s, uint32_t scene, hipStream_t st, uint32_t* morton, uint32_t* perm,
              uint32_t* children, uint32_t* parents_leaf, uint32_t* parents_internal,
              float* bboxes) {
    const DeviceBvh& b = s.bvh;
    if (scene + 1 >= s.off_host.size()) throw Error(PT_E_INVALID_ARG, "scene index out of range");
    const uint32_t base = s.off_host[scene];
    const uint32_t n = s.off_host[scene + 1] - base;
    if (n == 0) return;
    const size_t m = n - 1;
    DevBuf tmp;
    tmp.reserve(static_cast<size_t>(n) * 6 * 4 + m * 24 + 256);
    uint32_t* t_perm = tmp.as<uint32_t>();
    uint32_t* t_ch = t_perm + n;
    uint32_t* t_pl = t_ch + n;
    uint32_t* t_pi = t_pl + n;
    uint32_t* t_owner = t_pi + n;
    uint32_t* t_keys = t_owner + n;
    float* t_box = reinterpret_cast<float*>(t_keys + n);
    hipLaunchKernelGGL(k_dump_pairs, dim3(div_up(n, 256)), dim3(256), 0, st, b.pairs.as<uint2>(), base, n, t_keys, t_perm);
    if (n > 1) {
        hipLaunchKernelGGL(k_dump_nodes, dim3(div_up(n, 256)), dim3(256), 0, st, b.nodes.as<float4>(),
                           b.root_word.as<uint32_t>() + scene, b.root_box.as<float>() + 6 * static_cast<size_t>(scene),
                           base, n, t_box, t_ch, t_owner);
    }
    hipLaunchKernelGGL(k_dump_parents, dim3(div_up(n, 256)), dim3(256), 0, st, b.nodes.as<float4>(), t_owner, base, n,
                       t_pl, t_pi);
    PT_HIP(hipGetLastError());
    if (morton) PT_HIP(hipMemcpyAsync(morton, t_keys, n * 4ull, hipMemcpyDeviceToHost, st));
    if (perm) PT_HIP(hipMemcpyAsync(perm, t_perm, n * 4ull, hipMemcpyDeviceToHost, st));
    if (parents_leaf) PT_HIP(hipMemcpyAsync(parents_leaf, t_pl, n * 4ull, hipMemcpyDeviceToHost, st));
    if (m > 0) {
        if (children) PT_HIP(hipMemcpyAsync(children, t_ch, m * 4, hipMemcpyDeviceToHost, st));
        if (parents_internal) PT_HIP(hipMemcpyAsync(parents_internal, t_pi, m * 4, hipMemcpyDeviceToHost, st));
        if (bboxes) PT_HIP(hipMemcpyAsync(bboxes, t_box, m * 24, hipMemcpyDeviceToHost, st));
    }
    PT_HIP(hipStreamSynchronize(st));
}

}  // namespace pt
