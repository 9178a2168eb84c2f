// Device primitives and batched maintenance of the labelled adjacency.
//
//   scan_exclusive   device-wide exclusive prefix sum (replaces the reference's CUB
//                    DeviceScan::ExclusiveSum calls, match_gpu.cu:739, 784, ...).
//   batch build      the batch's arcs as a per-vertex sorted delta (replaces BuildTries /
//                    BuildTriesFromEdgeList, match_gpu.cu:302-322, 2296-2344: CUB radix sort + RLE +
//                    scan into a CSR).  Counting sort by source into per-vertex segments, then a
//                    sort of each segment; admission is decided on the way.
//   apply deletions  delete-compact of every touched list (extension; the reference is
//                    insertion-only).
//   apply insertions merge-insert of every touched list, relocating to a larger arena block when
//                    the capacity is exceeded (addTriesToGraph, indexing.cu:76-263; capacity rule
//                    roundCapacities, indexing.cu:46-59, computed with integer arithmetic).
#include "kernels.h"
#include "view.h"

namespace csm {
namespace {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr uint32_t kScanTile = kScanThreads * kScanItems;

template <typename T>
__global__ void __launch_bounds__(kScanThreads) k_scan_tile_sums(const T* in, const uint32_t* n_dev, uint32_t n_max, T* sums) {
    __shared__ unsigned long long sh[kScanThreads / 64];
    const uint32_t n = n_dev ? min(*n_dev, n_max) : n_max;
    const uint32_t base = blockIdx.x * kScanTile;
    if (base >= n && blockIdx.x != 0) { if (threadIdx.x == 0) sums[blockIdx.x] = T(0); return; }
    unsigned long long acc = 0, total;
    for (int k = 0; k < kScanItems; k++) {
        const uint32_t i = base + k * kScanThreads + threadIdx.x;
        if (i < n) acc += in[i];
    }
    block_scan<kScanThreads>(acc, sh, total);
    if (threadIdx.x == 0) sums[blockIdx.x] = static_cast<T>(total);
}

// Thread t of a tile owns its kScanItems consecutive elements: one block scan of the thread sums
// (a scan per row of kScanThreads elements took 10 us for one tile, all of it barriers).
template <typename T>
__global__ void __launch_bounds__(kScanThreads) k_scan_tiles(const T* in, T* out, const uint32_t* n_dev, uint32_t n_max,
                                                              const T* tile_offsets, bool write_total) {
    __shared__ unsigned long long sh[kScanThreads / 64];
    const uint32_t n = n_dev ? min(*n_dev, n_max) : n_max;
    const uint32_t base = blockIdx.x * kScanTile;
    if (base > n) return;
    const unsigned long long carry = tile_offsets ? tile_offsets[blockIdx.x] : T(0);
    const uint32_t i0 = base + threadIdx.x * kScanItems;
    T v[kScanItems];
    unsigned long long sum = 0, total;
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        v[k] = i0 + k < n ? in[i0 + k] : T(0);
        sum += v[k];
    }
    unsigned long long ex = carry + block_scan<kScanThreads>(sum, sh, total);
#pragma unroll
    for (int k = 0; k < kScanItems; k++) {
        if (i0 + k < n || (write_total && i0 + k == n)) out[i0 + k] = static_cast<T>(ex);  // at n: the sum of in[0..n)
        ex += v[k];
    }
}

}  // namespace

template <typename T>
void scan_exclusive(const T* in, T* out, const uint32_t* n_dev, uint32_t n_max, bool write_total, T* scratch, hipStream_t s) {
    // scratch must hold scratch_words_for_scan(n_max) elements of T.
    const uint32_t tiles = (n_max + 1 + kScanTile - 1) / kScanTile;
    if (tiles <= 1) {
        k_scan_tiles<T><<<1, kScanThreads, 0, s>>>(in, out, n_dev, n_max, nullptr, write_total);
        return;
    }
    T* sums = scratch;
    T* sums_scanned = scratch + tiles;
    k_scan_tile_sums<T><<<tiles, kScanThreads, 0, s>>>(in, n_dev, n_max, sums);
    scan_exclusive<T>(sums, sums_scanned, nullptr, tiles, false, scratch + 2 * tiles, s);
    k_scan_tiles<T><<<tiles, kScanThreads, 0, s>>>(in, out, n_dev, n_max, sums_scanned, write_total);
}

uint64_t scan_scratch_elems(uint32_t n_max) {
    uint64_t total = 0;
    uint64_t n = n_max;
    while (true) {
        const uint64_t tiles = (n + 1 + kScanTile - 1) / kScanTile;
        if (tiles <= 1) break;
        total += 2 * tiles;
        n = tiles;
    }
    return total + 16;
}

template void scan_exclusive<uint32_t>(const uint32_t*, uint32_t*, const uint32_t*, uint32_t, bool, uint32_t*, hipStream_t);
template void scan_exclusive<unsigned long long>(const unsigned long long*, unsigned long long*, const uint32_t*, uint32_t, bool,
                                                 unsigned long long*, hipStream_t);

// ---------------------------------------------------------------------------------------------
// Batch build.
// Arcs of update edge k: undirected -> (src, key_to_dst) and (dst, key_to_src) both in direction 0;
// directed -> (src, key_to_dst) in direction 0 and (dst, key_to_src) in direction 1.
namespace {

// Zeroes what a batch counts into: touched, segment and label counters of each direction, results.
__global__ void __launch_bounds__(256) k_batch_begin(BatchScratch w0, BatchScratch w1, uint32_t dirs, uint32_t labels, uint32_t* results,
                                                     uint32_t nresults) {
    const uint32_t i0 = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
    for (uint32_t d = 0; d < dirs; d++) {
        const BatchScratch& w = d ? w1 : w0;
        if (i0 == 0) {
            *w.n_touched = 0;
            *w.n_big = 0;
            *w.cursor = 0;
        }
        for (uint32_t i = i0; i < labels; i += stride) w.label_cur[i] = 0;
    }
    for (uint32_t i = i0; i < nresults; i += stride) results[i] = 0;
}

// Per arc: its rank among its vertex's insertions or deletions (w.rank, by arrival) from one packed
// 64-bit counter per vertex, whose first visitor lists the vertex.  One thread per edge; a block
// collects its new vertices in LDS and reserves their places with one device atomic per tile (atomics
// on one address serialise).
constexpr uint32_t kCountEdges = 2;  // edges per thread of a tile
constexpr uint32_t kCountTile = 256 * kCountEdges;

__global__ void __launch_bounds__(256) k_batch_count(BatchInput b, uint32_t lo, uint32_t n, int dirsel, BatchScratch w) {
    __shared__ uint32_t s_list[2 * kCountTile], s_n, s_base;
    for (uint32_t tile = blockIdx.x * kCountTile; tile < n; tile += gridDim.x * kCountTile) {  // block-uniform
        if (threadIdx.x == 0) s_n = 0;
        __syncthreads();
        uint32_t v[2 * kCountEdges];
        unsigned long long old[2 * kCountEdges];
#pragma unroll
        for (uint32_t e = 0; e < kCountEdges; e++) {
            const uint32_t k = tile + e * 256 + threadIdx.x;
#pragma unroll
            for (uint32_t side = 0; side < 2; side++) {
                old[2 * e + side] = 1;  // not a first visitor
                // directed: direction 0 takes the source arcs (dirsel 1), direction 1 the others (dirsel 2)
                if (k >= n || dirsel == (side ? 1 : 2)) continue;
                const bool del = b.op[lo + k];
                v[2 * e + side] = side ? b.dst[lo + k] : b.src[lo + k];
                old[2 * e + side] = atomicAdd(&w.cnt[v[2 * e + side]], del ? 1ull << 32 : 1ull);
                w.rank[2 * k + side] = static_cast<uint32_t>(del ? old[2 * e + side] >> 32 : old[2 * e + side]);
            }
        }
#pragma unroll
        for (uint32_t e = 0; e < 2 * kCountEdges; e++)
            if (!old[e]) s_list[atomicAdd(&s_n, 1u)] = v[e];
        __syncthreads();
        if (threadIdx.x == 0) s_base = s_n ? atomicAdd(w.n_touched, s_n) : 0u;
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < s_n; i += 256) w.touched[s_base + i] = s_list[i];
        __syncthreads();
    }
}

// Delta segments of the touched vertices.  Any disjoint placement will do, so a block scans its
// tile's counts and reserves its share of both arrays with one atomic on the packed cursor: one
// launch instead of a gather, two device-wide scans and a write (eight).
constexpr uint32_t kSegItems = 4;
__global__ void __launch_bounds__(256) k_batch_segments(BatchScratch w, DevDelta d) {
    __shared__ unsigned long long sh[4], s_base;
    const uint32_t T = *w.n_touched;
    for (uint32_t tile = blockIdx.x * 256 * kSegItems; tile < T; tile += gridDim.x * 256 * kSegItems) {  // block-uniform
        uint32_t v[kSegItems];
        unsigned long long c[kSegItems], sum = 0, total;
#pragma unroll
        for (uint32_t j = 0; j < kSegItems; j++) {
            const uint32_t i = tile + j * 256 + threadIdx.x;
            v[j] = i < T ? w.touched[i] : kNoVertex;
        }
#pragma unroll
        for (uint32_t j = 0; j < kSegItems; j++) {
            c[j] = v[j] != kNoVertex ? w.cnt[v[j]] : 0ull;
            sum += c[j];  // both halves stay under 2^32: a batch has fewer arcs
        }
        unsigned long long at = block_scan<256>(sum, sh, total);
        if (threadIdx.x == 0) s_base = atomicAdd(w.cursor, total);
        __syncthreads();
        at += s_base;
#pragma unroll
        for (uint32_t j = 0; j < kSegItems; j++) {
            if (v[j] != kNoVertex)
                d.seg[v[j]] = make_uint4(static_cast<uint32_t>(at), static_cast<uint32_t>(c[j]), static_cast<uint32_t>(at >> 32),
                                         static_cast<uint32_t>(c[j] >> 32));
            at += c[j];
        }
        __syncthreads();  // s_base is rewritten
    }
}

// Whether `key` is in v's base list of direction dir.
__device__ __forceinline__ bool base_contains(const DevGraph& g, int dir, uint32_t v, uint32_t key) {
    uint32_t lo, hi;
    if (g.sdir[dir] && g.id_bits < 32) {
        base_range(g, dir, v, key >> g.id_bits, lo, hi);
    } else {
        const uint2 a = g.dir[dir].adj[v];
        lo = a.x;
        hi = a.x + a.y;
    }
    return contains_u32(g.arena, lo, hi, key);
}

// Every arc's key to its place in the delta, and the preconditions of the update semantics per arc:
// an inserted arc must not be in the list (this also catches a delete and re-insert of one arc in the
// same batch), a deleted arc must be.  An undirected graph holds both arcs of an edge or neither:
// the source's list answers for both.  adm[1] |= a violation.
__global__ void __launch_bounds__(256) k_batch_scatter(DevGraph g, BatchInput b, uint32_t lo, uint32_t n, int dirsel, int dir, BatchScratch w,
                                                       unsigned long long* adm) {
    const DevDelta d = g.delta[dir];
    bool bad = false;
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k < n; k += gridDim.x * blockDim.x) {
        const bool del = b.op[lo + k];
        uint32_t* const out = del ? d.del : d.ins;
        const uint32_t sv = b.src[lo + k], dv = b.dst[lo + k], kf = b.key_fwd[lo + k], kb = b.key_bwd[lo + k];
        if (dirsel != 2) {
            const uint4 s = d.seg[sv];
            out[(del ? s.z : s.x) + w.rank[2 * k]] = kf;
        }
        if (dirsel != 1) {
            const uint4 s = d.seg[dv];
            out[(del ? s.z : s.x) + w.rank[2 * k + 1]] = kb;
        }
        bad = bad || (dirsel == 2 ? base_contains(g, dir, dv, kb) : base_contains(g, dir, sv, kf)) != del;
    }
    if (__ballot(bad) != 0 && lane_id() == 0) atomicOr(reinterpret_cast<uint32_t*>(&adm[1]), 1u);
}

// Sorting network with every comparator ascending ("mirror" first step per stage), so elements
// past n behave as +infinity padding and are never touched: valid for any n <= N = 2^k.  The sorts
// return whether a key occurs twice (in some lane).
constexpr uint32_t kSortLane = 8;
__device__ __forceinline__ bool lane_sort(uint32_t* a, uint32_t n) {
    // n <= kSortLane, one segment per lane: odd-even merge network in registers
    uint32_t v[kSortLane];
#pragma unroll
    for (uint32_t i = 0; i < kSortLane; i++) v[i] = i < n ? a[i] : 0xFFFFFFFFu;
#pragma unroll
    for (uint32_t k = 2; k <= kSortLane; k <<= 1) {
#pragma unroll
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
            for (uint32_t i = 0; i < kSortLane; i++) {
                const uint32_t p = (j == (k >> 1)) ? (i ^ (k - 1)) : (i ^ j);
                if (p > i) {
                    const uint32_t x = v[i], y = v[p];
                    v[i] = min(x, y);
                    v[p] = max(x, y);
                }
            }
        }
    }
    bool twice = false;
#pragma unroll
    for (uint32_t i = 0; i < kSortLane; i++) {
        if (i < n) a[i] = v[i];
        if (i > 0 && i < n && v[i] == v[i - 1]) twice = true;
    }
    return twice;
}

__device__ bool wave_sort_small(uint32_t* a, uint32_t n) {
    // n <= 64: one element per lane, exchanges through shuffles.
    const uint32_t lane = lane_id();
    uint32_t v = lane < n ? a[lane] : 0xFFFFFFFFu;
    for (uint32_t k = 2; k <= 64; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            const uint32_t partner = (j == (k >> 1)) ? (lane ^ (k - 1)) : (lane ^ j);
            const uint32_t pv = __shfl(v, static_cast<int>(partner), 64);
            v = lane < partner ? min(v, pv) : max(v, pv);
        }
    }
    if (lane < n) a[lane] = v;
    const uint32_t before = __shfl_up(v, 1, 64);
    return lane > 0 && lane < n && before == v;
}

__device__ bool wave_sort_lds(uint32_t* g, uint32_t n, uint32_t* sh) {
    // n <= kSortLdsWave: staged through this wave's LDS slice.
    const uint32_t lane = lane_id();
    for (uint32_t i = lane; i < n; i += 64) sh[i] = g[i];
    wave_sync();
    uint32_t N = 1;
    while (N < n) N <<= 1;
    for (uint32_t k = 2; k <= N; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = lane; i < N; i += 64) {
                const uint32_t p = (j == (k >> 1)) ? (i ^ (k - 1)) : (i ^ j);
                if (p > i && p < n) {
                    const uint32_t x = sh[i], y = sh[p];
                    if (y < x) { sh[i] = y; sh[p] = x; }
                }
            }
            wave_sync();
        }
    }
    bool twice = false;
    for (uint32_t i = lane; i < n; i += 64) {
        g[i] = sh[i];
        if (i > 0 && sh[i] == sh[i - 1]) twice = true;
    }
    wave_sync();
    return twice;
}

constexpr uint32_t kSortWaves = 4;

// Sorts the segments and finishes the admission: a key twice in a segment breaks a precondition (an
// undirected edge given as both (a, b) and (b, a) lands in a's segment twice), and adm[6 + c] +=
// the relocations into blocks of size class c under k_apply_insertions' rule.  A wave takes 64
// touched vertices, a lane each: most segments hold a few keys and are sorted in the lane's
// registers; the longer ones are then sorted by the whole wave in turn, the longest left to
// k_batch_segsort_big.  The vertices of a wave are a group count apart in the list: hubs are touched
// first, and 64 neighbours of the list's start held 64 long segments for one wave (500,000 edges:
// 625 us).  (A wave per vertex spent its time in the dependent loads of one vertex after the other.)
__global__ void __launch_bounds__(kSortWaves * 64) k_batch_segsort(DevGraph g, int dir, BatchScratch w, unsigned long long* adm) {
    __shared__ uint32_t sh[kSortWaves][kSortLdsWave];
    __shared__ uint32_t cls_n[kFreeClasses];  // relocations of this block by size class
    if (threadIdx.x < kFreeClasses) cls_n[threadIdx.x] = 0;
    __syncthreads();
    const DevDelta d = g.delta[dir];
    const DevAdj A = g.dir[dir];
    const uint32_t wid = threadIdx.x >> 6, lane = lane_id();
    const uint32_t T = *w.n_touched;
    bool bad = false;
    const uint32_t groups = (T + 63) / 64;
    for (uint32_t gi = blockIdx.x * kSortWaves + wid; gi < groups; gi += gridDim.x * kSortWaves) {
        uint4 s = make_uint4(0, 0, 0, 0);
        const uint32_t i = lane * groups + gi;
        if (i < T) {
            const uint32_t v = w.touched[i];
            s = d.seg[v];
            const uint2 a = A.adj[v];
            const uint32_t cap = A.cap[v];
            const uint32_t nd = a.y - s.w + s.y;
            if (s.w <= a.y && s.y && nd > cap) {
                uint32_t p2 = 1;
                while (p2 < nd) p2 <<= 1;
                atomicAdd(&cls_n[31u - __clz(max(kMinNbrSize, 2u * p2))], 1u);
            }
        }
#pragma unroll
        for (int which = 0; which < 2; which++) {
            uint32_t* const keys = which == 0 ? d.ins : d.del;
            const uint32_t off = which == 0 ? s.x : s.z, len = which == 0 ? s.y : s.w;
            if (len > 1 && len <= kSortLane) bad = lane_sort(keys + off, len) || bad;
            for (uint64_t m = __ballot(len > kSortLane); m; m &= m - 1) {
                const int l = __ffsll(static_cast<long long>(m)) - 1;
                const uint32_t o = uniform(__shfl(off, l, 64)), n = uniform(__shfl(len, l, 64));
                if (n <= 64) bad = wave_sort_small(keys + o, n) || bad;
                else if (n <= kSortLdsWave) bad = wave_sort_lds(keys + o, n, sh[wid]) || bad;
                else if (lane == 0) {
                    const uint32_t p = atomicAdd(w.n_big, 1u);
                    if (p < w.max_big) { w.big_ptr[p] = o; w.big_len[p] = n | (which ? 0x80000000u : 0u); }
                }
            }
        }
    }
    if (__ballot(bad) != 0 && lane == 0) atomicOr(reinterpret_cast<uint32_t*>(&adm[1]), 1u);
    __syncthreads();
    if (threadIdx.x < kFreeClasses && cls_n[threadIdx.x]) atomicAdd(&adm[6 + threadIdx.x], static_cast<unsigned long long>(cls_n[threadIdx.x]));
}

// Segments longer than one wave's LDS slice: one block each, the bitonic network in LDS, or in
// global memory when they do not fit there.
constexpr uint32_t kSortLdsBlock = 8192;
__device__ __forceinline__ void block_sort(uint32_t* a, uint32_t n) {
    uint32_t N = 1;
    while (N < n) N <<= 1;
    for (uint32_t k = 2; k <= N; k <<= 1) {
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            for (uint32_t i = threadIdx.x; i < N; i += blockDim.x) {
                const uint32_t p = (j == (k >> 1)) ? (i ^ (k - 1)) : (i ^ j);
                if (p > i && p < n) {
                    const uint32_t x = a[i], y = a[p];
                    if (y < x) { a[i] = y; a[p] = x; }
                }
            }
            __syncthreads();
        }
    }
}

__global__ void __launch_bounds__(1024) k_batch_segsort_big(BatchScratch w, DevDelta d, uint32_t* err, unsigned long long* adm) {
    __shared__ uint32_t sh[kSortLdsBlock];
    const uint32_t nb = min(*w.n_big, w.max_big);
    if (*w.n_big > w.max_big && threadIdx.x == 0 && blockIdx.x == 0) atomicOr(err, kErrSegmentTooLong);
    for (uint32_t s = blockIdx.x; s < nb; s += gridDim.x) {
        const uint32_t raw = w.big_len[s];
        const uint32_t n = raw & 0x7FFFFFFFu;
        uint32_t* a = ((raw >> 31) ? d.del : d.ins) + w.big_ptr[s];
        bool twice = false;
        if (n <= kSortLdsBlock) {
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) sh[i] = a[i];
            __syncthreads();
            block_sort(sh, n);
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
                a[i] = sh[i];
                if (i > 0 && sh[i] == sh[i - 1]) twice = true;
            }
            __syncthreads();  // sh is rewritten by the next segment
        } else {
            block_sort(a, n);
            for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
                if (i > 0 && a[i] == a[i - 1]) twice = true;
        }
        if (twice) atomicOr(reinterpret_cast<uint32_t*>(&adm[1]), 1u);
    }
}

// ---------------------------------------------------------------------------------------------
// Apply the batch to the base adjacency of one direction.
__global__ void __launch_bounds__(256) k_apply_deletions(DevGraph g, int dir, BatchScratch w) {
    const uint32_t lane = lane_id();
    const uint32_t wpb = blockDim.x >> 6;
    const uint32_t T = *w.n_touched;
    DevAdj A = g.dir[dir];
    DevDelta D = g.delta[dir];
    for (uint32_t i = blockIdx.x * wpb + (threadIdx.x >> 6); i < T; i += gridDim.x * wpb) {
        const uint32_t v = w.touched[i];
        const uint4 s = D.seg[v];
        if (s.w == 0) continue;
        const uint2 a = A.adj[v];
        uint32_t out = a.x, removed = 0;
        for (uint32_t c = a.x; c < a.x + a.y; c += 64) {
            const uint32_t idx = c + lane;
            const bool valid = idx < a.x + a.y;
            const uint32_t k = valid ? g.arena[idx] : 0u;
            const bool del = valid && contains_u32(D.del, s.z, s.z + s.w, k);
            const bool keep = valid && !del;
            const uint64_t km = __ballot(keep);
            const uint64_t dm = __ballot(del);
            wave_sync();
            if (keep) g.arena[out + lanes_below(km)] = k;
            out += static_cast<uint32_t>(__popcll(km));
            removed += static_cast<uint32_t>(__popcll(dm));
            wave_sync();
        }
        if (lane == 0) {
            A.adj[v].y = a.y - removed;
            if (removed != s.w) atomicOr(g.err, kErrPrecondition);
        }
    }
}

__global__ void __launch_bounds__(256) k_apply_insertions(DevGraph g, int dir, BatchScratch w, unsigned long long* nbytes) {
    const uint32_t lane = lane_id();
    uint64_t bytes = 0;  // lane 0 of each wave: 8 * (old + inserted) + 16 per list, 8 per inserted key
    const uint32_t wpb = blockDim.x >> 6;
    const uint32_t T = *w.n_touched;
    DevAdj A = g.dir[dir];
    DevDelta D = g.delta[dir];
    for (uint32_t i = blockIdx.x * wpb + (threadIdx.x >> 6); i < T; i += gridDim.x * wpb) {
        const uint32_t v = w.touched[i];
        const uint4 s = D.seg[v];
        if (s.y == 0) continue;
        const uint2 a = A.adj[v];
        const uint32_t cap = A.cap[v];
        const uint32_t nd = a.y + s.y;
        if (lane == 0) bytes += 8ull * nd + 16 + 8ull * s.y;
        const uint32_t* ins = D.ins + s.x;
        uint32_t dst = a.x;
        uint32_t newcap = cap;
        bool relocate = nd > cap;
        if (relocate) {
            uint32_t p2 = 1;
            while (p2 < nd) p2 <<= 1;
            newcap = max(kMinNbrSize, 2u * p2);
            unsigned long long base = ~0ull;
            if (lane == 0) {
                const uint32_t c = 31u - __clz(newcap);
                const uint2 cl = g.fl_cls[c];
                if (cl.y) {  // a block freed by an earlier batch
                    const int k = atomicSub(&g.fl_top[c], 1) - 1;
                    if (k >= 0) base = g.fl_blk[cl.x + k];
                }
                if (base == ~0ull) {
                    base = atomicAdd(g.arena_top, static_cast<unsigned long long>(newcap));
                    if (base + newcap > g.arena_words) { atomicOr(g.err, kErrArenaFull); base = ~0ull; }
                }
            }
            base = __shfl(base, 0, 64);
            if (base == ~0ull) continue;
            dst = static_cast<uint32_t>(base);
        }
        // Insert keys: final position = j + #old keys below, computed before any old key moves;
        // an equal old key violates the "inserted edges are new" precondition.
        for (uint32_t j = lane; j < s.y; j += 64) {
            const uint32_t b = ins[j];
            const uint32_t p = lower_bound_u32(g.arena, a.x, a.x + a.y, b);
            if (p < a.x + a.y && g.arena[p] == b) atomicOr(g.err, kErrPrecondition);
            w.ins_pos[s.x + j] = j + (p - a.x);
        }
        wave_sync();
        if (relocate) {
            for (uint32_t k = lane; k < a.y; k += 64) {
                const uint32_t x = g.arena[a.x + k];
                g.arena[dst + k + lower_bound_u32(ins, 0, s.y, x)] = x;
            }
        } else {
            // In place, back to front: every old key moves right by the number of inserted keys
            // below it; a chunk is read completely before any of it is written, and the keys not
            // yet read all sit left of the chunk, below every destination of the chunk.
            const uint32_t first = lower_bound_u32(g.arena, a.x, a.x + a.y, ins[0]) - a.x;
            uint32_t end = a.y;
            while (end > first) {
                const uint32_t start = end - min(64u, end - first);
                const uint32_t k = start + lane;
                const bool valid = k < end;
                const uint32_t x = valid ? g.arena[a.x + k] : 0u;
                const uint32_t pos = valid ? k + lower_bound_u32(ins, 0, s.y, x) : 0u;
                wave_sync();
                if (valid) g.arena[dst + pos] = x;
                wave_sync();
                end = start;
            }
        }
        for (uint32_t j = lane; j < s.y; j += 64) g.arena[dst + w.ins_pos[s.x + j]] = ins[j];
        wave_sync();
        if (lane == 0) {
            A.adj[v] = make_uint2(dst, nd);
            if (relocate) {
                A.cap[v] = newcap;
                const uint32_t c = 31u - __clz(cap);  // the old block (capacities are powers of two)
                const uint2 cl = g.fl_cls[c];
                const uint32_t j = cl.y ? atomicAdd(&g.fl_pend_n[c], 1u) : 0xFFFFFFFFu;
                if (j < cl.y) g.fl_pend[cl.x + j] = a.x;  // else the block stays unused
            }
        }
    }
    if (nbytes && lane == 0 && bytes) atomicAdd(nbytes, static_cast<unsigned long long>(bytes));
}

// After a batch: the blocks its relocations freed become available to the next batches.
__global__ void k_free_merge(DevGraph g) {
    for (uint32_t c = blockIdx.y; c < kFreeClasses; c += gridDim.y) {
        const uint2 cl = g.fl_cls[c];
        if (!cl.y) continue;
        const uint32_t t = static_cast<uint32_t>(max(g.fl_top[c], 0));
        const uint32_t n = min(g.fl_pend_n[c], cl.y - t);
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
            g.fl_blk[cl.x + t + i] = g.fl_pend[cl.x + i];
    }
}
__global__ void k_free_merge_counts(DevGraph g) {
    const uint32_t c = threadIdx.x;
    if (c >= kFreeClasses) return;
    const uint2 cl = g.fl_cls[c];
    const uint32_t t = static_cast<uint32_t>(max(g.fl_top[c], 0));
    g.fl_top[c] = static_cast<int>(t + min(g.fl_pend_n[c], cl.y - t));
    g.fl_pend_n[c] = 0;
}

// The built batch's verdict for the host: out[0..3] = {need, bad, arena top, error bits}, need = the
// words of the relocations that the free blocks of their classes cannot serve; the flag and the
// class counts adm[6..37] are cleared for the next batch.  One wave, a lane per class.
__global__ void __launch_bounds__(64) k_admit_finish(DevGraph g, unsigned long long* adm, unsigned long long* out) {
    const uint32_t c = threadIdx.x;
    unsigned long long need = 0;
    if (c < kFreeClasses) {
        const unsigned long long n = adm[6 + c];
        const unsigned long long avail = g.fl_cls[c].y ? static_cast<unsigned long long>(max(g.fl_top[c], 0)) : 0ull;
        if (n > avail) need = (n - avail) << c;
        adm[6 + c] = 0;
    }
    need = wave_sum_u64(need);
    if (c == 0) {
        out[0] = need;
        out[1] = adm[1];
        out[2] = *g.arena_top;
        out[3] = *g.err;
        adm[1] = 0;
    }
}

__global__ void k_batch_cleanup(BatchScratch w, DevDelta d) {
    const uint32_t T = *w.n_touched;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < T; i += gridDim.x * blockDim.x) {
        const uint32_t v = w.touched[i];
        d.seg[v] = make_uint4(0, 0, 0, 0);
        w.cnt[v] = 0;
    }
}

// Thread per (vertex, slot): row[s] = lower bound of key (s << id_bits) in the vertex's list;
// row[nslots] = end of the list.
__global__ void __launch_bounds__(256) k_slot_dir(DevGraph g, int dir, const uint32_t* list, const uint32_t* n_list, uint32_t max_n) {
    const uint32_t n = list ? min(*n_list, max_n) : g.dv;
    const uint32_t w = g.nslots + 1;
    const uint64_t total = static_cast<uint64_t>(n) * w;
    for (uint64_t t = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; t < total;
         t += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const uint32_t i = static_cast<uint32_t>(t / w), sl = static_cast<uint32_t>(t % w);
        const uint32_t v = list ? list[i] : i;
        const uint2 a = g.dir[dir].adj[v];
        const uint32_t key0 = sl == 0 ? 0u : (sl << g.id_bits);  // sl < nslots: fits the key width
        const uint32_t r = sl == g.nslots ? a.x + a.y : lower_bound_u32(g.arena, a.x, a.x + a.y, key0);
        g.sdir[dir][static_cast<uint64_t>(v) * w + sl] = r;
    }
}

// Label buckets of the touched vertices: a histogram, its scan, then a scatter.  With few labels
// every block counts in LDS and reserves its run of each bucket with one device atomic per label
// (a device atomic per vertex would serialise on the few bucket counters); with more labels than
// the LDS table holds, per-vertex device atomics.
constexpr uint32_t kBucketLds = 4096;

__global__ void __launch_bounds__(256) k_bucket_count(DevGraph g, BatchScratch w) {
    __shared__ uint32_t h[kBucketLds];
    const uint32_t T = *w.n_touched;
    const bool lds = g.nvl <= kBucketLds;
    if (lds) {
        for (uint32_t r = threadIdx.x; r < g.nvl; r += blockDim.x) h[r] = 0;
        __syncthreads();
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < T; i += gridDim.x * blockDim.x) {
        const uint32_t r = g.vrank[w.touched[i]];
        if (r >= g.nvl) continue;
        if (lds) atomicAdd(&h[r], 1u);
        else atomicAdd(&w.label_cur[r], 1u);
    }
    if (lds) {
        __syncthreads();
        for (uint32_t r = threadIdx.x; r < g.nvl; r += blockDim.x)
            if (h[r]) atomicAdd(&w.label_cur[r], h[r]);
    }
}

// Same walk over the touched vertices as k_bucket_count (same grid): each block counts again in
// LDS, reserves its runs from the bucket cursors, then places its vertices in them.
__global__ void __launch_bounds__(256) k_bucket_scatter(DevGraph g, BatchScratch w) {
    __shared__ uint32_t h[kBucketLds];
    const uint32_t T = *w.n_touched;
    if (g.nvl > kBucketLds) {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < T; i += gridDim.x * blockDim.x) {
            const uint32_t v = w.touched[i];
            const uint32_t r = g.vrank[v];
            if (r < g.nvl) w.by_label[atomicAdd(&w.label_cur[r], 1u)] = v;
        }
        return;
    }
    for (uint32_t r = threadIdx.x; r < g.nvl; r += blockDim.x) h[r] = 0;
    __syncthreads();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < T; i += gridDim.x * blockDim.x) {
        const uint32_t r = g.vrank[w.touched[i]];
        if (r < g.nvl) atomicAdd(&h[r], 1u);
    }
    __syncthreads();
    for (uint32_t r = threadIdx.x; r < g.nvl; r += blockDim.x)
        if (h[r]) h[r] = atomicAdd(&w.label_cur[r], h[r]);  // the block's first position in bucket r
    __syncthreads();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < T; i += gridDim.x * blockDim.x) {
        const uint32_t v = w.touched[i];
        const uint32_t r = g.vrank[v];
        if (r < g.nvl) w.by_label[atomicAdd(&h[r], 1u)] = v;
    }
}

}  // namespace

void batch_begin(const BatchScratch* w, int dirs, uint32_t nvl, uint32_t* results, uint32_t nresults, hipStream_t s) {
    const uint32_t most = std::max(nvl + 1, nresults);
    k_batch_begin<<<std::min<uint32_t>(256, (most + 255) / 256), 256, 0, s>>>(w[0], w[dirs - 1], static_cast<uint32_t>(dirs), nvl + 1, results, nresults);
}

// Builds the delta of batch edges [lo, lo + n) for one direction.  n_touched ends up on the
// device; the number of arcs bounds every grid.
void batch_build(const DevGraph& g, int dir, int dirsel, const BatchInput& b, uint32_t lo, uint32_t n, const BatchScratch& w,
                 unsigned long long* adm, hipStream_t s) {
    const uint32_t max_arcs = 2 * n;
    auto grid = [](uint32_t items, uint32_t per, uint32_t cap) { return std::min<uint32_t>(cap, (items + per - 1) / per); };
    k_batch_count<<<grid(n, kCountTile, 2048), 256, 0, s>>>(b, lo, n, dirsel, w);
    k_batch_segments<<<grid(max_arcs, 256 * kSegItems, 1024), 256, 0, s>>>(w, g.delta[dir]);
    k_batch_scatter<<<grid(n, 256, 4096), 256, 0, s>>>(g, b, lo, n, dirsel, dir, w, adm);
    k_batch_segsort<<<grid(max_arcs, kSortWaves * 64, 2048), kSortWaves * 64, 0, s>>>(g, dir, w, adm);
    if (max_arcs > kSortLdsWave) k_batch_segsort_big<<<grid(max_arcs, kSortLdsWave, 256), 1024, 0, s>>>(w, g.delta[dir], g.err, adm);
}

void batch_bucket(const DevGraph& g, uint32_t max_touched, const BatchScratch& w, hipStream_t s) {
    const int grid = static_cast<int>(std::min<uint32_t>(2048, (max_touched + 255) / 256 + 1));
    k_bucket_count<<<grid, 256, 0, s>>>(g, w);
    scan_exclusive<uint32_t>(w.label_cur, w.label_off, nullptr, g.nvl, true, w.label_tmp, s);
    copy_u32(w.label_off, w.label_cur, g.nvl, s);  // the scatter's cursors
    k_bucket_scatter<<<grid, 256, 0, s>>>(g, w);
}

void slot_dir_update(const DevGraph& g, int dir, const uint32_t* list, const uint32_t* n_list, uint32_t max_n, hipStream_t s) {
    if (!g.sdir[dir]) return;
    const uint64_t total = static_cast<uint64_t>(list ? max_n : g.dv) * (g.nslots + 1);
    const int grid = static_cast<int>(std::max<uint64_t>(1, std::min<uint64_t>(8192, (total + 255) / 256)));
    k_slot_dir<<<grid, 256, 0, s>>>(g, dir, list, n_list, max_n);
}

void batch_apply_deletions(const DevGraph& g, int dir, uint32_t max_touched, const BatchScratch& w, hipStream_t s) {
    const int grid = static_cast<int>(std::min<uint32_t>(8192, (max_touched + 3) / 4 + 1));
    k_apply_deletions<<<grid, 256, 0, s>>>(g, dir, w);
}

void batch_apply_insertions(const DevGraph& g, int dir, uint32_t max_touched, const BatchScratch& w, unsigned long long* bytes,
                            hipStream_t s) {
    const int grid = static_cast<int>(std::min<uint32_t>(8192, (max_touched + 3) / 4 + 1));
    k_apply_insertions<<<grid, 256, 0, s>>>(g, dir, w, bytes);
}

void batch_admit_finish(const DevGraph& g, unsigned long long* adm, unsigned long long* out, hipStream_t s) {
    k_admit_finish<<<1, 64, 0, s>>>(g, adm, out);
}

void free_blocks_merge(const DevGraph& g, hipStream_t s) {
    k_free_merge<<<dim3(64, kFreeClasses), 256, 0, s>>>(g);
    k_free_merge_counts<<<1, 64, 0, s>>>(g);
}

void batch_cleanup(const DevGraph& g, int dir, uint32_t max_touched, const BatchScratch& w, hipStream_t s) {
    const int grid = static_cast<int>(std::min<uint32_t>(4096, (max_touched + 255) / 256 + 1));
    k_batch_cleanup<<<grid, 256, 0, s>>>(w, g.delta[dir]);
}

}  // namespace csm
