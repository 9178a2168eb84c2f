// Edge-anchored incremental enumeration on wave64.
//
//   init_from_pairs / init_from_set   initial partial results of the first matching-order edge
//                                      (write_initial_partial_results, enumeration.cu:24-79)
//   extend                             depth-first search down to end_depth, a wave with an LDS stack
//                                      of batches of up to 64 partial results; counts and
//                                      hashes complete embeddings or writes partial results of
//                                      end_depth (a BFS level when end_depth = d0 + 1).  Replaces
//                                      extendBFSDFSRegTwo (enumeration.cu:407-781) and gamma_enumerate
//                                      (gamma_enumeration.cu:359-880).
//   direct_search                      the same search from the anchor pairs of many small steps in one
//                                      launch, without a local index
//   level_prepare / level_flat         one breadth-first level flattened over its candidates: per
//   (and the _chain variants)          record, the runs of every backward entry and the shortest as
//                                      the generator, then four candidates per lane tested in
//                                      lock-step; the _chain variants read their size from the
//                                      levels before them, so a step's levels run without the host.
//   cp_prepare / cp_enumerate          Cartesian-product flattening of trailing tree leaves
//                                      (GetNumTree + enumerateCartesianProductTree,
//                                      cartesian_product.cu:193-284).
// In the depth-first kernels, candidates of a depth come from the shortest of the first backward
// neighbours' view runs; each is tested for its bit in the candidate bitmap, injectivity against the
// matched prefix, and membership in every other backward neighbour's view run by binary search
// (search.cuh:7-25 semantics).
#include "dfs_grid.h"
#include "kernels.h"
#include "range_word.h"
#include "view.h"

namespace csm {
namespace {

constexpr uint32_t kWaves = kDfsWaves;

// Per-wave state of the depth-first search in LDS.  The wave searches batches of up to 64 partial
// results: frame j extends its rows (partial results of depth d0 + j, at most one per lane) by the
// vertex of that depth.  Behind the header (dynamic LDS, per wave): the current frame's matched
// vertices, one row of 64 words per position below end_depth, then one child buffer per frame that
// is followed by another.
constexpr uint32_t kDfsIlp = 2;                       // candidates a lane tests together
constexpr uint32_t kDfsBuf = 64 + 64 * kDfsIlp;       // a round finds fewer than 64 rows waiting
constexpr uint32_t kDfsRuns = 4;                      // entries whose runs are kept per row; the others are looked up per candidate
struct DfsHdr {
    unsigned long long ph[64];   // prefix hash of the row
    uint4 runs[kDfsRuns][64];    // view runs of the row's backward entries
    uint32_t pre[64];            // exclusive prefix of the rows' generating lengths
    uint32_t gen[64];            // generating entry of the row (the shortest of the kept runs)
    uint32_t skip[64];           // first generated element (a record cut into chunks)
    uint32_t rec[64];            // record of each row of frame 0
    uint32_t chunk[64], chunks[64];
    uint32_t rows[kMaxQV], waiting[kMaxQV], cur[kMaxQV], tot[kMaxQV];
};
struct DfsBuf {
    uint32_t cand[kDfsBuf];   // vertex matched at the frame's depth
    uint8_t parent[kDfsBuf];  // row of the frame it extends
};

__host__ __device__ constexpr uint32_t wave_lds_bytes(uint32_t d0, uint32_t end_depth) {
    const uint32_t bufs = end_depth > d0 + 1 ? end_depth - 1 - d0 : 0u;
    return static_cast<uint32_t>((sizeof(DfsHdr) + (end_depth - 1) * 256u + bufs * sizeof(DfsBuf) + 15u) & ~15u);
}

__device__ __forceinline__ const uint32_t* entry_delta(const DevGraph& g, const StepDesc& d, const BackEntry& e) {
    return phase_delta(g, e.dir, d.phase);
}

// A uniform entry in two scalar loads (its bytes one by one would be vector loads).
__device__ __forceinline__ BackEntry load_entry(const BackEntry* p) {
    static_assert(sizeof(BackEntry) == 8 && alignof(BackEntry) == 4, "two words");
    uint32_t w[2];
    __builtin_memcpy(w, p, 8);
    BackEntry e;
    e.slot = w[0];
    e.pos = static_cast<uint8_t>(w[1]);
    e.view = static_cast<uint8_t>(w[1] >> 8);
    e.dir = static_cast<uint8_t>(w[1] >> 16);
    e.pad = 0;
    return e;
}

// Last record r with off[r] <= item, given off[0] <= item < off[n]: a 64-ary search in which every
// lane probes one of 64 evenly spaced offsets per round.
__device__ __forceinline__ uint32_t find_record(const unsigned long long* off, uint32_t n, unsigned long long item, uint32_t lane) {
    uint32_t lo = 0, hi = n;
    while (hi - lo > 1) {
        const uint32_t step = (hi - lo + 63) / 64;
        const uint32_t p = lo + lane * step;
        const uint64_t m = __ballot(p < hi && off[p] <= item);
        lo += (63u - static_cast<uint32_t>(__clzll(m))) * step;
        hi = min(hi, lo + step);
    }
    return uniform(lo);
}

// ---- Range donation (work stealing) of the depth-first kernel --------------------------------
// Each wave owns a pair of words per launch (range_word.h): the candidate range [cur, end) of its current
// frame 0 still to be explored, and which items that frame holds.  The owner takes its next 64-candidate
// round by moving cur up; a wave out of work takes the upper half of another wave's range by moving
// that wave's end down to the midpoint.  Both are compare-and-swaps on the range word, so the rounds taken
// and the halves donated never overlap.  The owner publishes only when its range is used up, and then
// another version, so a thief's swap fails if the range was published anew since it was read.  Ranges only
// shrink, so every wave's search ends.  All of it is relaxed, the agent-scope acquire and release of an
// ordered protocol (an L1 invalidation per probe, an L2 write-back per publication) took more than half
// of the kernel's time: the two words are the only data the waves exchange, and a thief uses a frame
// word only if it carries the range's version, whatever order the two stores become visible in.
// (The reference's disabled design: gamma_enumeration.cu:209-357.)
constexpr uint32_t kStealRounds = 8;  // victim probes of 64 waves each before a wave gives up

// Owner (one lane): the next round [t, t_end) of its published range, false when it is used up.
__device__ __forceinline__ bool claim_round(unsigned long long* slot, uint32_t& t, uint32_t& t_end) {
    unsigned long long w = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    for (;;) {
        const uint32_t cur = range_cur(w), end = range_end(w);
        if (cur >= end) return false;
        const uint32_t nc = min(cur + 64u, end);
        const unsigned long long nw = (w & ~(static_cast<unsigned long long>(kRangeMask) << kRangeBits)) |
                                      (static_cast<unsigned long long>(nc) << kRangeBits);
        const unsigned long long seen = atomicCAS(slot, w, nw);
        if (seen == w) {
            t = cur;
            t_end = nc;
            return true;
        }
        w = seen;
    }
}

// Thief (whole wave): the upper half of some wave's range with at least two rounds left.
__device__ __forceinline__ bool steal_range(unsigned long long* donate, uint32_t total_waves, uint32_t gw, uint32_t lane, uint32_t& grp,
                                            uint32_t& first, uint32_t& lo, uint32_t& hi) {
    for (uint32_t a = 0; a < kStealRounds; a++) {
        const uint32_t v = (gw + 1 + a * 64 + lane * (1 + a)) % total_waves;
        const unsigned long long w = v != gw ? __hip_atomic_load(donate + 2ull * v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        const uint32_t cur = range_cur(w), end = range_end(w);
        const uint32_t rem = end > cur ? end - cur : 0u;
        uint32_t key = rem << 6 | lane;  // rem < 2^24: fits
        for (int o = 32; o > 0; o >>= 1) key = max(key, static_cast<uint32_t>(__shfl_xor(key, o, 64)));
        if ((key >> 6) < 128u) continue;
        const uint32_t src = key & 63u;
        uint32_t got = 0, mid = 0;
        unsigned long long r = 0;
        if (lane == src) {
            mid = cur + (((rem >> 1) + 63u) & ~63u);  // cur + 64 <= mid < end
            r = __hip_atomic_load(donate + 2ull * v + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long nw = (w & ~static_cast<unsigned long long>(kRangeMask)) | mid;
            got = same_publication(w, r) && atomicCAS(donate + 2ull * v, w, nw) == w ? 1u : 0u;
        }
        if (__shfl(got, src, 64)) {
            grp = __shfl(frame_group(r), src, 64);
            first = __shfl(frame_first(r), src, 64);
            lo = __shfl(mid, src, 64);
            hi = __shfl(end, src, 64);
            return true;
        }
    }
    return false;
}

// Membership of key[j] in the sorted a[lo[j], hi[j]) for the active j, N searches advancing in
// lock-step (each round issues all N loads before using any).  A present key is always probed: a
// lower-bound search probes the position it ends on unless that position is hi.
template <uint32_t N>
__device__ __forceinline__ void contains_many(const uint32_t* a, const uint32_t* lo0, const uint32_t* hi0, const uint32_t* key,
                                              const bool* act, bool* found) {
    uint32_t lo[N], n[N];
    bool more = false;
#pragma unroll
    for (uint32_t j = 0; j < N; j++) {
        lo[j] = lo0[j];
        n[j] = act[j] ? hi0[j] - lo0[j] : 0u;
        found[j] = false;
        more = more || n[j] != 0;
    }
    while (more) {
        uint32_t v[N];
#pragma unroll
        for (uint32_t j = 0; j < N; j++) v[j] = n[j] ? a[lo[j] + (n[j] >> 1)] : 0u;
        more = false;
#pragma unroll
        for (uint32_t j = 0; j < N; j++) {
            if (!n[j]) continue;
            const uint32_t h = n[j] >> 1;
            if (v[j] == key[j]) {
                found[j] = true;
                n[j] = 0;
            } else if (v[j] < key[j]) {
                lo[j] += h + 1;
                n[j] -= h + 1;
            } else {
                n[j] = h;
            }
            more = more || n[j] != 0;
        }
    }
}

// Matched vertices, prefix hashes, backward runs and generating lengths of the rows of frame j; the
// frame's candidates are the rows' generating runs one after another.  Returns their number, and in
// `rows` how many of the rows it took: the first ones that have at most kFrameMax candidates together, or
// one row alone (a list is shorter than 2^31), since 64 rows may share a list and their sum has 32 bits.
// The rows of frame 0 are records `stride` words apart; with kRanged, row r takes the elements
// [chunk[r], chunks[r]) of its run instead of a whole chunk of it, and all rows are taken: a number past
// kFrameMax then only says that there are too many.
constexpr uint32_t kFrameMax = kRangeMask;  // a frame of several rows fits a donated range
template <bool kRanged>
__device__ __forceinline__ uint32_t dfs_rows(const DevGraph& g, const StepDesc& d, uint32_t d0, uint32_t j, uint32_t& rows, const uint32_t* in,
                                             uint32_t stride, DfsHdr& H, uint32_t* f, const DfsBuf* buf, uint32_t lane, unsigned long long& bytes,
                                             bool count_bytes) {
    const uint32_t depth = d0 + j, e0 = d.boff[depth], ne = d.boff[depth + 1] - e0;
    uint32_t len = 0, skip = 0;
    unsigned long long row_bytes = 0;
    if (lane < rows) {
        unsigned long long h = 0;
        uint32_t r = lane;
        for (uint32_t p = depth; p-- > d0;) {
            const uint32_t v = buf[p - d0].cand[r];
            f[p * 64 + lane] = v;
            h += pair_hash(d.order[p], v);
            r = buf[p - d0].parent[r];
        }
        const uint32_t* rec = in + static_cast<uint64_t>(H.rec[r]) * stride;
        for (uint32_t p = 0; p < d0; p++) {
            const uint32_t v = rec[p];
            f[p * 64 + lane] = v;
            h += pair_hash(d.order[p], v);
        }
        H.ph[lane] = h;
        RunView rv[kDfsRuns];
#pragma unroll
        for (uint32_t e = 0; e < kDfsRuns; e++) {
            if (e >= ne) break;
            const BackEntry be = d.be[e0 + e];
            rv[e] = make_run(g, d.phase, be.view, be.dir, f[be.pos * 64 + lane], be.slot);
        }
        uint32_t best = 0xFFFFFFFFu, gen = 0;
#pragma unroll
        for (uint32_t e = 0; e < kDfsRuns; e++) {
            if (e >= ne) break;
            H.runs[e][lane] = make_uint4(rv[e].lo, rv[e].hi, rv[e].dlo, rv[e].dhi);
            const uint32_t l = run_seq_len(rv[e], d.be[e0 + e].view);
            if (l < best) {
                best = l;
                gen = e;
            }
            if (count_bytes && (j || (kRanged ? H.chunks[lane] == 0xFFFFFFFFu : H.chunk[lane] == 0))) row_bytes += 4ull * ((rv[e].hi - rv[e].lo) + (rv[e].dhi - rv[e].dlo));
        }
        H.gen[lane] = gen;
        len = best;
        if (kRanged) {
            if (j == 0) {
                skip = min(best, H.chunk[lane]);
                len = min(best, H.chunks[lane]) - skip;
            }
        } else if (j == 0 && H.chunks[lane] > 1) {  // the record's candidates are cut into whole 64-candidate chunks
            const uint32_t width = ((best + H.chunks[lane] - 1) / H.chunks[lane] + 63u) & ~63u;
            skip = min(best, H.chunk[lane] * width);
            len = min(best - skip, width);
        }
    }
    const uint32_t part = min(len, kFrameMax + 1);  // 64 of them stay under 2^31
    uint32_t total;
    uint32_t pre = wave_prefix(part, total);
    total = uniform(total);
    if (!kRanged && total > kFrameMax) {
        rows = max(1u, static_cast<uint32_t>(__popcll(__ballot(lane < rows && pre + part <= kFrameMax))));
        total = uniform(__shfl(rows == 1 ? len : pre + part, static_cast<int>(rows) - 1, 64));
        if (lane >= rows) pre = total;
    }
    if (lane < rows) bytes += row_bytes;
    H.pre[lane] = pre;
    H.skip[lane] = skip;
    wave_sync();
    return total;
}

// One round of a frame's candidates, flattened elements cur + 64 u + lane below tot: their row k, vertex
// c, and whether it extends the row (candidate bitmap, injectivity, every backward entry's view).
__device__ __forceinline__ void dfs_round(const DevGraph& g, const StepDesc& d, uint32_t depth, uint32_t cur, uint32_t tot, const DfsHdr& H,
                                          const uint32_t* f, uint32_t lane, uint32_t* k, uint32_t* c, bool* ok) {
    const uint32_t e0 = d.boff[depth], ne = d.boff[depth + 1] - e0;
    uint32_t key[kDfsIlp], gen[kDfsIlp];
#pragma unroll
    for (uint32_t u = 0; u < kDfsIlp; u++) {
        const uint32_t e = cur + 64 * u + lane;
        ok[u] = e < tot;
        k[u] = 0;
#pragma unroll
        for (uint32_t st = 32; st; st >>= 1)
            if (H.pre[k[u] + st] <= e) k[u] += st;  // rows past the last hold the total
        gen[u] = H.gen[k[u]];
        key[u] = 0;
        if (ok[u]) {
            const uint4 x = H.runs[gen[u]][k[u]];
            const BackEntry be = d.be[e0 + gen[u]];
            const RunView rv{x.x, x.y, x.z, x.w};
            key[u] = run_elem(g, entry_delta(g, d, be), rv, run_base_len(rv, be.view), H.skip[k[u]] + (e - H.pre[k[u]]));
        }
        c[u] = key[u] & g.id_mask;
    }
#pragma unroll
    for (uint32_t u = 0; u < kDfsIlp; u++) ok[u] = ok[u] && bit_test(as_global(d.filter[depth]), c[u]);
    for (uint32_t im = d.inj[depth]; im; im &= im - 1) {
        const uint32_t q = static_cast<uint32_t>(__ffs(im)) - 1;
#pragma unroll
        for (uint32_t u = 0; u < kDfsIlp; u++) ok[u] = ok[u] && f[q * 64 + k[u]] != c[u];
    }
    for (uint32_t e = 0; e < ne; e++) {  // every entry's view; the generating entry's base run holds the candidate by construction
        const BackEntry be = d.be[e0 + e];
        const uint32_t hi_bits = be.slot << g.id_bits;
        uint32_t pk[kDfsIlp];
        bool act[kDfsIlp];
#pragma unroll
        for (uint32_t u = 0; u < kDfsIlp; u++) {
            pk[u] = hi_bits | c[u];
            act[u] = ok[u] && (gen[u] != e || be.view == kViewBaseMinusDelta);
        }
        if (e < kDfsRuns) {
            uint32_t lo[kDfsIlp], hi[kDfsIlp];
            bool sb[kDfsIlp], inb[kDfsIlp], ind[kDfsIlp], need[kDfsIlp];
#pragma unroll
            for (uint32_t u = 0; u < kDfsIlp; u++) {
                const uint4 x = H.runs[e][k[u]];
                lo[u] = x.x;
                hi[u] = x.y;
                sb[u] = act[u] && be.view != kViewDelta && gen[u] != e;
                inb[u] = false;
            }
            contains_many<kDfsIlp>(g.arena, lo, hi, pk, sb, inb);
#pragma unroll
            for (uint32_t u = 0; u < kDfsIlp; u++) {
                inb[u] = inb[u] || gen[u] == e;
                const uint4 x = H.runs[e][k[u]];
                lo[u] = x.z;
                hi[u] = x.w;
                need[u] = act[u] && (be.view == kViewDelta || (be.view == kViewBasePlusDelta ? !inb[u] : be.view == kViewBaseMinusDelta && inb[u]));
                ind[u] = false;
            }
            if (be.view != kViewBase) contains_many<kDfsIlp>(entry_delta(g, d, be), lo, hi, pk, need, ind);
#pragma unroll
            for (uint32_t u = 0; u < kDfsIlp; u++) {
                if (!act[u]) continue;
                switch (be.view) {
                    case kViewBase: ok[u] = inb[u]; break;
                    case kViewBasePlusDelta: ok[u] = inb[u] || ind[u]; break;
                    case kViewDelta: ok[u] = ind[u]; break;
                    default: ok[u] = inb[u] && !ind[u]; break;
                }
            }
        } else {
#pragma unroll
            for (uint32_t u = 0; u < kDfsIlp; u++)
                if (act[u]) ok[u] = view_contains(g, d.phase, be.view, be.dir, be.slot, f[be.pos * 64 + k[u]], pk[u]);
        }
    }
}

// Back from frame j + 1 to frame j: the rows just searched leave frame j's buffer.
__device__ __forceinline__ void dfs_pop(DfsHdr& H, DfsBuf* buf, uint32_t j, uint32_t lane) {
    const uint32_t done = uniform(H.rows[j + 1]);
    const uint32_t left = uniform(H.waiting[j]) - done;
    for (uint32_t x0 = 0; x0 < left; x0 += 64) {  // 64 at a time: what is written is not read any more
        const uint32_t x = x0 + lane;
        const uint32_t c = x < left ? buf[j].cand[done + x] : 0u;
        const uint8_t p = x < left ? buf[j].parent[done + x] : uint8_t(0);
        wave_sync();
        if (x < left) {
            buf[j].cand[x] = c;
            buf[j].parent[x] = p;
        }
        wave_sync();
    }
    if (lane == 0) H.waiting[j] = left;
    wave_sync();
}

// Depth-first search from the records at depth d0.  The search is latency-bound, and one partial
// result at a time left most lanes without a candidate (a run has a few elements), so a wave holds a
// stack of batches instead: a frame's rows are the partial results found by the frame above it, its
// candidates are flattened over the lanes, and the rows found wait until there are 64 of them or
// the frame is used up.  A returned-to frame looks its rows up again rather than keeping 64 runs per
// depth in LDS.  Items (records, or chunks of records) are taken in groups of up to 64, sized so
// that the grid has a few groups per resident wave.
constexpr uint32_t kDfsGroupWaves = 2048;
template <int kMode>
__global__ void __launch_bounds__(kWaves * 64) k_extend(DevGraph g, StepDesc d, uint32_t d0, uint32_t end_depth, Ring r, MatchOut out,
                                                         const unsigned long long* split, unsigned long long* work, int schedule,
                                                         unsigned long long* donate) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    unsigned char* const wave_base = lds_raw + (threadIdx.x >> 6) * wave_lds_bytes(d0, end_depth);
    DfsHdr& H = *reinterpret_cast<DfsHdr*>(wave_base);
    uint32_t* const f = reinterpret_cast<uint32_t*>(wave_base + sizeof(DfsHdr));  // f[position * 64 + row]
    DfsBuf* const buf = reinterpret_cast<DfsBuf*>(wave_base + sizeof(DfsHdr) + (end_depth - 1) * 256u);
    const uint32_t lane = lane_id();
    const uint32_t nrec = min(*r.in_count, r.in_max);
    const unsigned long long nitems = split ? split[nrec] : nrec;
    const uint32_t total_waves = gridDim.x * kWaves;
    const uint32_t gw = blockIdx.x * kWaves + (threadIdx.x >> 6);
    const uint32_t G = static_cast<uint32_t>(min(64ull, max(1ull, nitems / kDfsGroupWaves)));
    const unsigned long long ngroups = (nitems + G - 1) / G;
    const uint32_t last = end_depth - 1 - d0;  // the frame whose candidates complete
    unsigned long long my_cnt = 0, my_hash = 0, my_bytes = 0;

    const bool donating = schedule == 2;
    uint32_t version = 0, sub = 0;  // sub: items of the group that earlier frames took
    unsigned long long group;
    if (schedule == 0) group = gw;
    else {
        unsigned long long t = 0;
        if (lane == 0) t = atomicAdd(work, 1ull);
        group = __shfl(t, 0, 64);
    }
    for (;;) {
        // the next group of the launch, else (donating) a range taken from another wave
        uint32_t grp, first = sub, s_lo = 0, s_hi = 0;
        bool stolen = false;
        if (group < ngroups) {
            grp = static_cast<uint32_t>(group);
        } else if (donating && steal_range(donate, total_waves, gw, lane, grp, first, s_lo, s_hi)) {
            stolen = true;
        } else {
            break;
        }
        if (kMode == kWriteAtEnd && uniform(__hip_atomic_load(r.overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) break;
        // frame 0: the group's items from `first` on, one per lane
        const unsigned long long item = static_cast<unsigned long long>(grp) * G + first + lane;
        const uint32_t items = static_cast<uint32_t>(min(static_cast<unsigned long long>(G), nitems - static_cast<unsigned long long>(grp) * G));
        uint32_t rows0 = items - first;
        if (lane < rows0) {
            uint32_t rec = static_cast<uint32_t>(item), chunk = 0, chunks = 1;
            if (split) {  // last record with split[rec] <= item
                uint32_t lo = 0, hi = nrec;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (split[mid] <= item) lo = mid;
                    else hi = mid;
                }
                rec = lo;
                chunk = static_cast<uint32_t>(item - split[rec]);
                chunks = static_cast<uint32_t>(split[rec + 1] - split[rec]);
            }
            H.rec[lane] = rec;
            H.chunk[lane] = chunk;
            H.chunks[lane] = chunks;
        }
        wave_sync();
        uint32_t j = 0, built = 0;
        const uint32_t total0 = dfs_rows<false>(g, d, d0, 0, rows0, r.in, d0, H, f, buf, lane, my_bytes, !stolen && out.bytes);
        // donating: publish frame 0's candidates and take the first round from the word (a single row
        // of more than kRangeMask candidates stays the wave's own)
        uint32_t cur0 = stolen ? s_lo : 0u, end0 = stolen ? s_hi : total0;
        const bool published = donating && end0 <= kRangeMask;
        if (published) {
            version = next_version(version);
            uint32_t t = 0, t_end = 0;
            if (lane == 0) {
                __hip_atomic_store(donate + 2ull * gw + 1, frame_word(version, grp, first), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(donate + 2ull * gw, range_word(version, cur0, end0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (!claim_round(donate + 2ull * gw, t, t_end)) t = t_end = 0;
            }
            cur0 = __shfl(t, 0, 64);
            end0 = __shfl(t_end, 0, 64);
        }
        if (lane == 0) {
            H.rows[0] = rows0;
            H.waiting[0] = 0;
            H.cur[0] = cur0;
            H.tot[0] = end0;
        }
        wave_sync();
        for (;;) {
            uint32_t cur = uniform(H.cur[j]), tot = uniform(H.tot[j]);
            if (j == 0 && cur >= tot && published) {  // frame 0's next round from the published range
                uint32_t t = 0, t_end = 0;
                if (lane == 0 && !claim_round(donate + 2ull * gw, t, t_end)) t = t_end = 0;
                cur = uniform(__shfl(t, 0, 64));
                tot = uniform(__shfl(t_end, 0, 64));
                if (lane == 0) {
                    H.cur[0] = cur;
                    H.tot[0] = tot;
                }
                wave_sync();
            }
            const uint32_t waiting = j < last ? uniform(H.waiting[j]) : 0u;
            if (waiting >= 64 || (cur >= tot && waiting)) {  // descend with a batch
                uint32_t rows = min(64u, waiting);
                j += 1;
                const uint32_t t = dfs_rows<false>(g, d, d0, j, rows, r.in, d0, H, f, buf, lane, my_bytes, out.bytes != nullptr);
                built = j;
                if (lane == 0) {
                    H.rows[j] = rows;
                    H.waiting[j] = 0;
                    H.cur[j] = 0;
                    H.tot[j] = t;
                }
                wave_sync();
                continue;
            }
            if (cur >= tot) {
                if (j == 0) break;
                j -= 1;
                dfs_pop(H, buf, j, lane);
                continue;
            }
            if (built != j) {
                uint32_t rows = uniform(H.rows[j]);
                dfs_rows<false>(g, d, d0, j, rows, r.in, d0, H, f, buf, lane, my_bytes, false);
                built = j;
            }
            // one round of frame j's candidates
            const uint32_t depth = d0 + j;
            uint32_t k[kDfsIlp], c[kDfsIlp];
            bool ok[kDfsIlp];
            dfs_round(g, d, depth, cur, tot, H, f, lane, k, c, ok);
            uint64_t m[kDfsIlp];
            uint32_t found = 0;
#pragma unroll
            for (uint32_t u = 0; u < kDfsIlp; u++) {
                m[u] = __ballot(ok[u]);
                found += static_cast<uint32_t>(__popcll(m[u]));
            }
            if (lane == 0) {
                H.cur[j] = cur + 64 * kDfsIlp;
                my_bytes += 4ull * found;
            }
            if (j < last) {
                uint32_t at = waiting;
#pragma unroll
                for (uint32_t u = 0; u < kDfsIlp; u++) {
                    if (ok[u]) {
                        const uint32_t x = at + lanes_below(m[u]);
                        buf[j].cand[x] = c[u];
                        buf[j].parent[x] = static_cast<uint8_t>(k[u]);
                    }
                    at += static_cast<uint32_t>(__popcll(m[u]));
                }
                if (lane == 0) H.waiting[j] = at;
            } else if (kMode == kCountAtEnd) {
#pragma unroll
                for (uint32_t u = 0; u < kDfsIlp; u++)
                    if (ok[u]) {
                        my_cnt += 1;
                        my_hash += embedding_hash(H.ph[k[u]] + pair_hash(d.order[depth], c[u]));
                    }
            } else if (found) {
                uint32_t base = 0;
                if (lane == 0) base = atomicAdd(r.out_count, found);
                base = __shfl(base, 0, 64);
                if (static_cast<uint64_t>(base) + found > r.out_cap) {
                    if (lane == 0) atomicOr(r.overflow, 1u);
                } else {
#pragma unroll
                    for (uint32_t u = 0; u < kDfsIlp; u++) {
                        if (ok[u]) {
                            uint32_t* o = r.out + static_cast<uint64_t>(base + lanes_below(m[u])) * end_depth;
                            for (uint32_t p = 0; p < depth; p++) o[p] = f[p * 64 + k[u]];
                            o[depth] = c[u];
                        }
                        base += static_cast<uint32_t>(__popcll(m[u]));
                    }
                }
            }
            wave_sync();
        }
        if (stolen) continue;  // the launch's items are used up: steal again
        sub += rows0;
        if (sub < items) continue;  // the rest of the group
        sub = 0;
        if (schedule == 0) group += total_waves;
        else {
            unsigned long long t2 = 0;
            if (lane == 0) t2 = atomicAdd(work, 1ull);
            group = __shfl(t2, 0, 64);
        }
    }
    if (kMode == kCountAtEnd) {  // one pair of device atomics per block
        __shared__ unsigned long long s_cnt[kWaves], s_hash[kWaves];
        my_cnt = wave_sum_u64(my_cnt);
        my_hash = wave_sum_u64(my_hash);
        if (lane == 0) { s_cnt[threadIdx.x >> 6] = my_cnt; s_hash[threadIdx.x >> 6] = my_hash; }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long c = 0, h = 0;
            for (uint32_t w = 0; w < kWaves; w++) { c += s_cnt[w]; h += s_hash[w]; }
            if (c) { atomicAdd(out.count, c); atomicAdd(out.hash, h); }
        }
    }
    if (out.bytes) {
        my_bytes = wave_sum_u64(my_bytes);
        if (lane == 0 && my_bytes) atomicAdd(out.bytes, my_bytes);
    }
}

// ---- Direct steps: whole steps searched depth-first from their anchors --------------------------
// Pass 0 (grid.y = step): a wave searches groups of the step's anchor pairs, records of depth 2, with
// the batches above; the global candidate bitmaps filter, so a step needs no local index, no levels
// and no host.  A few heavy anchors would keep single waves busy for milliseconds, so a wave that has
// taken its pass's rounds for a task hands the rest of its stack on: the unfinished ranges of its
// rows and the partial results still waiting become items, up to kDirectTask of them a task, which
// the waves of the next pass share.  Items go to kDirectShards queues, wave by wave: one counter
// would serialise their reservations.  A step that is too large (anchors, candidates, items, tasks
// left after the last pass) is given up: nothing of it is counted, and the host runs it with its local
// index and levels.  The search is bound by the latency of its rounds (about 10 us each: row lookups, a
// list element, the bitmap, binary searches); what it saves is the launches, gaps and host waits of the
// other path, about 30 launches of 3 to 20 us per group of lanes.  Round trips without and with direct
// steps: 32 queries, 1,024-edge batches 4.7, 0.91 ms, 2K to 64K edges 45.5, 10.0 ms; 64 queries, 65,536 edges
// 58.4, 45.9 ms.
constexpr uint32_t kDirectPoll = 8;     // rounds between looks at the step's state
constexpr uint32_t kDirectTask = 16;    // items per task
constexpr uint32_t kDirectPiece = 512;  // candidates of one row per item
constexpr uint32_t kDirectGrid = 1536;  // blocks of the later passes: what is resident at eight query vertices
static_assert(kDirectGrid * kWaves % kDirectShards == 0, "the waves of a pass share the queues evenly");

// Appends the active lanes' items (one each) to the pass's queue: record(p) is the lane's vertex at
// position p below depth.  Returns false when the shard is full.
template <class Record>
__device__ __forceinline__ bool direct_emit(const DirectQueue& q, uint32_t shard, uint32_t job, uint32_t depth, bool active, uint32_t lo,
                                            uint32_t hi, Record record) {
    const uint64_t m = __ballot(active);
    const uint32_t n = static_cast<uint32_t>(__popcll(m)), lane = lane_id();
    if (!n) return true;
    const uint32_t nt = (n + kDirectTask - 1) / kDirectTask;
    unsigned long long at = 0;
    if (lane == 0) at = atomicAdd(q.out_n + shard * 16, static_cast<unsigned long long>(nt) << 32 | n);
    const uint32_t ib = uniform(__shfl(static_cast<uint32_t>(at), 0, 64)), tb = uniform(__shfl(static_cast<uint32_t>(at >> 32), 0, 64));
    const bool fits = static_cast<uint64_t>(ib) + n <= q.cap;
    if (lane < nt && static_cast<uint64_t>(tb) + lane < q.cap)  // a task that does not fit is empty
        q.out_tasks[static_cast<uint64_t>(shard) * q.cap + tb + lane] =
            make_uint4(job, depth, ib + lane * kDirectTask, fits ? min(kDirectTask, n - lane * kDirectTask) : 0u);
    if (!fits) return false;
    if (active) {
        uint32_t* o = q.out_items + (static_cast<uint64_t>(shard) * q.cap + ib + lanes_below(m)) * q.stride;
        o[0] = lo;
        o[1] = hi;
        for (uint32_t p = 0; p < depth; p++) o[2 + p] = record(p);
    }
    return true;
}

template <bool kFirst>
__global__ void __launch_bounds__(kWaves * 64) k_direct_search(DevGraph g, const DirectJob* __restrict__ jobs, DirectCtr* ctr,
                                                                const uint32_t* pairs, uint32_t cap, DirectQueue q, uint32_t max_rounds,
                                                                unsigned long long max_work) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
    const uint32_t gw = (kFirst ? blockIdx.y * gridDim.x + blockIdx.x : blockIdx.x) * kWaves + wv;
    const uint32_t out_shard = gw % kDirectShards;
    unsigned char* const wave_base = lds_raw + wv * q.wave_lds;
    DfsHdr& H = *reinterpret_cast<DfsHdr*>(wave_base);
    uint32_t* const f = reinterpret_cast<uint32_t*>(wave_base + sizeof(DfsHdr));

    // this wave's tasks: groups of the job's anchors, or every so-many-th task of its queue
    uint32_t job = blockIdx.y, ntasks, G = 0, np = 0, t, t_step;
    if (kFirst) {
        np = ctr[job].n_pairs;
        if (!np) return;
        if (np > cap) {
            if (blockIdx.x == 0 && threadIdx.x == 0) ctr[job].fail = 1;
            return;
        }
        t = blockIdx.x * kWaves + wv;
        t_step = gridDim.x * kWaves;
        G = min(64u, (np + t_step - 1) / t_step);
        ntasks = (np + G - 1) / G;
    } else {
        ntasks = static_cast<uint32_t>(min(q.in_n[out_shard * 16] >> 32, static_cast<unsigned long long>(q.cap)));
        t = gw / kDirectShards;
        t_step = gridDim.x * kWaves / kDirectShards;
    }
    for (; t < ntasks; t += t_step) {
        uint32_t depth0 = 2, rows0, stride = 2;
        const uint32_t* in = pairs + 2ull * cap * job;
        if (kFirst) {
            rows0 = min(G, np - t * G);
            if (lane < rows0) {
                H.rec[lane] = t * G + lane;
                H.chunk[lane] = 0;
                H.chunks[lane] = 0xFFFFFFFFu;
            }
        } else {
            const uint4 task = q.in_tasks[static_cast<uint64_t>(out_shard) * q.cap + t];
            job = uniform(task.x);
            depth0 = uniform(task.y);
            rows0 = uniform(task.w);
            stride = q.stride;
            in = q.in_items + (static_cast<uint64_t>(out_shard) * q.cap + uniform(task.z)) * stride;
            if (lane < rows0) {
                H.rec[lane] = lane;
                H.chunk[lane] = in[lane * stride];
                H.chunks[lane] = in[lane * stride + 1];
            }
            in += 2;
        }
        DirectCtr& C = ctr[job];
        const StepDesc& d = jobs[job].d;
        if (!rows0 || uniform(__hip_atomic_load(&C.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) continue;
        unsigned long long my_cnt = 0, my_hash = 0, my_bytes = 0;
        const bool count_bytes = q.bytes != nullptr;  // of rows that are new: the pieces of a row are counted with the row
        if (kFirst && d.n == 2) {
            if (lane < rows0) {
                const uint32_t* r = in + 2 * (t * G + lane);
                my_cnt = 1;
                my_hash = embedding_hash(pair_hash(d.order[0], r[0]) + pair_hash(d.order[1], r[1]));
            }
        } else {
            wave_sync();
            DfsBuf* const buf = reinterpret_cast<DfsBuf*>(wave_base + sizeof(DfsHdr) + (d.n - 1) * 256u);
            const uint32_t last = d.n - 1 - depth0;
            uint32_t j = 0, built = 0, rounds = 0, state = 0;  // state 1: hand the rest on, 2: given up
            const uint32_t total0 = dfs_rows<true>(g, d, depth0, 0, rows0, in, stride, H, f, buf, lane, my_bytes, count_bytes);
            if (total0 > kFrameMax) state = 2;  // far more than a step may have
            unsigned long long work = total0;
            if (lane == 0) {
                H.rows[0] = rows0;
                H.waiting[0] = 0;
                H.cur[0] = 0;
                H.tot[0] = total0;
            }
            wave_sync();
            while (!state) {
                const uint32_t cur = uniform(H.cur[j]), tot = uniform(H.tot[j]);
                const uint32_t waiting = j < last ? uniform(H.waiting[j]) : 0u;
                const bool down = waiting >= 64 || (cur >= tot && waiting);
                if (!down && cur >= tot) {
                    if (j == 0) break;
                    j -= 1;
                    dfs_pop(H, buf, j, lane);
                    continue;
                }
                rounds += 1;
                if (rounds % kDirectPoll == 0 || rounds > max_rounds) {
                    unsigned long long w = 0;
                    if (lane == 0) w = atomicAdd(&C.work, work);
                    work = 0;
                    if (uniform(__shfl(static_cast<uint32_t>(w > max_work), 0, 64)) ||
                        uniform(__hip_atomic_load(&C.fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
                        state = 2;
                    else if (rounds > max_rounds) state = 1;
                    if (state) break;
                }
                if (down) {  // descend with a batch
                    uint32_t rows = min(64u, waiting);
                    j += 1;
                    const uint32_t tj = dfs_rows<true>(g, d, depth0, j, rows, in, stride, H, f, buf, lane, my_bytes, count_bytes);
                    if (tj > kFrameMax) state = 2;
                    work += tj;
                    built = j;
                    if (lane == 0) {
                        H.rows[j] = rows;
                        H.waiting[j] = 0;
                        H.cur[j] = 0;
                        H.tot[j] = tj;
                    }
                    wave_sync();
                    continue;
                }
                if (built != j) {
                    uint32_t rows = uniform(H.rows[j]);
                    dfs_rows<true>(g, d, depth0, j, rows, in, stride, H, f, buf, lane, my_bytes, false);
                    built = j;
                }
                const uint32_t depth = depth0 + j;
                uint32_t k[kDfsIlp], c[kDfsIlp];
                bool ok[kDfsIlp];
                dfs_round(g, d, depth, cur, tot, H, f, lane, k, c, ok);
                if (lane == 0) H.cur[j] = cur + 64 * kDfsIlp;
                if (count_bytes)
                    for (uint32_t u = 0; u < kDfsIlp; u++) my_bytes += ok[u] ? 4u : 0u;
                if (j < last) {
                    uint32_t at = waiting;
#pragma unroll
                    for (uint32_t u = 0; u < kDfsIlp; u++) {
                        const uint64_t m = __ballot(ok[u]);
                        if (ok[u]) {
                            const uint32_t x = at + lanes_below(m);
                            buf[j].cand[x] = c[u];
                            buf[j].parent[x] = static_cast<uint8_t>(k[u]);
                        }
                        at += static_cast<uint32_t>(__popcll(m));
                    }
                    if (lane == 0) H.waiting[j] = at;
                } else {
#pragma unroll
                    for (uint32_t u = 0; u < kDfsIlp; u++)
                        if (ok[u]) {
                            my_cnt += 1;
                            my_hash += embedding_hash(H.ph[k[u]] + pair_hash(d.order[depth], c[u]));
                        }
                }
                wave_sync();
            }
            if (state == 1) {  // the rest of every frame, deepest first
                if (lane == 0) __hip_atomic_store(&C.handed, q.pass + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                uint32_t searched = 0;  // rows of the frame's buffer that are the next frame's
                bool fits = true;
                for (uint32_t jj = j + 1; jj-- > 0;) {
                    uint32_t rows = uniform(H.rows[jj]);
                    const uint32_t cur = uniform(H.cur[jj]), tot = uniform(H.tot[jj]), depth = depth0 + jj;
                    if (built != jj) {
                        dfs_rows<true>(g, d, depth0, jj, rows, in, stride, H, f, buf, lane, my_bytes, false);
                        built = jj;
                    }
                    const uint32_t pre = H.pre[lane], end = lane < 63 ? H.pre[lane + 1] : tot, from = max(cur, pre);
                    uint32_t lo = 0, hi = 0;
                    if (lane < rows && from < end) {
                        lo = H.skip[lane] + (from - pre);
                        hi = H.skip[lane] + (end - pre);
                    }
                    while (__ballot(lo < hi)) {
                        fits = direct_emit(q, out_shard, job, depth, lo < hi, lo, min(hi, lo + kDirectPiece),
                                           [&](uint32_t p) { return f[p * 64 + lane]; }) && fits;
                        lo += kDirectPiece;  // runs are shorter than 2^32 - kDirectPiece
                    }
                    if (jj < last) {
                        const uint32_t waiting = uniform(H.waiting[jj]);
                        for (uint32_t x0 = searched; x0 < waiting; x0 += 64) {
                            const uint32_t x = x0 + lane;
                            const uint32_t par = x < waiting ? buf[jj].parent[x] : 0u, v = x < waiting ? buf[jj].cand[x] : 0u;
                            fits = direct_emit(q, out_shard, job, depth + 1, x < waiting, 0u, 0xFFFFFFFFu,
                                               [&](uint32_t p) { return p < depth ? f[p * 64 + par] : v; }) && fits;
                        }
                    }
                    searched = rows;
                    wave_sync();
                }
                if (!fits) state = 2;
            }
            if (lane == 0) {
                if (state == 2) __hip_atomic_store(&C.fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (work) atomicAdd(&C.work, work);
            }
        }
        my_cnt = wave_sum_u64(my_cnt);
        my_hash = wave_sum_u64(my_hash);
        if (lane == 0 && my_cnt) { atomicAdd(&C.count, my_cnt); atomicAdd(&C.hash, my_hash); }
        if (count_bytes) {
            my_bytes = wave_sum_u64(my_bytes);
            if (lane == 0 && my_bytes) atomicAdd(q.bytes, my_bytes);
        }
    }
}

__global__ void __launch_bounds__(256) k_direct_commit(const DirectJob* jobs, const DirectCtr* ctr, uint32_t njobs, DirectQueue q,
                                                       uint32_t committed, unsigned long long* results, uint32_t* state) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kDirectShards) state[njobs + i] = static_cast<uint32_t>(q.out_n[i * 16] >> 32);
    if (i >= njobs) return;
    const DirectCtr& C = ctr[i];
    if (committed && C.handed < committed) return;  // an earlier commit's
    const bool on = C.handed == q.pass + 1;
    state[i] = C.fail ? 1u : on ? 2u : 0u;
    if (C.fail || on || !C.count) return;
    unsigned long long* r = results + 4ull * jobs[i].result + 2 * jobs[i].d.phase;
    atomicAdd(r, C.count);
    atomicAdd(r + 1, C.hash);
}

// ---- One level, flattened over the whole level ------------------------------------------------
// k_level_len: per record, the view runs of all backward entries of depth d0 (entry order, stored
// at runs[i * E ..], E = entries of the depth) and the entry whose view sequence is the shortest:
// that one generates the record's candidates, the others are probed (the candidate set is their
// intersection whichever entry generates it).  Its length goes to len[i] and, when counting, the
// record's prefix hash to ph[i].  After an exclusive scan, k_level_flat gives one thread per
// candidate of the whole level: thread t finds its record by binary search over the offsets, so
// skewed records spread over the grid, and probes the precomputed runs (no directory or delta
// segment lookups per candidate).
// Algorithmic bytes (as the DFS kernel's frames): every view run of the depth's backward lists
// read once per record, plus 4 per passing candidate (counted by k_level_flat).
constexpr uint32_t kRunsUnroll = 4;  // entries whose lookups are all issued before the first store

__device__ __forceinline__ uint32_t record_runs(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* f, uint4* runs,
                                                uint4* prun, uint8_t* piv, unsigned long long* ph, unsigned long long& bytes,
                                                bool count_bytes) {
    const uint32_t e0 = d.boff[d0], ne = d.boff[d0 + 1] - e0;
    uint32_t best = 0xFFFFFFFFu, tag = 0;
    uint4 brun = make_uint4(0, 0, 0, 0);
    auto take = [&](uint32_t e, const RunView& rv) {
        const BackEntry be = d.be[e0 + e];
        const uint4 x = make_uint4(rv.lo, rv.hi, rv.dlo, rv.dhi);
        if (ne > 1) runs[e] = x;
        const uint32_t len = run_seq_len(rv, be.view);
        if (len < best) {
            best = len;
            brun = x;
            tag = e | static_cast<uint32_t>(be.view) << 4 | static_cast<uint32_t>(be.dir) << 6;
        }
        if (count_bytes) bytes += 4ull * ((rv.hi - rv.lo) + (rv.dhi - rv.dlo));
    };
    // the stores below may alias the graph for the compiler: look the first entries up first, so
    // their dependent loads overlap
    RunView rv[kRunsUnroll];
#pragma unroll
    for (uint32_t e = 0; e < kRunsUnroll; e++) {
        if (e >= ne) break;
        const BackEntry be = d.be[e0 + e];
        rv[e] = make_run(g, d.phase, be.view, be.dir, f[be.pos], be.slot);
    }
    unsigned long long h = 0;
    if (ph)
        for (uint32_t j = 0; j < d0; j++) h += pair_hash(d.order[j], f[j]);
#pragma unroll
    for (uint32_t e = 0; e < kRunsUnroll; e++) {
        if (e >= ne) break;
        take(e, rv[e]);
    }
    for (uint32_t e = kRunsUnroll; e < ne; e++) {
        const BackEntry be = d.be[e0 + e];
        take(e, make_run(g, d.phase, be.view, be.dir, f[be.pos], be.slot));
    }
    *prun = brun;
    *piv = static_cast<uint8_t>(tag);
    if (ph) *ph = h;
    return best;
}

constexpr uint32_t kSmallThreads = 1024;
// Multi-block level preparation: 256-thread blocks (small enough to find room beside the other
// lanes' kernels), two records per thread.
constexpr uint32_t kLenThreads = 256;
constexpr uint32_t kLenItems = 2;
constexpr uint32_t kLenTile = kLenThreads * kLenItems;
static_assert(kLenTile == kLevelTile, "tile totals are sized by kLevelTile");
constexpr int kChainLenGrid = 512;    // blocks of a chained level's preparation (they loop over tiles)
constexpr int kChainFlatGrid = 1024;  // blocks of a chained level's candidate kernel (four per CU)

// Where level k of a device chain reads its records: false when the level does not run (an
// earlier level stopped the chain or overflowed, or its own input is empty, larger than one call
// takes, or large enough for the host's Cartesian-product decision).  Every thread computes the
// same answer from the host-known start and the counters of the levels before k.
__device__ __forceinline__ bool chain_at(const LevelChain& c, uint32_t k, uint64_t& off, uint32_t& n) {
    const uint32_t* ctr = as_global(c.ctr);
    off = c.off0;
    n = c.n0;
    for (uint32_t j = 0;; j++) {
        if (n == 0 || n > c.cap[j] || n >= c.stop_at[j]) return false;
        if (j == k) return true;
        if (ctr[2 * j + 1]) return false;
        off += static_cast<uint64_t>(n) * (c.depth0 + j);
        n = ctr[2 * j];
    }
}

// Multi-block levels: lengths and runs of the records of tiles blockIdx.x, blockIdx.x + gridDim.x,
// ..., and each tile's candidate total in tile_sum[tile]; level_scan then turns the lengths into
// offsets.
__device__ __forceinline__ void level_len_tiles(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, uint32_t n,
                                                unsigned long long* len, uint4* prun, uint4* runs, uint8_t* piv, unsigned long long* ph,
                                                unsigned long long* tile_sum, unsigned long long* bytes_out) {
    rec = as_global(rec);
    len = as_global(len);
    prun = as_global(prun);
    runs = as_global(runs);
    piv = as_global(piv);
    ph = as_global(ph);
    tile_sum = as_global(tile_sum);
    bytes_out = as_global(bytes_out);
    __shared__ unsigned long long s_wave[kLenThreads / 64];
    const uint32_t ne = d.boff[d0 + 1] - d.boff[d0];
    const uint32_t tiles = (n + kLenTile - 1) / kLenTile;
    unsigned long long bytes = 0;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        unsigned long long l[kLenItems], sum = 0;
#pragma unroll
        for (uint32_t j = 0; j < kLenItems; j++) {
            const uint32_t i = tile * kLenTile + j * kLenThreads + threadIdx.x;
            l[j] = 0;
            if (i >= n) continue;
            l[j] = record_runs(g, d, d0, rec + static_cast<uint64_t>(i) * d0, runs + static_cast<uint64_t>(i) * ne, prun + i, piv + i,
                               ph ? ph + i : nullptr, bytes, bytes_out != nullptr);
            sum += l[j];
        }
        if (tiles == 1) {  // a one-tile level is scanned here (item rows in record order); level_scan skips it
            unsigned long long carry = 0;
#pragma unroll
            for (uint32_t j = 0; j < kLenItems; j++) {
                unsigned long long row;
                const unsigned long long ex = block_scan<kLenThreads>(l[j], s_wave, row);
                const uint32_t i = j * kLenThreads + threadIdx.x;
                if (i < n) len[i] = carry + ex;
                carry += row;
            }
            if (threadIdx.x == 0) len[n] = carry;
            continue;
        }
#pragma unroll
        for (uint32_t j = 0; j < kLenItems; j++) {
            const uint32_t i = tile * kLenTile + j * kLenThreads + threadIdx.x;
            if (i < n) len[i] = l[j];
        }
        unsigned long long total;
        block_scan<kLenThreads>(sum, s_wave, total);
        if (threadIdx.x == 0) tile_sum[tile] = total;
    }
    if (bytes_out) {
        bytes = wave_sum_u64(bytes);
        if (lane_id() == 0 && bytes) atomicAdd(bytes_out, bytes);
    }
}

__global__ void __launch_bounds__(kLenThreads) k_level_len(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, uint32_t n,
                                                             unsigned long long* len, uint4* prun, uint4* runs, uint8_t* piv,
                                                             unsigned long long* ph, unsigned long long* tile_sum, uint32_t* zero,
                                                             unsigned long long* bytes_out) {
    if (zero && blockIdx.x == 0 && threadIdx.x == 0) { zero[0] = 0; zero[1] = 0; }
    level_len_tiles(g, d, d0, rec, n, len, prun, runs, piv, ph, tile_sum, bytes_out);
}

__global__ void __launch_bounds__(kLenThreads) k_level_len_chain(DevGraph g, StepDesc d, LevelChain c, uint32_t k, unsigned long long* len,
                                                                   uint4* prun, uint4* runs, uint8_t* piv, unsigned long long* ph,
                                                                   unsigned long long* tile_sum, unsigned long long* bytes_out) {
    if (k == 0 && blockIdx.x == 0 && threadIdx.x < 2 * kMaxQV) c.ctr[threadIdx.x] = 0;
    uint64_t off;
    uint32_t n;
    if (!chain_at(c, k, off, n)) return;
    level_len_tiles(g, d, c.depth0 + k, c.ring + off, n, len, prun, runs, piv, ph, tile_sum, bytes_out);
}

// Exclusive scan of the lengths in place (total at off[n]): the block of a tile adds the totals of
// the tiles before it (at most a few thousand words, read by the whole block) to the tile's scan.
__device__ __forceinline__ void level_scan_tiles(unsigned long long* off, uint32_t n, const unsigned long long* tile_sum) {
    off = as_global(off);
    tile_sum = as_global(tile_sum);
    __shared__ unsigned long long s_wave[kLenThreads / 64];
    const uint32_t tiles = (n + kLenTile - 1) / kLenTile;
    if (tiles == 1) return;  // scanned by level_len_tiles
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        unsigned long long carry = 0, total;
        for (uint32_t t = threadIdx.x; t < tile; t += kLenThreads) carry += tile_sum[t];
        carry = wave_sum_u64(carry);
        if (lane_id() == 0) s_wave[threadIdx.x >> 6] = carry;
        __syncthreads();
        carry = 0;
        for (uint32_t w = 0; w < kLenThreads / 64; w++) carry += s_wave[w];
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < kLenItems; j++) {
            const uint32_t i = tile * kLenTile + j * kLenThreads + threadIdx.x;
            const unsigned long long v = i < n ? off[i] : 0ull;
            const unsigned long long ex = block_scan<kLenThreads>(v, s_wave, total);
            if (i < n) off[i] = carry + ex;
            carry += total;
        }
        if (tile == tiles - 1 && threadIdx.x == 0) off[n] = carry;
    }
}

__global__ void __launch_bounds__(kLenThreads) k_level_scan(unsigned long long* off, uint32_t n, const unsigned long long* tile_sum) {
    level_scan_tiles(off, n, tile_sum);
}

__global__ void __launch_bounds__(kLenThreads) k_level_scan_chain(LevelChain c, uint32_t k, unsigned long long* off,
                                                                    const unsigned long long* tile_sum) {
    uint64_t o;
    uint32_t n;
    if (!chain_at(c, k, o, n)) return;
    level_scan_tiles(off, n, tile_sum);
}

// Levels of under kSmallLevel records (most of them): sizes and scan in one single-block launch.
constexpr uint32_t kSmallItems = 4;
constexpr uint32_t kSmallLevel = kSmallThreads * kSmallItems;

__global__ void __launch_bounds__(kSmallThreads) k_level_len_small(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, uint32_t n,
                                                                   unsigned long long* off, uint4* prun, uint4* runs, uint8_t* piv,
                                                                   unsigned long long* ph, uint32_t* zero, unsigned long long* bytes_out) {
    __shared__ unsigned long long s_wave[kSmallThreads / 64];
    const uint32_t tid = threadIdx.x;
    if (zero && tid == 0) { zero[0] = 0; zero[1] = 0; }
    const uint32_t ne = d.boff[d0 + 1] - d.boff[d0];
    unsigned long long len[kSmallItems], bytes = 0;
    // thread tid owns records j * kSmallThreads + tid (independent lookups in flight together)
#pragma unroll
    for (uint32_t j = 0; j < kSmallItems; j++) {
        const uint32_t i = j * kSmallThreads + tid;
        len[j] = 0;
        if (i >= n) continue;
        len[j] = record_runs(g, d, d0, rec + static_cast<uint64_t>(i) * d0, runs + static_cast<uint64_t>(i) * ne, prun + i, piv + i,
                             ph ? ph + i : nullptr, bytes, bytes_out != nullptr);
    }
    // exclusive scan in record order: one block scan per item row, carried over the rows
    unsigned long long carry = 0;
    for (uint32_t j = 0; j < kSmallItems && j * kSmallThreads < n; j++) {
        unsigned long long total;
        const unsigned long long ex = block_scan<kSmallThreads>(len[j], s_wave, total);
        const uint32_t i = j * kSmallThreads + tid;
        if (i < n) off[i] = carry + ex;
        carry += total;
    }
    if (tid == 0) off[n] = carry;
    if (bytes_out) {
        bytes = wave_sum_u64(bytes);
        if (lane_id() == 0 && bytes) atomicAdd(bytes_out, bytes);
    }
}

// Each wave walks one contiguous range of the level's candidates (equal shares, multiples of
// kLevelStep).  It finds the record of its first candidate with a 64-ary search; per kLevelStep
// candidates it loads the next kLevelStep + 1 record offsets into LDS (coalesced) and each lane
// finds the records of its kLevelIlp candidates there (a global search only past the window, when
// records have under one candidate each).  The kLevelIlp candidates of a lane are tested in
// lock-step so their independent loads are in flight together: the kernel is latency-bound.  Four
// candidates per lane keep the kernel at 76 VGPRs, six waves per SIMD; with the lock-step searches
// that beat eight (four waves per SIMD) and two on the 400K-vertex Chung-Lu workload.
constexpr uint32_t kLevelIlp = 4;
constexpr uint32_t kLevelStep = 64 * kLevelIlp;
static_assert((kLevelStep & (kLevelStep - 1)) == 0, "the window search takes power-of-two steps");

// Write mode stages passing (record, candidate) pairs per wave in LDS and reserves ring space once
// per kOutFlush pairs: an atomic per iteration would put its round trip on every iteration.
constexpr uint32_t kOutFlush = 256;
constexpr uint32_t kOutBuf = kOutFlush + kLevelStep;

__device__ __forceinline__ void flush_records(const uint32_t* rec, uint32_t d0, const uint32_t* sk, const uint32_t* sc, uint32_t cnt, Ring& r,
                                              uint32_t lane) {
    uint32_t wb = 0;
    if (lane == 0) wb = atomicAdd(r.out_count, cnt);
    wb = uniform(__shfl(wb, 0, 64));
    if (static_cast<uint64_t>(wb) + cnt > r.out_cap) {
        if (lane == 0) atomicOr(r.overflow, 1u);
        return;
    }
    // consecutive words of the reserved region: coalesced stores
    const uint32_t rw = d0 + 1;
    uint32_t* o = r.out + static_cast<uint64_t>(wb) * rw;
    for (uint32_t w = lane; w < cnt * rw; w += 64) {
        const uint32_t e = w / rw, q = w - e * rw;
        uint32_t v = sc[e];  // read before the branch: one load of either would be a flat one
        if (q < d0) v = rec[static_cast<uint64_t>(sk[e]) * d0 + q];
        o[w] = v;
    }
}

template <int kMode>
__device__ __forceinline__ void level_flat_body(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, uint32_t n,
                                                const unsigned long long* off, const uint4* prun, const uint4* runs, const uint8_t* piv,
                                                const unsigned long long* ph, Ring r, MatchOut out) {
    rec = as_global(rec);
    off = as_global(off);
    prun = as_global(prun);
    runs = as_global(runs);
    piv = as_global(piv);
    ph = as_global(ph);
    r.out = as_global(r.out);
    r.out_count = as_global(r.out_count);
    r.overflow = as_global(r.overflow);
    out = MatchOut{as_global(out.count), as_global(out.hash), as_global(out.bytes)};
    // window of record offsets, relative to off[rb] (a window spans fewer than 2^32 candidates)
    __shared__ uint32_t s_win[4][kLevelStep + 1];
    __shared__ uint32_t s_out[4][kMode == kWriteAtEnd ? 2 * kOutBuf : 1];
    const uint32_t lane = lane_id();
    uint32_t* win = s_win[threadIdx.x >> 6];
    uint32_t* const out_k = s_out[threadIdx.x >> 6];
    uint32_t* const out_c = out_k + (kMode == kWriteAtEnd ? kOutBuf : 0);
    uint32_t staged = 0;  // pairs in the wave's LDS buffer
    const uint32_t e0 = d.boff[d0], ne = d.boff[d0 + 1] - e0;
    const uint32_t* filter = as_global(d.filter[d0]);
    const uint32_t qv = d.order[d0], inj = uniform(d.inj[d0]);
    const unsigned long long total = off[n];
    const unsigned long long waves = static_cast<unsigned long long>(gridDim.x) * (blockDim.x >> 6);
    const unsigned long long gw = static_cast<unsigned long long>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const unsigned long long per = ((total + waves - 1) / waves + kLevelStep - 1) / kLevelStep * kLevelStep;
    const unsigned long long w0 = gw * per, w1 = min(total, w0 + per);
    unsigned long long cnt = 0, hsum = 0, bytes = 0;
    uint32_t rb = w0 < total ? find_record(off, n, w0, lane) : 0u;  // off[rb] <= w0
    for (unsigned long long t0 = w0; t0 < w1; t0 += kLevelStep) {
        // a level that overflows is redone by the host with fewer records: stop early (polled every
        // 16 iterations; a load per iteration would sit on every iteration's latency chain)
        if (kMode == kWriteAtEnd && ((t0 - w0) & (16ull * kLevelStep - 1)) == 0 && t0 != w0 &&
            uniform(__hip_atomic_load(r.overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
            break;
        const unsigned long long wbase = off[rb];
        auto rel = [&](uint32_t i) {
            return static_cast<uint32_t>(min(off[min(rb + i, n)] - wbase, 0xFFFFFFFFull));
        };
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) win[lane + 64 * j] = rel(lane + 64 * j);
        if (lane == 0) win[kLevelStep] = rel(kLevelStep);
        wave_sync();
        unsigned long long t[kLevelIlp];
        uint32_t k[kLevelIlp], key[kLevelIlp], c[kLevelIlp];
        bool ok[kLevelIlp];
        // record of each candidate: last i < kLevelStep with win[i] <= t - off[rb] (win[0] <= t0 <= t),
        // a fixed-step search run for all kLevelIlp candidates at once so their LDS reads overlap
        uint32_t tr[kLevelIlp], pos[kLevelIlp];
        bool past = false;
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) {
            t[j] = t0 + 64 * j + lane;
            ok[j] = t[j] < w1;
            const unsigned long long x = ok[j] ? t[j] - wbase : 0ull;  // < 2^32: inside record rb or the window
            tr[j] = static_cast<uint32_t>(min(x, 0xFFFFFFFFull));
            past = past || (ok[j] && win[kLevelStep] <= x);
            pos[j] = 0;
        }
#pragma unroll
        for (uint32_t st = kLevelStep / 2; st; st >>= 1) {
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++)
                if (win[pos[j] + st] <= tr[j]) pos[j] += st;
        }
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) k[j] = rb + pos[j];
        if (past) {  // records with fewer than one candidate each: last k in [rb + kLevelStep, n) with off[k] <= t
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) {
                if (!ok[j] || win[kLevelStep] > t[j] - wbase) continue;
                uint32_t lo = rb + kLevelStep, hi = n;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (off[mid] <= t[j]) lo = mid;
                    else hi = mid;
                }
                k[j] = lo;
            }
        }
        // the record's generating run (prun) and its entry | view << 4 | dir << 6 (piv): independent loads
        RunView rv[kLevelIlp];
        unsigned long long base[kLevelIlp];
        uint32_t pv[kLevelIlp];
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) {
            rv[j] = RunView{0, 0, 0, 0};
            base[j] = 0;
            pv[j] = 0;
            if (!ok[j]) continue;
            const uint4 x = prun[k[j]];
            rv[j] = RunView{x.x, x.y, x.z, x.w};
            pv[j] = piv[k[j]];
            base[j] = k[j] - rb < kLevelStep ? wbase + win[k[j] - rb] : off[k[j]];
        }
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) {
            const uint32_t view = (pv[j] >> 4) & 3u;
            key[j] = ok[j] ? run_elem(g, phase_delta(g, pv[j] >> 6, d.phase), rv[j], run_base_len(rv[j], view),
                                      static_cast<uint32_t>(t[j] - base[j]))
                           : 0u;
            c[j] = key[j] & g.id_mask;
        }
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++) ok[j] = ok[j] && bit_test(filter, c[j]);
#pragma unroll
        for (uint32_t j = 0; j < kLevelIlp; j++)
            ok[j] = ok[j] && run_elem_live(phase_delta(g, pv[j] >> 6, d.phase), rv[j], (pv[j] >> 4) & 3u, key[j]);
        for (uint32_t im = inj; im; im &= im - 1) {
            const uint32_t q = static_cast<uint32_t>(__ffs(im)) - 1;
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) ok[j] = ok[j] && rec[static_cast<uint64_t>(k[j]) * d0 + q] != c[j];
        }
        // probe the other entries' precomputed runs (each with its own slot bits); the searches of
        // the kLevelIlp candidates advance in lock-step so their loads are in flight together
        for (uint32_t e = 0; e < ne; e++) {
            const BackEntry be = load_entry(d.be + e0 + e);
            const uint32_t hi_bits = be.slot << g.id_bits;
            // runs as {lo, hi} / {dlo, dhi} halves: the delta half is loaded only for views that use it
            const uint2* rh = reinterpret_cast<const uint2*>(runs);
            uint32_t pk[kLevelIlp];
            bool act[kLevelIlp], inb[kLevelIlp], ind[kLevelIlp];
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) {
                act[j] = ok[j] && (pv[j] & 15u) != e;
                pk[j] = hi_bits | c[j];
                inb[j] = false;
                ind[j] = false;
            }
            if (be.view != kViewDelta) {
                uint32_t lo[kLevelIlp], hi[kLevelIlp];
#pragma unroll
                for (uint32_t j = 0; j < kLevelIlp; j++) {
                    const uint2 x = act[j] ? rh[2 * (static_cast<uint64_t>(k[j]) * ne + e)] : make_uint2(0, 0);
                    lo[j] = x.x;
                    hi[j] = x.y;
                }
                contains_many<kLevelIlp>(g.arena, lo, hi, pk, act, inb);
            }
            if (be.view != kViewBase) {
                const uint32_t* dl = phase_delta(g, be.dir, d.phase);
                uint32_t lo[kLevelIlp], hi[kLevelIlp];
                bool need[kLevelIlp];
#pragma unroll
                for (uint32_t j = 0; j < kLevelIlp; j++) {
                    need[j] = act[j] && (be.view == kViewDelta || (be.view == kViewBasePlusDelta ? !inb[j] : inb[j]));
                    const uint2 x = need[j] ? rh[2 * (static_cast<uint64_t>(k[j]) * ne + e) + 1] : make_uint2(0, 0);
                    lo[j] = x.x;
                    hi[j] = x.y;
                }
                contains_many<kLevelIlp>(dl, lo, hi, pk, need, ind);
            }
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) {
                if (!act[j]) continue;
                switch (be.view) {
                    case kViewBase: ok[j] = inb[j]; break;
                    case kViewBasePlusDelta: ok[j] = inb[j] || ind[j]; break;
                    case kViewDelta: ok[j] = ind[j]; break;
                    default: ok[j] = inb[j] && !ind[j]; break;
                }
            }
        }
        if (kMode == kCountAtEnd) {
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++)
                if (ok[j]) {
                    cnt += 1;
                    hsum += embedding_hash(ph[k[j]] + pair_hash(qv, c[j]));
                }
        } else {
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) {
                const uint64_t m = __ballot(ok[j]);
                if (ok[j]) {
                    const uint32_t idx = staged + lanes_below(m);
                    out_k[idx] = k[j];
                    out_c[idx] = c[j];
                }
                staged += static_cast<uint32_t>(__popcll(m));
            }
            if (staged >= kOutFlush || t0 + kLevelStep >= w1) {
                wave_sync();
                if (staged) flush_records(rec, d0, out_k, out_c, staged, r, lane);
                staged = 0;
            }
        }
        if (out.bytes) {
#pragma unroll
            for (uint32_t j = 0; j < kLevelIlp; j++) bytes += ok[j] ? 4 : 0;
        }
        rb = uniform(__shfl(k[kLevelIlp - 1], 63, 64));  // highest record of this step (all lanes valid unless last)
        wave_sync();                                    // the window is rewritten next iteration
    }
    if (kMode == kCountAtEnd) {
        // one pair of device atomics per block (they serialise on one address across the grid)
        __shared__ unsigned long long s_cnt[4], s_hash[4];
        cnt = wave_sum_u64(cnt);
        hsum = wave_sum_u64(hsum);
        if (lane == 0) { s_cnt[threadIdx.x >> 6] = cnt; s_hash[threadIdx.x >> 6] = hsum; }
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long c = 0, h = 0;
            for (uint32_t w = 0; w < (blockDim.x >> 6); w++) { c += s_cnt[w]; h += s_hash[w]; }
            if (c) { atomicAdd(out.count, c); atomicAdd(out.hash, h); }
        }
    }
    if (out.bytes) {
        bytes = wave_sum_u64(bytes);
        if (lane == 0 && bytes) atomicAdd(out.bytes, bytes);
    }
}

template <int kMode>
__global__ void __launch_bounds__(256) k_level_flat(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, uint32_t n,
                                                    const unsigned long long* off, const uint4* prun, const uint4* runs,
                                                    const uint8_t* piv, const unsigned long long* ph, Ring r, MatchOut out) {
    level_flat_body<kMode>(g, d, d0, rec, n, off, prun, runs, piv, ph, r, out);
}

// Level k of a device chain: reads its records where chain_at says and writes the records of the
// next depth right after them ({count, overflow} in ctr[2k], ctr[2k + 1]).
template <int kMode>
__global__ void __launch_bounds__(256) k_level_flat_chain(DevGraph g, StepDesc d, LevelChain c, uint32_t k, const unsigned long long* off,
                                                          const uint4* prun, const uint4* runs, const uint8_t* piv,
                                                          const unsigned long long* ph, MatchOut out) {
    uint64_t o;
    uint32_t n;
    if (!chain_at(c, k, o, n)) return;
    const uint32_t d0 = c.depth0 + k;
    const uint64_t out_off = o + static_cast<uint64_t>(n) * d0;
    const uint64_t room = out_off < c.ring_words ? (c.ring_words - out_off) / (d0 + 1) : 0ull;
    const Ring r{c.ring + o, nullptr, n, c.ring + out_off, c.ctr + 2 * k, static_cast<uint32_t>(min(room, 0xFFFFFFFFull)),
                 c.ctr + 2 * k + 1};
    level_flat_body<kMode>(g, d, d0, c.ring + o, n, off, prun, runs, piv, ph, r, out);
}

// Level k of many steps' chains (grid.y = job): the kernels above with the job's descriptor, chain
// and scratch read from the job table (uniform per block: scalar loads).
__global__ void __launch_bounds__(kLenThreads) k_level_len_chain_multi(DevGraph g, const ChainJob* jobs, uint32_t k) {
    const ChainJob& J = jobs[blockIdx.y];
    if (k > J.L) return;
    if (k == 0 && blockIdx.x == 0 && threadIdx.x < 2 * kMaxQV) as_global(J.c.ctr)[threadIdx.x] = 0;
    uint64_t off;
    uint32_t n;
    if (!chain_at(J.c, k, off, n)) return;
    const bool counting = k == J.L;
    level_len_tiles(g, J.d, J.c.depth0 + k, J.c.ring + off, n, J.ls.off, J.ls.prun, J.ls.runs, J.ls.piv, counting ? J.ls.ph : nullptr,
                    J.ls.tile_sum, counting ? J.out.bytes : J.write_bytes);
}

__global__ void __launch_bounds__(kLenThreads) k_level_scan_chain_multi(const ChainJob* jobs, uint32_t k) {
    const ChainJob& J = jobs[blockIdx.y];
    if (k > J.L) return;
    uint64_t o;
    uint32_t n;
    if (!chain_at(J.c, k, o, n)) return;
    level_scan_tiles(J.ls.off, n, J.ls.tile_sum);
}

// At least six waves per SIMD (74 and 80 VGPRs, no spills).  The kernel is latency-bound and shares the
// GPU with the other teams' launches: six waves measured faster than the five that the writing form
// takes unbounded.
template <int kMode>
__global__ void __launch_bounds__(256, 6) k_level_flat_chain_multi(DevGraph g, const ChainJob* jobs, uint32_t k) {
    const ChainJob& J = jobs[blockIdx.y];
    if (k > J.L || (k == J.L) != (kMode == kCountAtEnd)) return;
    uint64_t o;
    uint32_t n;
    if (!chain_at(J.c, k, o, n)) return;
    const uint32_t d0 = J.c.depth0 + k;
    const uint64_t out_off = o + static_cast<uint64_t>(n) * d0;
    const uint64_t room = out_off < J.c.ring_words ? (J.c.ring_words - out_off) / (d0 + 1) : 0ull;
    const Ring r{J.c.ring + o, nullptr, n, J.c.ring + out_off, J.c.ctr + 2 * k, static_cast<uint32_t>(min(room, 0xFFFFFFFFull)),
                 J.c.ctr + 2 * k + 1};
    const MatchOut out = kMode == kCountAtEnd ? J.out : MatchOut{nullptr, nullptr, J.write_bytes};
    level_flat_body<kMode>(g, J.d, d0, J.c.ring + o, n, J.ls.off, J.ls.prun, J.ls.runs, J.ls.piv, J.ls.ph, r, out);
}

__global__ void __launch_bounds__(256) k_root_chunks(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, const uint32_t* n_rec,
                                                     uint32_t max_rec, uint32_t max_chunks, unsigned long long* chunks) {
    const uint32_t n = min(*n_rec, max_rec);
    const BackEntry be = d.be[d.pivot[d0]];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t v = rec[static_cast<uint64_t>(i) * d0 + be.pos];
        const RunView rv = make_run(g, d.phase, be.view, be.dir, v, be.slot);
        chunks[i] = min(max_chunks, (run_seq_len(rv, be.view) + 63u) / 64u);
    }
}

__global__ void k_init_from_pairs(const uint32_t* pairs, const uint32_t* n_pairs, uint32_t max_pairs, int swap, uint32_t* out,
                                  uint32_t* out_count) {
    const uint32_t n = min(*n_pairs, max_pairs);
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t a = pairs[2 * i], b = pairs[2 * i + 1];
        out[2 * i] = swap ? b : a;
        out[2 * i + 1] = swap ? a : b;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *out_count = n;
}

// Pairs (v, x) with v in the start list, x in the view run of v along a->b and x in filter(b).
// The runs of a wave's G start vertices are flattened (a wave prefix of their lengths, one element
// per lane per round, its vertex found by a search of the prefix in LDS), and the wave reserves
// its survivors' output once per round of kInitIlp elements a lane, whose loads are in flight
// together: most start vertices have a run of a few elements.
constexpr uint32_t kInitIlp = 4;
__device__ __forceinline__ void init_set_body(const DevGraph& g, InitJob J) {
    J.list = as_global(J.list);
    J.len = as_global(J.len);
    J.filter_b = as_global(J.filter_b);
    J.out = as_global(J.out);
    J.out_count = as_global(J.out_count);
    J.overflow = as_global(J.overflow);
    __shared__ uint32_t s_pre[4][65];
    __shared__ RunView s_run[4][64];
    __shared__ uint32_t s_nb[4][64], s_v[4][64];
    const uint32_t lane = lane_id(), wv = threadIdx.x >> 6;
    const uint32_t gw = blockIdx.x * (blockDim.x >> 6) + wv, waves = gridDim.x * (blockDim.x >> 6);
    const uint32_t n = min(*J.len, J.max_len);
    const uint32_t* dl = phase_delta(g, J.dir, J.phase);
    const uint32_t G = items_per_wave(n);
    for (uint32_t base = gw * G; base < n; base += waves * G) {
        const uint32_t i = base + lane;
        uint32_t tot = 0, nb = 0, v = 0;
        RunView r{0, 0, 0, 0};
        if (lane < G && i < n) {
            v = J.list[i];
            r = make_run(g, J.phase, J.view, J.dir, v, J.slot);
            nb = run_base_len(r, J.view);
            tot = run_seq_len(r, J.view);
        }
        uint32_t T;
        const uint32_t pre = wave_prefix(tot, T);
        s_pre[wv][lane] = pre;
        s_run[wv][lane] = r;
        s_nb[wv][lane] = nb;
        s_v[wv][lane] = v;
        if (lane == 63) s_pre[wv][64] = T;
        wave_sync();
        for (uint32_t e0 = 0; e0 < T; e0 += 64 * kInitIlp) {  // wave-uniform trip count
            uint32_t k[kInitIlp], key[kInitIlp], sv[kInitIlp];
            bool ok[kInitIlp];
            uint64_t m[kInitIlp];
            uint32_t c = 0;
#pragma unroll
            for (uint32_t u = 0; u < kInitIlp; u++) {
                const uint32_t e = e0 + 64 * u + lane;
                ok[u] = e < T;
                k[u] = ok[u] ? owner_of(s_pre[wv], e) : 0u;
                sv[u] = s_v[wv][k[u]];
                key[u] = ok[u] ? run_elem(g, dl, s_run[wv][k[u]], s_nb[wv][k[u]], e - s_pre[wv][k[u]]) : 0u;
            }
#pragma unroll
            for (uint32_t u = 0; u < kInitIlp; u++) {
                const uint32_t x = key[u] & g.id_mask;
                ok[u] = ok[u] && x != sv[u] && bit_test(J.filter_b, x);
            }
#pragma unroll
            for (uint32_t u = 0; u < kInitIlp; u++) {
                ok[u] = ok[u] && run_elem_live(dl, s_run[wv][k[u]], J.view, key[u]);
                m[u] = __ballot(ok[u]);
                c += static_cast<uint32_t>(__popcll(m[u]));
            }
            if (!c) continue;  // wave-uniform
            uint32_t o = 0;
            if (lane == 0) o = atomicAdd(J.out_count, c);
            o = uniform(__shfl(o, 0, 64));
            if (static_cast<uint64_t>(o) + c > J.out_cap) {
                if (lane == 0) atomicOr(J.overflow, 1u);
                continue;
            }
#pragma unroll
            for (uint32_t u = 0; u < kInitIlp; u++) {
                if (ok[u]) reinterpret_cast<uint2*>(J.out)[o + lanes_below(m[u])] = make_uint2(sv[u], key[u] & g.id_mask);
                o += static_cast<uint32_t>(__popcll(m[u]));
            }
        }
        wave_sync();  // the LDS rows are rewritten by the next items
    }
}

__global__ void __launch_bounds__(256) k_init_from_set(DevGraph g, InitJob J) { init_set_body(g, J); }

__global__ void __launch_bounds__(256) k_init_from_set_multi(DevGraph g, const InitJob* jobs) { init_set_body(g, jobs[blockIdx.y]); }

// ---- Cartesian product -------------------------------------------------------------------------
// The trailing leaves d0 .. n-1 of a record each hang off one matched vertex.  A segment is one
// (record, leaf) pair, segment i = record * leaves + leaf.  k_cp_len sizes every segment's view run
// and the record's prefix hash; after a scan, k_cp_filter tests every run element (load-balanced
// over the grid, as k_level_flat) against the leaf's candidate bitmap, deletion liveness and the
// matched prefix, and appends survivors to the segment's list (order within a list is free: the
// enumeration takes every combination once); k_cp_products multiplies the list lengths per record.
__global__ void __launch_bounds__(256) k_cp_len(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, uint32_t n, CpScratch c) {
    const uint32_t nl = d.n - d0;
    const uint64_t nseg = static_cast<uint64_t>(n) * nl;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < nseg; i += static_cast<uint64_t>(gridDim.x) * blockDim.x) {
        const uint32_t r = static_cast<uint32_t>(i / nl), kk = static_cast<uint32_t>(i % nl);
        const uint32_t* f = rec + static_cast<uint64_t>(r) * d0;
        const BackEntry be = d.be[d.boff[d0 + kk]];
        const RunView rv = make_run(g, d.phase, be.view, be.dir, f[be.pos], be.slot);
        c.seg_off[i] = run_seq_len(rv, be.view);
        c.seg_run[i] = make_uint4(rv.lo, rv.hi, rv.dlo, rv.dhi);
        c.seg_cnt[i] = 0;
        if (kk == 0) {
            unsigned long long h = 0;
            for (uint32_t j = 0; j < d0; j++) h += pair_hash(d.order[j], f[j]);
            c.rec_hash[r] = h;
        }
    }
}

__global__ void __launch_bounds__(256) k_cp_filter(DevGraph g, StepDesc d, uint32_t d0, const uint32_t* rec, uint32_t nseg, CpScratch c) {
    __shared__ unsigned long long s_win[4][65];
    const uint32_t lane = lane_id();
    unsigned long long* win = s_win[threadIdx.x >> 6];
    const uint32_t nl = d.n - d0;
    const unsigned long long* off = c.seg_off;
    const unsigned long long total = off[nseg];
    if (total > c.lists_cap) {  // lists do not fit: the host counts these records another way
        if (blockIdx.x == 0 && threadIdx.x == 0) atomicOr(c.err, kErrScratchFull);
        return;
    }
    const unsigned long long waves = static_cast<unsigned long long>(gridDim.x) * (blockDim.x >> 6);
    const unsigned long long gw = static_cast<unsigned long long>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const unsigned long long per = ((total + waves - 1) / waves + 63) & ~63ull;
    const unsigned long long w0 = gw * per, w1 = min(total, w0 + per);
    uint32_t rb = w0 < total ? find_record(off, nseg, w0, lane) : 0u;  // off[rb] <= w0
    for (unsigned long long t0 = w0; t0 < w1; t0 += 64) {
        win[lane] = off[min(rb + lane, nseg)];
        if (lane == 0) win[64] = off[min(rb + 64, nseg)];
        wave_sync();
        const unsigned long long t = t0 + lane;
        uint32_t i = rb, x = 0;
        unsigned long long base = 0;
        bool ok = false;
        if (t < w1) {
            if (win[64] <= t) {
                uint32_t lo = rb + 64, hi = nseg;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (off[mid] <= t) lo = mid;
                    else hi = mid;
                }
                i = lo;
            } else {
                uint32_t lo = 0, hi = 64;
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (win[mid] <= t) lo = mid;
                    else hi = mid;
                }
                i = rb + lo;
            }
            const uint32_t r = i / nl, kk = i % nl;
            const BackEntry be = d.be[d.boff[d0 + kk]];
            const uint32_t* dl = phase_delta(g, be.dir, d.phase);
            const uint4 x4 = c.seg_run[i];
            const RunView rv{x4.x, x4.y, x4.z, x4.w};
            base = i - rb < 64 ? win[i - rb] : off[i];
            const uint32_t key = run_elem(g, dl, rv, run_base_len(rv, be.view), static_cast<uint32_t>(t - base));
            x = key & g.id_mask;
            ok = bit_test(d.filter[d0 + kk], x) && run_elem_live(dl, rv, be.view, key);
            const uint32_t* f = rec + static_cast<uint64_t>(r) * d0;
            for (uint32_t im = d.inj[d0 + kk] & ((1u << d0) - 1u); im && ok; im &= im - 1) ok = f[__ffs(im) - 1] != x;
        }
        // One counter reservation per segment per wave: the lanes of a segment are consecutive
        // (i never decreases along the lanes), so each group's first lane reserves for the group.
        const uint64_t pm = __ballot(ok);
        const uint64_t starts = __ballot(lane == 0 || __shfl_up(i, 1, 64) != i);
        const uint64_t lt = (1ull << lane) - 1ull;
        const uint32_t leader = 63u - static_cast<uint32_t>(__clzll(starts & (lt | (1ull << lane))));
        const uint64_t after = starts & ~(lt | (1ull << lane));  // group starts above this lane
        const uint64_t grp_end = after ? (after & (0ull - after)) : 0ull;  // lowest later start (0: lane 63 ends)
        const uint64_t grp = (grp_end ? grp_end - 1ull : ~0ull) & ~((1ull << leader) - 1ull);
        uint32_t wb = 0;
        if (lane == leader) {
            const uint32_t cnt = static_cast<uint32_t>(__popcll(pm & grp));
            if (cnt) wb = atomicAdd(&c.seg_cnt[i], cnt);
        }
        wb = __shfl(wb, static_cast<int>(leader), 64);
        if (ok) c.lists[base + wb + static_cast<uint32_t>(__popcll(pm & lt & grp))] = x;
        rb = uniform(__shfl(i, 63, 64));
        wave_sync();
    }
}

// Thread per record: the product of its leaf list lengths (0 when a list is empty).
__global__ void __launch_bounds__(256) k_cp_products(StepDesc d, uint32_t d0, uint32_t n, CpScratch c) {
    const uint32_t nl = d.n - d0;
    unsigned long long mx = 0;
    for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
        unsigned long long prod = 1;
        bool overflow = false;
        for (uint32_t kk = 0; kk < nl; kk++) {
            const uint32_t sz = c.seg_cnt[static_cast<uint64_t>(r) * nl + kk];
            if (sz == 0) { prod = 0; break; }
            if (prod > (~0ull >> 1) / sz) overflow = true;
            else prod *= sz;
        }
        if (overflow) {
            atomicOr(c.err, kErrProductOverflow);
            prod = 0;
        }
        c.prod[r] = prod;
        mx = max(mx, prod);
    }
    for (int o = 32; o > 0; o >>= 1) mx = max(mx, static_cast<unsigned long long>(__shfl_xor(mx, o, 64)));
    if (lane_id() == 0 && mx) atomicMax(c.max_prod, mx);
}

// Thread per flattened combination t: record r owns [off[r], off[r+1]); digits of t - off[r] in the
// mixed radix of the leaf list sizes select one candidate per leaf; leaves must be distinct.
__global__ void __launch_bounds__(256) k_cp_enumerate(StepDesc d, uint32_t d0, uint32_t n, CpScratch c, MatchOut out) {
    __shared__ unsigned long long sc[256], sh[256];
    const unsigned long long T = c.prod[n];
    const uint32_t nl = d.n - d0;
    unsigned long long cnt = 0, hsum = 0;
    for (unsigned long long t = blockIdx.x * static_cast<unsigned long long>(blockDim.x) + threadIdx.x; t < T;
         t += static_cast<unsigned long long>(gridDim.x) * blockDim.x) {
        // last record with off[r] <= t
        uint32_t lo = 0, hi = n;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (c.prod[mid] <= t) lo = mid; else hi = mid;
        }
        const uint32_t r = lo;
        unsigned long long local = t - c.prod[r];
        uint32_t x[kMaxQV];
        unsigned long long h = c.rec_hash[r];
        bool ok = true;
        for (uint32_t k = 0; k < nl; k++) {
            const uint64_t i = static_cast<uint64_t>(r) * nl + k;
            const uint32_t sz = c.seg_cnt[i];
            const uint32_t idx = static_cast<uint32_t>(local % sz);
            local /= sz;
            x[k] = c.lists[c.seg_off[i] + idx];
            for (uint32_t j = 0; j < k; j++) ok = ok && (!(d.inj[d0 + k] >> (d0 + j) & 1u) || x[j] != x[k]);
            h += pair_hash(d.order[d0 + k], x[k]);
        }
        if (ok) { cnt += 1; hsum += embedding_hash(h); }
    }
    sc[threadIdx.x] = cnt;
    sh[threadIdx.x] = hsum;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) { sc[threadIdx.x] += sc[threadIdx.x + o]; sh[threadIdx.x] += sh[threadIdx.x + o]; }
        __syncthreads();
    }
    if (threadIdx.x == 0 && sc[0]) { atomicAdd(out.count, sc[0]); atomicAdd(out.hash, sh[0]); }
}

__global__ void __launch_bounds__(256) k_count_records(StepDesc d, const uint32_t* rec, const uint32_t* n_rec, uint32_t max_rec,
                                                       MatchOut out) {
    __shared__ unsigned long long sc[256], sh[256];
    const uint32_t n = min(*n_rec, max_rec);
    unsigned long long cnt = 0, hsum = 0;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        unsigned long long h = 0;
        for (uint32_t j = 0; j < d.n; j++) h += pair_hash(d.order[j], rec[static_cast<uint64_t>(i) * d.n + j]);
        cnt += 1;
        hsum += embedding_hash(h);
    }
    sc[threadIdx.x] = cnt;
    sh[threadIdx.x] = hsum;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if (threadIdx.x < o) { sc[threadIdx.x] += sc[threadIdx.x + o]; sh[threadIdx.x] += sh[threadIdx.x + o]; }
        __syncthreads();
    }
    if (threadIdx.x == 0 && sc[0]) { atomicAdd(out.count, sc[0]); atomicAdd(out.hash, sh[0]); }
}

__global__ void __launch_bounds__(256) k_bitmap_to_list(const uint32_t* bitmap, uint32_t dv, uint32_t* list, uint32_t* len) {
    const uint32_t words = (dv + 31) / 32;
    for (uint32_t w = blockIdx.x * blockDim.x + threadIdx.x; w < words; w += gridDim.x * blockDim.x) {
        uint32_t b = bitmap[w];
        if (!b) continue;
        const uint32_t p = atomicAdd(len, static_cast<uint32_t>(__popc(b)));
        uint32_t k = 0;
        while (b) {
            const uint32_t bit = static_cast<uint32_t>(__ffs(b)) - 1;
            list[p + k++] = w * 32 + bit;
            b &= b - 1;
        }
    }
}

int grid_for(uint64_t n, int per_block, int cap) {
    return static_cast<int>(std::max<uint64_t>(1, std::min<uint64_t>(static_cast<uint64_t>(cap), (n + per_block - 1) / per_block)));
}

}  // namespace

void init_from_pairs(const uint32_t* pairs, const uint32_t* n_pairs, uint32_t max_pairs, bool swap, uint32_t* out,
                     uint32_t* out_count, hipStream_t s) {
    k_init_from_pairs<<<grid_for(max_pairs, 256, 4096), 256, 0, s>>>(pairs, n_pairs, max_pairs, swap ? 1 : 0, out, out_count);
}

void init_from_set(const DevGraph& g, uint32_t phase, uint32_t view, uint32_t dir, uint32_t slot, const uint32_t* list,
                   const uint32_t* len, uint32_t max_len, const uint32_t* filter_b, Ring r, hipStream_t s) {
    const InitJob J{phase, view, dir, slot, list, len, filter_b, r.out, r.out_count, r.overflow, r.out_cap, max_len};
    k_init_from_set<<<grid_for(max_len, 4 * 64, 512), 256, 0, s>>>(g, J);
}

void init_from_set_multi(const DevGraph& g, const InitJob* jobs, uint32_t njobs, hipStream_t s) {
    if (njobs) k_init_from_set_multi<<<dim3(256, njobs), 256, 0, s>>>(g, jobs);
}

void count_records(const StepDesc& d, const uint32_t* rec, const uint32_t* n_rec, uint32_t max_rec, MatchOut out, hipStream_t s) {
    k_count_records<<<grid_for(max_rec, 256, 4096), 256, 0, s>>>(d, rec, n_rec, max_rec, out);
}

void bitmap_to_list(const uint32_t* bitmap, uint32_t dv, uint32_t* list, uint32_t* len, hipStream_t s) {
    k_bitmap_to_list<<<grid_for((dv + 31) / 32, 256, 4096), 256, 0, s>>>(bitmap, dv, list, len);
}

void extend(const DevGraph& g, const StepDesc& d, uint32_t d0, uint32_t end_depth, int mode, Ring r, MatchOut out,
            const unsigned long long* split, unsigned long long* work_counter, int schedule, int blocks, Donation dn, hipStream_t s) {
    // Persistent grid, never more waves than records (a split launch has at least as many items as records
    // with candidates; a donating launch keeps the full grid, its waves share the heavy records' ranges).
    const uint32_t grid = dfs_grid(static_cast<uint32_t>(blocks), r.in_max, split || schedule == 2);
    const size_t lds = static_cast<size_t>(kWaves) * wave_lds_bytes(d0, end_depth);
    if (schedule == 2) fill_u32(reinterpret_cast<uint32_t*>(dn.words), 0u, 4ull * grid * kWaves, s);  // every pair: nothing to take
    if (mode == kCountAtEnd)
        k_extend<kCountAtEnd><<<grid, kWaves * 64, lds, s>>>(g, d, d0, end_depth, r, out, split, work_counter, schedule, dn.words);
    else
        k_extend<kWriteAtEnd><<<grid, kWaves * 64, lds, s>>>(g, d, d0, end_depth, r, out, split, work_counter, schedule, dn.words);
}

uint32_t direct_wave_lds(uint32_t max_qn) { return wave_lds_bytes(2, std::max<uint32_t>(max_qn, 3)); }

void direct_search(const DevGraph& g, const DirectJob* jobs, uint32_t njobs, DirectCtr* ctr, const uint32_t* pairs, uint32_t cap,
                   const DirectQueue& q, uint32_t max_rounds, unsigned long long max_work, hipStream_t s) {
    const size_t lds = static_cast<size_t>(kWaves) * q.wave_lds;
    if (q.pass == 0) {  // about the waves that are resident at once over all steps, at least eight blocks a step
        const uint32_t blocks = std::max<uint32_t>(8, std::min<uint32_t>(128, 2048 / njobs));
        k_direct_search<true><<<dim3(blocks, njobs), kWaves * 64, lds, s>>>(g, jobs, ctr, pairs, cap, q, max_rounds, max_work);
    } else {
        k_direct_search<false><<<kDirectGrid, kWaves * 64, lds, s>>>(g, jobs, ctr, pairs, cap, q, max_rounds, max_work);
    }
}

void direct_commit(const DirectJob* jobs, const DirectCtr* ctr, uint32_t njobs, const DirectQueue& q, uint32_t committed,
                   unsigned long long* results, uint32_t* state, hipStream_t s) {
    k_direct_commit<<<(std::max(njobs, kDirectShards) + 255) / 256, 256, 0, s>>>(jobs, ctr, njobs, q, committed, results, state);
}

void level_prepare(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, uint32_t n, const LevelScratch& ls,
                   bool with_hash, uint32_t* zero, unsigned long long* bytes, hipStream_t s) {
    unsigned long long* ph = with_hash ? ls.ph : nullptr;
    if (n < kSmallLevel) {
        k_level_len_small<<<1, kSmallThreads, 0, s>>>(g, d, d0, rec, n, ls.off, ls.prun, ls.runs, ls.piv, ph, zero, bytes);
        return;
    }
    const uint32_t tiles = (n + kLenTile - 1) / kLenTile;
    k_level_len<<<tiles, kLenThreads, 0, s>>>(g, d, d0, rec, n, ls.off, ls.prun, ls.runs, ls.piv, ph, ls.tile_sum, zero, bytes);
    k_level_scan<<<tiles, kLenThreads, 0, s>>>(ls.off, n, ls.tile_sum);
}

void level_flat(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, uint32_t n, int mode, const LevelScratch& ls,
                Ring r, MatchOut out, hipStream_t s) {
    // Waves take equal contiguous shares of the level's candidates (their total is known on the
    // device only): the grid follows the record count, so small levels do not dispatch thousands
    // of idle waves.
    const int grid = static_cast<int>(std::min<uint32_t>(2048, std::max<uint32_t>(16, n / 2)));
    if (mode == kCountAtEnd)
        k_level_flat<kCountAtEnd><<<grid, 256, 0, s>>>(g, d, d0, rec, n, ls.off, ls.prun, ls.runs, ls.piv, ls.ph, r, out);
    else
        k_level_flat<kWriteAtEnd><<<grid, 256, 0, s>>>(g, d, d0, rec, n, ls.off, ls.prun, ls.runs, ls.piv, ls.ph, r, out);
}

void level_prepare_chain(const DevGraph& g, const StepDesc& d, const LevelChain& c, uint32_t k, const LevelScratch& ls, bool with_hash,
                         unsigned long long* bytes, hipStream_t s) {
    k_level_len_chain<<<kChainLenGrid, kLenThreads, 0, s>>>(g, d, c, k, ls.off, ls.prun, ls.runs, ls.piv, with_hash ? ls.ph : nullptr,
                                                           ls.tile_sum, bytes);
    k_level_scan_chain<<<kChainLenGrid, kLenThreads, 0, s>>>(c, k, ls.off, ls.tile_sum);
}

void level_flat_chain(const DevGraph& g, const StepDesc& d, const LevelChain& c, uint32_t k, int mode, const LevelScratch& ls,
                      MatchOut out, hipStream_t s) {
    // Level sizes are device-side, so the grid is fixed: four four-wave blocks per CU, short of a
    // full residency (six per CU at four candidates per lane) so the other lanes' kernels keep
    // finding room (measured on a 400K-vertex Chung-Lu graph with 65,536-edge batches: 1024 blocks
    // beat 768 and 1536 at four candidates per lane, as 512-768 beat 256, 1024 and 2048 at eight)
    if (mode == kCountAtEnd)
        k_level_flat_chain<kCountAtEnd><<<kChainFlatGrid, 256, 0, s>>>(g, d, c, k, ls.off, ls.prun, ls.runs, ls.piv, ls.ph, out);
    else
        k_level_flat_chain<kWriteAtEnd><<<kChainFlatGrid, 256, 0, s>>>(g, d, c, k, ls.off, ls.prun, ls.runs, ls.piv, ls.ph, out);
}

void level_prepare_chain_multi(const DevGraph& g, const ChainJob* jobs, uint32_t njobs, uint32_t k, int blocks, hipStream_t s) {
    if (!njobs) return;
    const dim3 grid(static_cast<uint32_t>(std::max(16, blocks / 2)), njobs);
    k_level_len_chain_multi<<<grid, kLenThreads, 0, s>>>(g, jobs, k);
    k_level_scan_chain_multi<<<grid, kLenThreads, 0, s>>>(jobs, k);
}

void level_flat_chain_multi(const DevGraph& g, const ChainJob* jobs, uint32_t njobs, uint32_t k, int mode, int blocks, hipStream_t s) {
    if (!njobs) return;
    const dim3 grid(static_cast<uint32_t>(std::max(16, blocks)), njobs);
    if (mode == kCountAtEnd) k_level_flat_chain_multi<kCountAtEnd><<<grid, 256, 0, s>>>(g, jobs, k);
    else k_level_flat_chain_multi<kWriteAtEnd><<<grid, 256, 0, s>>>(g, jobs, k);
}

uint32_t level_max_records(const StepDesc& d, uint32_t d0, const LevelScratch& ls) {
    const uint32_t ne = d.boff[d0 + 1] - d.boff[d0];
    return static_cast<uint32_t>(std::min<uint64_t>(ls.cap, ne > 1 ? ls.runs_cap / ne : ls.cap));
}

void root_chunks(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, const uint32_t* n_rec, uint32_t max_rec,
                 uint32_t max_chunks, unsigned long long* chunks, unsigned long long* scan_tmp, hipStream_t s) {
    k_root_chunks<<<grid_for(max_rec, 256, 4096), 256, 0, s>>>(g, d, d0, rec, n_rec, max_rec, max_chunks, chunks);
    scan_exclusive<unsigned long long>(chunks, chunks, n_rec, max_rec, true, scan_tmp, s);
}

void cp_prepare(const DevGraph& g, const StepDesc& d, uint32_t d0, const uint32_t* rec, uint32_t n, CpScratch c, hipStream_t s) {
    const uint32_t nseg = n * (d.n - d0);
    k_cp_len<<<grid_for(nseg, 256, 4096), 256, 0, s>>>(g, d, d0, rec, n, c);
    scan_exclusive<unsigned long long>(c.seg_off, c.seg_off, nullptr, nseg, true, c.scan_tmp, s);
    k_cp_filter<<<static_cast<int>(std::min<uint32_t>(2048, std::max<uint32_t>(16, nseg / 2))), 256, 0, s>>>(g, d, d0, rec, nseg, c);
    k_cp_products<<<grid_for(n, 256, 4096), 256, 0, s>>>(d, d0, n, c);
    scan_exclusive<unsigned long long>(c.prod, c.prod, nullptr, n, true, c.scan_tmp, s);
}

void cp_enumerate(const StepDesc& d, uint32_t d0, uint32_t n, CpScratch c, MatchOut out, hipStream_t s) {
    k_cp_enumerate<<<static_cast<int>(std::min<uint32_t>(4096, std::max<uint32_t>(64, n))), 256, 0, s>>>(d, d0, n, c, out);
}

}  // namespace csm
