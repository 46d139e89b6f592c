// Filter form of the plain scan, for selective queries of one weight: most
// objects that such a query touches occur in one of its lists only, and the
// top k is made of those that occur in several.
//
// k_scan_hash inserts every posting into an LDS hash table (a compare-and-swap
// and its probes each, eight tiles and eight radix selects a query on LSH
// batches) to find that out.  Here a tile's ids first go through a bit per
// hashed id: an id that meets its bit set is entered in a small table and
// counted; a second pass over the same ids (kept in registers) counts those that
// met it clear, where they are in the table, so that every object of two or more
// postings has its exact count.
// Tiles hold four times the postings.  A tile whose table fills up (many of its
// objects have several postings, as where buckets go together), or with far
// more postings than its share, is counted by k_filter_fill, a quarter at a
// time with every id in the table.  Queries left
// with fewer than k such objects take the smallest ids among the objects of one
// posting (k_filter_fill).
#pragma once
#include "kernels_hash.h"
#include "kernels_runs.h"

namespace gh {

constexpr int kFiltThreads = 1024;
constexpr int kFiltWaves = kFiltThreads / kWave;
constexpr uint32_t kFiltBitsLog = 18;          // 32 KiB of bits: 1 in 16 set when a full tile is done
constexpr uint32_t kFiltLogSlots = 13;         // table slots, 32 KiB
constexpr uint32_t kFiltTarget = 16384;        // postings per (query, tile) aimed at
constexpr uint32_t kFiltMost = kFiltTarget + kFiltTarget / 8;  // bits set: a tile of more is counted in parts
constexpr uint32_t kFiltParts = 4;             // parts of a tile whose table fills up
constexpr uint32_t kFiltProbes = 256;          // taken slots in a row after which the table counts as full,
constexpr uint32_t kFiltPartProbes = 1024;     // ... and a part's (97% of the slots)
constexpr uint32_t kFiltMaxK = 1024;
// Fewer filter tiles than this run on the hash kernel where chunks are compiled
// for other queries anyway: the filter's three kernels take about 35 us however
// few the tiles, and save 0.05 us a tile (25 us for 512 tiles at a time; the hash
// kernel 20 us for 768 of a quarter).  78 queries of two tiles, 22 of them the
// filter's: 119 us on the hash kernel, 148 with the filter.
constexpr uint32_t kFiltFew = 640;
constexpr uint32_t kFiltUnit = 4 * kWave;      // ids a wave loads at a time, 16 bytes a lane
constexpr int kFiltUnits = 5;                  // units a wave keeps in registers
constexpr uint32_t kFiltSeen = 8;              // units of a wave whose hits pass 1 counts, a bit an id
constexpr uint32_t kFiltLater = 1u << 31;      // an entered id that pass 2 counts (ids are below 2^30)
constexpr uint32_t kFiltList = 2048;           // ids on their way into (or counted in) the table, a part a wave
constexpr uint32_t kFiltFillMost = (1u << kHashLogMax) / 4 * 3;  // postings k_filter_fill enters in its table

struct FilterArgs {
    ScanArgs s;
    const uint32_t* work;       // [n_work][2]: query, tile
    const uint4* hq;            // [n_queries]: directory tiles per tile, key bits, weight, tiles (0: other kernels)
    const uint32_t* fq;         // [n_fq] the queries (fill)
    const genie_dim_t* items;   // one key each
    uint32_t n_items;
    const uint32_t* item_qptr;
    uint2* spans;               // [tiles][n_items] every item's postings that can hold ids of the tile
    uint32_t* over_n;           // [n_queries] tiles to count in parts
    uint32_t* over;             // [n_queries][max_tiles] these tiles
    uint32_t max_tiles;
    uint32_t* hov;
    uint32_t* hov_any;
    unsigned long long* gkey;
};

// Every item's span in every tile of its query, resolved once: the key and
// directory reads are scattered, and a workgroup per (query, tile) whose waves
// each made them spent most of its time there (4M x 64 LSH: 0.53 of 0.82 ms).
__global__ void __launch_bounds__(256) k_filter_spans(FilterArgs fa, KeyPos kp)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= fa.n_items)
        return;
    const genie_dim_t it = fa.items[i];
    const uint4 prm = fa.hq[it.query];
    if (prm.w == 0)
        return;
    const ScanArgs& a = fa.s;
    fa.over_n[it.query] = 0;
    const bool empty = it.end_pos <= it.start_pos || it.weight == 0.0f;
    const uint32_t sp = empty ? 0u : (uint32_t)it.start_pos, ep = empty ? 0u : (uint32_t)it.end_pos;
    uint32_t ks = 0, doff = kNoDir;
    if (!empty && prm.w > 1) {
        const uint32_t k = key_at(kp, sp);
        ks = kp.key_start[k];
        doff = a.dir_off[k];
    }
    for (uint32_t t = 0; t < prm.w; ++t) {
        uint32_t lo = sp, hi = ep;
        if (doff != kNoDir)
            dir_clip(a.dir, doff, ks, t * prm.x, min(t * prm.x + prm.x, a.n_dtiles), a.n_dtiles, lo, hi);
        fa.spans[(uint64_t)t * fa.n_items + i] = make_uint2(lo, max(lo, hi));
    }
}

// f(lo, hi) for the query's items, 64 at a time, one a lane: the spans of tile
// t, or (whole) the items' own.  Called by whole waves.
template <class F>
__device__ __forceinline__ void filter_spans(const FilterArgs& fa, uint32_t q, uint32_t t, bool whole, F f)
{
    const uint32_t i0 = fa.item_qptr[q], i1 = fa.item_qptr[q + 1], lane = lane_id();
    for (uint32_t ib = i0; ib < i1; ib += kWave) {
        uint2 sp = make_uint2(0, 0);
        if (ib + lane < i1) {
            if (whole) {
                const genie_dim_t it = fa.items[ib + lane];
                if (it.end_pos > it.start_pos && it.weight != 0.0f)
                    sp = make_uint2((uint32_t)it.start_pos, (uint32_t)it.end_pos);
            } else {
                sp = fa.spans[(uint64_t)t * fa.n_items + ib + lane];
            }
        }
        f(sp.x, sp.y);
    }
}

// Bit of an id: a full-rate 24-bit product (bits of an id above 24 do not
// enter; ids that share a bit only pass the filter together).
__device__ __forceinline__ uint32_t filter_bit(uint32_t loc)
{
    return ((loc & 0xFFFFFFu) * 0x9E3779u) >> (32u - kFiltBitsLog);
}

// One workgroup per (query, tile).  Ids are kept tile-local; lanes past a
// span's end, and ids of other tiles, hold 0xFFFFFFFF.
// 4M x 64 LSH (8,192 buckets), 4,096 queries: k_scan_hash 1.20 ms; here the
// spans 21 us, this kernel 475 us (488 when pass 1 entered without counting and
// pass 2 counted every posting) and the fill 25 us.  Where four fifths of a
// 1,000-object cluster share a bucket (1M x 64 in 4,096 buckets), 1,024
// queries: k_scan_hash 306 us, here 317; a tenth of 3,000: 1,270 and 165.
__global__ void __launch_bounds__(kFiltThreads, 8) k_scan_filter(FilterArgs fa)
{
    __shared__ uint32_t s_bits[1u << (kFiltBitsLog - 5)];
    __shared__ uint32_t s_tab[1u << kFiltLogSlots];
    __shared__ uint32_t s_red[3 * kMaxWaves];
    __shared__ uint32_t s_res[8];
    __shared__ uint32_t s_list[kFiltList];
    __shared__ uint32_t s_set;    // bits set
    __shared__ uint32_t s_n;      // some id is listed
    const ScanArgs& a = fa.s;
    const uint32_t q = fa.work[2 * blockIdx.x], t = fa.work[2 * blockIdx.x + 1];
    const uint4 prm = fa.hq[q];
    const uint32_t kb = prm.y, w = prm.z;
    const uint32_t obj0 = t * prm.x * kDirTile;
    const uint32_t nobj = min(prm.x * kDirTile, a.n_objects - obj0);
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (uint32_t i = tid; i < 1u << (kFiltBitsLog - 7); i += kFiltThreads)
        reinterpret_cast<uint4*>(s_bits)[i] = make_uint4(0, 0, 0, 0);
    for (uint32_t i = tid; i < 1u << (kFiltLogSlots - 2); i += kFiltThreads)
        reinterpret_cast<uint4*>(s_tab)[i] = make_uint4(0, 0, 0, 0);
    if (tid == 0) {
        s_res[7] = 0;
        s_set = 0;
        s_n = 0;
    }
    __syncthreads();

    // every 16th unit of the spans (uint4 of the lanes from an aligned
    // position), the first kFiltUnits of the wave in registers; take(v) on
    // the units past them, in each pass
    auto units = [&](auto&& keep, auto&& take) {
        uint32_t turn = wv, mine = 0;
        filter_spans(fa, q, t, false, [&](uint32_t lo, uint32_t hi) {
            const uint32_t len = hi - lo;
            const uint32_t nu = len ? ((lo & 3u) + len + (kFiltUnit - 1)) / kFiltUnit : 0u;
            const uint32_t incl = wave_incl_scan(nu);
            const uint32_t total = __builtin_amdgcn_readlane(incl, kWave - 1);
            for (uint32_t u = turn; u < total; u += kFiltWaves, ++mine) {
                const int r = __popcll(ballot(incl <= u));
                const uint32_t s = __builtin_amdgcn_readlane(lo, r), n = __builtin_amdgcn_readlane(len, r);
                const uint32_t p = (s & ~3u) + (u - __builtin_amdgcn_readlane(incl - nu, r)) * kFiltUnit + 4u * lane;
                auto load = [&]() {
                    uint4 v = make_uint4(0, 0, 0, 0);
                    if (p + 4u > s && p < s + n)  // (the postings are padded to whole loads)
                        v = *reinterpret_cast<const uint4*>(a.post + p);
                    // tile-local ids; those of other tiles and other spans are ~0
                    const uint32_t d = p - s;
                    v.x = d < n && v.x - obj0 < nobj ? v.x - obj0 : ~0u;
                    v.y = d + 1u < n && v.y - obj0 < nobj ? v.y - obj0 : ~0u;
                    v.z = d + 2u < n && v.z - obj0 < nobj ? v.z - obj0 : ~0u;
                    v.w = d + 3u < n && v.w - obj0 < nobj ? v.w - obj0 : ~0u;
                    return v;
                };
                if (mine < (uint32_t)kFiltUnits)
                    keep(mine, load);
                else
                    take(load(), mine);
            }
            turn = (turn + kFiltWaves - total % kFiltWaves) % kFiltWaves;
        });
    };
    uint32_t bits = 0, seen = 0, listed = 0;
    auto enter = [&](uint32_t id) {
        if (!hash_add(s_tab, kFiltLogSlots, kb, id & ~kFiltLater, id & kFiltLater ? 0u : w, kFiltProbes))
            s_res[7] = 1;
    };
    // past the list: none is tried once one has failed (each goes past kFiltProbes slots)
    auto enter_now = [&](uint32_t id) {
        if (!*(volatile uint32_t*)&s_res[7])
            enter(id);
    };
    // the few ids that hit go on the wave's part of the list, which all lanes
    // work off together afterwards (a hash insert by the odd lane of nearly
    // every wave took most of the kernel's instructions); `now` when it is full
    auto list_hit = [&](bool hit, uint32_t id, auto&& now) {
        const uint64_t b = ballot(hit);
        if (!b)
            return;
        const uint32_t at = listed + lane_prefix(b);
        listed += (uint32_t)__popcll(b);
        if (hit) {
            if (at < kFiltList / kFiltWaves)
                s_list[wv * (kFiltList / kFiltWaves) + at] = id;
            else
                now(id);
        }
    };
    auto pass1 = [&](const uint4& v, uint32_t m) {  // the wave's unit m
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
        uint32_t old[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t h = filter_bit(x[j]);
            old[j] = 0;
            if (x[j] != ~0u)  // (lanes without an id would meet in one word)
                old[j] = atomicOr(&s_bits[h >> 5], 1u << (h & 31u)) >> (h & 31u) & 1u;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            bits += (uint32_t)__popcll(ballot(x[j] != ~0u && !old[j]));
            if (m < kFiltSeen)  // uniform
                seen |= old[j] << (4u * m + j);
            list_hit(old[j] != 0, m < kFiltSeen ? x[j] : x[j] | kFiltLater, enter_now);
        }
    };
    // counts a posting of an id that is in the table (another id of its bit is not)
    auto count = [&](uint32_t id) {
        const uint32_t key = (id + 1u) << (32u - kb), kmask = ~0u << (32u - kb);
        uint32_t s = (id * 0x9E3779B1u) >> (32u - kFiltLogSlots);
        for (uint32_t probe = 0; probe < 1u << kFiltLogSlots; ++probe) {
            const uint32_t y = s_tab[s];
            if (y == 0)
                break;
            if ((y & kmask) == key) {
                atomicAdd(&s_tab[s], w);
                break;
            }
            s = (s + 1u) & ((1u << kFiltLogSlots) - 1u);
        }
    };
    auto pass2 = [&](const uint4& v, uint32_t m) {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
        uint32_t in[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t h = filter_bit(x[j]);
            in[j] = s_bits[h >> 5] >> (h & 31u) & 1u;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            list_hit(in[j] != 0 && x[j] != ~0u && (m >= kFiltSeen || !((seen >> (4u * m + j)) & 1u)), x[j], count);
    };
    // f on the listed ids, every lane of the wave one
    auto list_all = [&](auto&& f) {
        for (uint32_t i = lane; i < min(listed, kFiltList / kFiltWaves); i += kWave)
            f(s_list[wv * (kFiltList / kFiltWaves) + i]);
    };
    uint4 kept[kFiltUnits];
#pragma unroll
    for (int i = 0; i < kFiltUnits; ++i)
        kept[i] = make_uint4(~0u, ~0u, ~0u, ~0u);
    units([&](uint32_t m, auto&& load) {
        const uint4 v = load();
#pragma unroll
        for (int i = 0; i < kFiltUnits; ++i)
            if (m == (uint32_t)i)  // uniform
                kept[i] = v;
    }, pass1);
#pragma unroll
    for (int i = 0; i < kFiltUnits; ++i)
        pass1(kept[i], (uint32_t)i);
    list_all(enter);
    if (lane == 0) {
        atomicAdd(&s_set, bits);
        if (listed)
            s_n = 1;
    }
    __syncthreads();
    if (s_res[7] || s_set > kFiltMost) {
        if (tid == 0)
            fa.over[(uint64_t)q * fa.max_tiles + atomicAdd(&fa.over_n[q], 1u)] = t;
        return;
    }
    if (s_n == 0)
        return;  // no object of two postings
    // the bits of the table's ids in place of those of every id
    for (uint32_t i = tid; i < 1u << (kFiltBitsLog - 7); i += kFiltThreads)
        reinterpret_cast<uint4*>(s_bits)[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < (1u << kFiltLogSlots) / kFiltThreads; ++i) {
        const uint32_t y = s_tab[tid + i * kFiltThreads];
        if (y) {
            const uint32_t h = filter_bit((y >> (32u - kb)) - 1u);
            atomicOr(&s_bits[h >> 5], 1u << (h & 31u));
        }
    }
    listed = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFiltUnits; ++i)
        pass2(kept[i], (uint32_t)i);
    units([](uint32_t, auto&&) {}, pass2);
    list_all(count);
    __syncthreads();
    hash_select(a, fa.gkey, s_tab, 1u << kFiltLogSlots, kb, q, obj0, s_res, s_red, a.kq[q], 2u * w, 0xFFFFFFFFu, true);
}

// Marks an id in the fill's table: a word of key << (32 - kb) | 1 after one
// posting, | 3 after more.  The table is at most three quarters full.
__device__ __forceinline__ void fill_add(uint32_t* tab, uint32_t kb, uint32_t id)
{
    const uint32_t key = (id + 1u) << (32u - kb), kmask = ~0u << (32u - kb);
    uint32_t h = (id * 0x9E3779B1u) >> (32u - kHashLogMax);
    for (uint32_t probe = 0; probe < 1u << kHashLogMax; ++probe) {
        const uint32_t v = atomicCAS(&tab[h], 0u, key | 1u);
        if (v == 0)
            return;
        if ((v & kmask) == key) {
            atomicOr(&tab[h], 2u);
            return;
        }
        h = (h + 1u) & ((1u << kHashLogMax) - 1u);
    }
}

// First the query's tiles left to be counted in parts: the objects of several
// postings of a quarter at a time, every posting counted in the table.
// Queries that the filter left with fewer than k candidates: the smallest ids
// among the objects of one posting.  Lists ascend, so these lie in the first
// postings of every list: all ids below a bound are counted in a table, the
// bound first set for the number needed and doubled until enough objects of
// one posting are below it, or halved back when more than the table takes are.
__global__ void __launch_bounds__(kFiltThreads, 8) k_filter_fill(FilterArgs fa)
{
    __shared__ uint32_t s_tab[1u << kHashLogMax];
    __shared__ uint32_t s_red[3 * kMaxWaves];
    __shared__ uint32_t s_res[8];
    __shared__ uint32_t s_posts, s_in, s_ones;
    const ScanArgs& a = fa.s;
    const uint32_t q = fa.fq[blockIdx.x];
    const uint32_t k = a.kq[q], n_over = fa.over_n[q];
    uint32_t have = a.cand_cnt[q];
    if (have >= k && n_over == 0)
        return;
    const uint32_t w = fa.hq[q].z;
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll 1
    for (uint32_t i = 0; i < n_over * kFiltParts; ++i) {
        const uint32_t t = fa.over[(uint64_t)q * fa.max_tiles + i / kFiltParts];
        const uint32_t part = fa.hq[q].x * (kDirTile / kFiltParts), tile0 = t * fa.hq[q].x * kDirTile;
        const uint32_t o0 = tile0 + i % kFiltParts * part;  // ids [o0, o0 + part), keys from the part's start
        if (o0 >= a.n_objects)
            continue;
        for (uint32_t j = tid; j < 1u << kHashLogMax; j += kFiltThreads)
            s_tab[j] = 0;
        if (tid == 0)
            s_res[7] = 0;
        __syncthreads();
        filter_spans(fa, q, t, false, [&](uint32_t lo, uint32_t hi) {
            const uint64_t some = ballot(hi > lo);
            for (uint32_t r = wv; r < (uint32_t)kWave; r += kFiltWaves) {
                if (!((some >> r) & 1u))
                    continue;
                const uint32_t s = __builtin_amdgcn_readlane(lo, r), e = __builtin_amdgcn_readlane(hi, r);
                for (uint32_t p = s + lane; p < e; p += kWave) {
                    const uint32_t loc = a.post[p] - o0;
                    if (loc < part && !*(volatile uint32_t*)&s_res[7] &&
                        !hash_add(s_tab, kHashLogMax, fa.hq[q].y, loc, w, kFiltPartProbes))
                        s_res[7] = 1;
                }
            }
        });
        __syncthreads();
        if (s_res[7]) {
            if (tid == 0) {
                fa.hov[q] = 1u;  // the direct kernels
                *fa.hov_any = 1u;
            }
            return;
        }
        hash_select(a, fa.gkey, s_tab, 1u << kHashLogMax, fa.hq[q].y, q, o0, s_res, s_red, k, 2u * w, 0xFFFFFFFFu, true);
        __syncthreads();
    }
    if (n_over) {  // the loop added to it
        if (tid == 0)
            s_in = __hip_atomic_load(&a.cand_cnt[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        have = s_in;
    }
    if (have >= k)
        return;
    const uint32_t need = k - have;
    if (tid == 0)
        s_posts = 0;
    __syncthreads();
    if (wv == 0) {
        uint32_t n = 0;
        filter_spans(fa, q, 0, true, [&](uint32_t lo, uint32_t hi) { n += hi - lo; });
        n = wave_sum(n);
        if (lane == 0)
            s_posts = n;
    }
    __syncthreads();
    const uint32_t posts = s_posts;
    if (posts == 0)
        return;
    // ids that should lie below the bound: those needed, the objects of more
    // postings, and a margin.  Ids crowd in places, so a bound with too many
    // below it is halved towards the largest that had too few.
    uint64_t x = (uint64_t)a.n_objects * (need + need / 4 + 64u) / posts + 1;
    uint32_t few = 0, many = 0;  // bounds with too few and (once met) too many ids below
    for (;;) {
        const uint32_t bound = (uint32_t)min<uint64_t>(x, a.n_objects);
        const uint32_t kb = 32u - (uint32_t)__builtin_clz(bound);  // keys are 1..bound (below 2^30)
        // f(id) for the ids below the bound, a wave a span, every 16th of 64
        auto below = [&](auto&& f) {
            filter_spans(fa, q, 0, true, [&](uint32_t lo, uint32_t hi) {
                const uint64_t some = ballot(hi > lo);
                for (uint32_t r = wv; r < (uint32_t)kWave; r += kFiltWaves) {
                    if (!((some >> r) & 1u))
                        continue;
                    const uint32_t s = __builtin_amdgcn_readlane(lo, r), e = __builtin_amdgcn_readlane(hi, r);
                    for (uint32_t p = s; p < e; p += kWave) {
                        const uint32_t id = p + lane < e ? a.post[p + lane] : ~0u;
                        if (id < bound)
                            f(id);
                        if (ballot(id < bound) != ~0ull)
                            break;  // the list ascends: the rest is past the bound
                    }
                }
            });
        };
        for (uint32_t i = tid; i < 1u << kHashLogMax; i += kFiltThreads)
            s_tab[i] = 0;
        if (tid == 0) {
            s_in = 0;
            s_ones = 0;
        }
        __syncthreads();
        uint32_t in = 0;
        below([&](uint32_t) { ++in; });
        in = wave_sum(in);
        if (lane == 0)
            atomicAdd(&s_in, in);
        __syncthreads();
        const bool crowded = s_in > kFiltFillMost;
        if (!crowded)
            below([&](uint32_t id) { fill_add(s_tab, kb, id); });
        __syncthreads();
        uint32_t ones = 0;
#pragma unroll
        for (uint32_t i = 0; i < (1u << kHashLogMax) / kFiltThreads; ++i) {
            const uint32_t y = s_tab[tid + i * kFiltThreads];
            ones += y != 0 && (y & ((1u << (32u - kb)) - 1u)) == 1u;
        }
        ones = wave_sum(ones);
        if (lane == 0)
            atomicAdd(&s_ones, ones);
        __syncthreads();
        if (!crowded && (s_ones >= need || bound == a.n_objects)) {
            hash_select(a, fa.gkey, s_tab, 1u << kHashLogMax, kb, q, 0, s_res, s_red, need, 1u, 1u, false, w);
            return;
        }
        (crowded ? many : few) = bound;
        if (many != 0 && many - few <= 1u) {
            if (tid == 0) {
                fa.hov[q] = 1u;  // more at one id than the table takes: the direct kernels
                *fa.hov_any = 1u;
            }
            return;
        }
        x = many ? few + (many - few) / 2 : 2 * x;
        __syncthreads();
    }
}

}  // namespace gh
