// Direct-mapped scan over tile-major postings ("runs"): a second copy of the
// posting lists with the ids of one 65,536-object tile together, key after
// key, as 16-bit ids within the tile.  An item's postings in a tile are then
// one contiguous run, however many keys its range covers.
//
// The per-key lists (k_scan_tile) give a range over many values one span per
// (key, tile): 81 spans of about 50 ids for each item of a 400,000 x 48 table
// with 2,048 values a dim, each a wave's visit with its own latency.
#pragma once
#include "kernels.h"

namespace gh {

constexpr uint32_t kRunTileLog = 16;
constexpr uint32_t kRunTile = 1u << kRunTileLog;  // ids are 16 bits
constexpr int kRunThreads = 1024;
constexpr int kRunWaves = kRunThreads / kWave;
constexpr uint32_t kRunUnit = 8 * kWave;          // ids a wave takes at a time, 16 bytes a lane
constexpr uint32_t kRunPad = kRunUnit;            // ids past the last run that a unit may read
// The copy is built for indexes whose lists hold at least this many ids per
// full tile on average: its directory (8 B per key and tile) is then at most
// a sixth of the postings' bytes.  Shorter lists (LSH buckets) are searched by
// the hash form.
constexpr uint32_t kRunMinPerTile = 12;

// tf[t * K + k]: x = first id of key k in tile t in the tile-major copy, y =
// position in the posting lists of the key's first id at or past the tile.
// Entry n_tiles * K ends the copy.
struct RunIndex {
    const uint16_t* ids;
    const uint2* tf;
    uint32_t n_keys, n_tiles;
};

// ---- index creation --------------------------------------------------------

// One thread per (tile of 2^log objects, key): the position of the key's first
// id at or past the tile, and (cnt) the ids the key holds in the tile.  `keys`:
// the keys of the copy (null: all n_keys of the index).
__global__ void __launch_bounds__(256) k_run_first(const uint32_t* __restrict__ post,
                                                   const uint32_t* __restrict__ key_start,
                                                   const uint32_t* __restrict__ keys, uint32_t n_keys,
                                                   uint32_t n_tiles, uint32_t log, uint2* __restrict__ tf,
                                                   uint32_t* __restrict__ cnt)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n_keys * n_tiles)
        return;
    const uint32_t t = i / n_keys, k = keys ? keys[i % n_keys] : i % n_keys;
    const uint32_t s = key_start[k], e = key_start[k + 1];
    auto first_at = [&](uint64_t target) {
        uint32_t lo = s, hi = e;
        while (lo < hi) {
            const uint32_t mid = lo + ((hi - lo) >> 1);
            if ((uint64_t)post[mid] < target)
                lo = mid + 1;
            else
                hi = mid;
        }
        return lo;
    };
    const uint32_t a = first_at((uint64_t)t << log), b = first_at((uint64_t)(t + 1) << log);
    tf[i].y = a;
    cnt[i] = b - a;
}

// The prefix of the counts into tf[].x (and the end entry).
__global__ void __launch_bounds__(256) k_run_start(const uint32_t* __restrict__ prefix, uint32_t n, uint32_t total,
                                                   uint2* __restrict__ tf)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n)
        tf[i].x = prefix[i];
    else if (i == n)
        tf[i] = make_uint2(total, total);
}

// A workgroup per key, or every gridDim.x-th: its ids within the tiles (log <= 16) to their runs.
__global__ void __launch_bounds__(256) k_run_fill(const uint32_t* __restrict__ post,
                                                  const uint32_t* __restrict__ key_start,
                                                  const uint32_t* __restrict__ keys, uint32_t n_keys, uint32_t log,
                                                  const uint2* __restrict__ tf, uint16_t* __restrict__ ids)
{
    for (uint32_t r = blockIdx.x; r < n_keys; r += gridDim.x) {
        const uint32_t k = keys ? keys[r] : r;
        for (uint32_t p = key_start[k] + threadIdx.x; p < key_start[k + 1]; p += blockDim.x) {
            const uint32_t o = post[p];
            const uint2 f = tf[(uint64_t)(o >> log) * n_keys + r];
            ids[f.x + (p - f.y)] = (uint16_t)(o & ((1u << log) - 1u));
        }
    }
}

// ---- per run ---------------------------------------------------------------

// The key of a posting position: the buckets of the index's PosIndex leave a
// search of a few keys (a binary search of all 524,288 keys of an LSH index
// takes 19 dependent loads).
struct KeyPos {
    const uint32_t* first;
    uint32_t n, shift;
    const uint32_t* key_start;
};

__device__ __forceinline__ uint32_t key_at(const KeyPos& kp, uint32_t pos)
{
    const uint32_t b = min(pos >> kp.shift, kp.n - 1u);
    uint32_t lo = kp.first[b], hi = kp.first[b + 1];
    while (lo < hi) {  // first key that starts past pos
        const uint32_t mid = (lo + hi) >> 1;
        if (kp.key_start[mid] <= pos)
            lo = mid + 1;
        else
            hi = mid;
    }
    return lo - 1u;
}

// First and last key of every item (items without postings get none).
__global__ void __launch_bounds__(256) k_item_keys(const genie_dim_t* __restrict__ items, uint32_t n_items, KeyPos kp,
                                                   uint32_t* __restrict__ k0, uint32_t* __restrict__ k1)
{
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n_items)
        return;
    const genie_dim_t it = items[i];
    if (it.end_pos <= it.start_pos)
        return;
    k0[i] = key_at(kp, (uint32_t)it.start_pos);
    k1[i] = key_at(kp, (uint32_t)it.end_pos - 1);
}

struct RunArgs {
    ScanArgs s;
    RunIndex r;
    const genie_dim_t* items;   // sorted by query, posting positions
    const uint32_t* item_qptr;
    const uint32_t *k0, *k1;    // first and last key of every item
    uint32_t first;             // (tile, query) of the launch's first workgroup
};

// A unit of a run: 512 ids from an 8-id boundary, 8 a lane.
struct RunUnit {
    uint4 v;
    uint32_t pos;    // the lane's first id in the copy
    uint32_t s, len; // its run
    uint32_t w;
};

// Adds w to the counters of eight 16-bit ids.  MASK: only those whose position
// lies in the run [s, s + len); the others, ids of another run, add zero.
template <int LB, bool MASK>
__device__ __forceinline__ void run_count8(const RunUnit& u, uint32_t* cnt)
{
    const uint32_t x[4] = {u.v.x, u.v.y, u.v.z, u.v.w};
    char* base = reinterpret_cast<char*>(cnt);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t id = j & 1 ? x[j >> 1] >> 16 : x[j >> 1] & 0xFFFFu;
        const uint32_t w = !MASK || u.pos + j - u.s < u.len ? u.w : 0u;
        if constexpr (LB == 8)
            atomicAdd(reinterpret_cast<uint32_t*>(base + (id & 0xFFFCu)), w << ((id & 3u) * 8u));
        else
            atomicAdd(reinterpret_cast<uint32_t*>(base + (id & 0xFFFEu) * 2u), w << ((id & 1u) * 16u));
    }
}

// Exact tile top-k of the packed counters under (count desc, id asc), pruned
// by the query's adaptive threshold: the keys that tile_select emits, in three
// passes over the counters (largest and eligible counts; histogram; emission).
// A tile where fewer than k objects reach the threshold needs no histogram.
// The histogram's bins are four copies a bin, a lane's copy by its number, so
// that the few bins most objects share take a quarter of the conflicts.
constexpr uint32_t kRunBins = 256;
struct RunSel {
    uint32_t hist[4 * kRunBins];
    uint32_t wv[2 * kRunWaves];
    uint32_t tie[kRunWaves * 8];
    uint32_t res[8];
};

template <int LB>
__device__ __forceinline__ void run_select(const ScanArgs& a, const uint4* cnt4, uint32_t q, uint32_t obj0, RunSel& S)
{
    constexpr int PER = 32 / LB;                                // objects a word
    constexpr int NQ = (int)(kRunTile / PER / 4) / kRunThreads; // quads of words a thread
    constexpr uint32_t kMask = LB == 8 ? 255u : 65535u;
    const int tid = threadIdx.x, lane = lane_id(), wv = tid >> 6;
    const uint32_t k = a.kq[q];
    if (tid == 0)  // one read, shared, so that every thread takes the same branches
        S.res[6] = __hip_atomic_load(&a.gthr[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const uint32_t lower = max(1u, S.res[6]);
    // f(count, object) for every object of this thread, in id order per j
    auto each = [&](int j, auto f) {
        const uint4 v = cnt4[j * kRunThreads + tid];
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
        const uint32_t o0 = (uint32_t)(j * kRunThreads + tid) * (4 * PER);
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int b = 0; b < PER; ++b)
                f((x[c] >> (LB * b)) & kMask, o0 + c * PER + b);
    };
    uint32_t m = 0, e = 0;
#pragma unroll 1
    for (int j = 0; j < NQ; ++j)
        each(j, [&](uint32_t c, uint32_t) {
            m = max(m, c);
            e += c >= lower;
        });
    m = wave_max(m);
    e = wave_sum(e);
    if (lane == 0) {
        S.wv[wv] = m;
        S.wv[kRunWaves + wv] = e;
    }
    __syncthreads();
    uint32_t M = 0, E = 0;
    for (int i = 0; i < kRunWaves; ++i) {
        M = max(M, S.wv[i]);
        E += S.wv[kRunWaves + i];
    }
    if (M < lower)
        return;  // nothing in this tile can reach the query's top k

    // the k-th count, in windows of 256 counts from the top
    uint32_t ct = lower, ngt = E, neq = 0;
    const bool found = E >= k;
    if (found) {
        uint32_t top = M, cum = 0;
        for (;;) {
            const uint32_t wlo = top >= lower + (kRunBins - 1) ? top - (kRunBins - 1) : lower;
            __syncthreads();
            for (uint32_t i = tid; i < 4 * kRunBins; i += kRunThreads)
                S.hist[i] = 0;
            __syncthreads();
#pragma unroll 1
            for (int j = 0; j < NQ; ++j)
                each(j, [&](uint32_t c, uint32_t) {
                    if (c >= wlo && c <= top)
                        atomicAdd(&S.hist[(c - wlo) * 4 + (lane & 3)], 1u);
                });
            __syncthreads();
            if (wv == 0) {
                // lane l holds bins 255 - 4 l .. 252 - 4 l, counted from the top
                const uint32_t b0 = kRunBins - 1 - 4u * (uint32_t)lane;
                uint32_t h[4], sum = 0;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    const uint4 c4 = reinterpret_cast<const uint4*>(S.hist)[b0 - b];
                    h[b] = c4.x + c4.y + c4.z + c4.w;
                    sum += h[b];
                }
                const uint32_t incl = wave_incl_scan(sum);
                uint32_t above = cum + incl - sum;
                const bool here = above < k && above + sum >= k;
                if (here) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        if (above + h[b] >= k) {
                            S.res[1] = wlo + b0 - b;
                            S.res[2] = above;
                            S.res[3] = h[b];
                            break;
                        }
                        above += h[b];
                    }
                }
                const uint64_t any = ballot(here);
                if (lane == kWave - 1) {
                    S.res[0] = any != 0;
                    S.res[7] = cum + incl;
                }
            }
            __syncthreads();
            if (S.res[0]) {
                ct = S.res[1];
                ngt = S.res[2];
                neq = S.res[3];
                break;
            }
            // E >= k: the k-th count lies in a lower window
            cum = S.res[7];
            top = wlo - 1;
        }
    }
    const uint32_t need = found ? k - ngt : 0;
    const bool trim = found && neq > need;
    const uint32_t nemit = ngt + min(neq, need);
    if (tid == 0) {
        uint32_t base = atomicAdd(&a.cand_cnt[q], nemit);
        if ((uint64_t)base + nemit > a.cand_cap[q]) {
            atomicOr(a.overflow, 1u);
            base = kEmitFail;
        }
        if (found)
            atomicMax(&a.gthr[q], ct);
        S.res[4] = base;
        S.res[5] = 0;  // unordered slot counter
    }
    __syncthreads();
    const uint32_t base = S.res[4];
    if (base == kEmitFail)
        return;
    uint64_t* out = a.cand + a.cand_base[q] + base;

    // objects strictly above ct in any order (with those equal to it when
    // none of them is left out); the ties counted on the way
    const uint32_t cut = trim ? ct + 1 : ct;
    constexpr uint32_t kPb = 32 / NQ;  // bits of a packed tie count (at most 4 * PER objects a quad)
    static_assert((4u * PER) >> kPb == 0, "tie counts fit their fields");
    uint32_t ties = 0;
#pragma unroll 1
    for (int j = 0; j < NQ; ++j) {
        uint32_t t = 0;
        each(j, [&](uint32_t c, uint32_t o) {
            t += c == ct;
            if (c >= cut)
                out[atomicAdd(&S.res[5], 1u)] = make_key(c, obj0 + o);
        });
        ties |= t << (kPb * j);
    }
    if (!trim)
        return;
    // the `need` smallest ids tied at ct: rank by (j, thread, object)
    constexpr uint32_t kPm = (1u << kPb) - 1u;
#pragma unroll 1
    for (int j = 0; j < NQ; ++j) {
        const uint32_t sum = wave_sum((ties >> (kPb * j)) & kPm);
        if (lane == 0)
            S.tie[j * kRunWaves + wv] = sum;
    }
    __syncthreads();
    if (wv == 0) {  // exclusive prefix of the NQ x 16 wave totals, two a lane
        const uint32_t i0 = 2u * (uint32_t)lane;
        const uint32_t a0 = i0 < NQ * kRunWaves ? S.tie[i0] : 0u, a1 = i0 + 1 < NQ * kRunWaves ? S.tie[i0 + 1] : 0u;
        const uint32_t ex = wave_incl_scan(a0 + a1) - a0 - a1;
        if (i0 < NQ * kRunWaves) {
            S.tie[i0] = ex;
            S.tie[i0 + 1] = ex + a0;
        }
    }
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < NQ; ++j) {
        const uint32_t w0 = S.tie[j * kRunWaves + wv];  // uniform
        if (w0 >= need)
            break;  // later ranks are larger
        const uint32_t mine = (ties >> (kPb * j)) & kPm;
        uint32_t r = w0 + wave_incl_scan(mine) - mine;
        if (mine && r < need)
            each(j, [&](uint32_t c, uint32_t o) {
                if (c == ct) {
                    if (r < need)
                        out[ngt + r] = make_key(ct, obj0 + o);
                    ++r;
                }
            });
    }
}

// One workgroup per (tile, query), tile-major.  The counters of the tile's
// 65,536 objects fill LDS (64 KiB at 8 bits, two workgroups a CU; 128 KiB at
// 16).  Every wave resolves the query's items itself, 64 at a time, one a lane
// (the directory entries come from L1 after the first wave), and takes every
// 16th unit of their runs, the next unit's ids loaded while it counts one: no
// barrier between items, and no list of spans in LDS.
template <int LB>
__global__ void __launch_bounds__(kRunThreads, 8) k_scan_runs(RunArgs ra)
{
    constexpr uint32_t kWords = kRunTile / (32 / LB);
    __shared__ uint4 s_cnt4[kWords / 4];
    __shared__ RunSel s_sel;
    const ScanArgs& a = ra.s;
    uint32_t* cnt = reinterpret_cast<uint32_t*>(s_cnt4);
    const uint32_t nql = a.qlist ? a.n_qlist : a.n_queries;
    const uint32_t b = ra.first + blockIdx.x, t = b / nql;
    const uint32_t q = a.qlist ? a.qlist[b % nql] : b % nql;
    const int tid = threadIdx.x, lane = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (uint32_t i = tid; i < kWords / 4; i += kRunThreads)
        s_cnt4[i] = make_uint4(0, 0, 0, 0);
    __syncthreads();

    const uint2* tf = ra.r.tf + (uint64_t)t * ra.r.n_keys;
    const uint32_t i0 = ra.item_qptr[q], i1 = ra.item_qptr[q + 1];
    uint32_t turn = wv;  // first unit of the window that this wave takes
    for (uint32_t ib = i0; ib < i1; ib += kWave) {
        // one item a lane: its run in this tile (items may start or end
        // inside a key), and the units before the end of it
        uint32_t start = 0, len = 0, w = 0;
        if (ib + lane < i1) {
            const genie_dim_t it = ra.items[ib + lane];
            w = (uint32_t)it.weight;
            if (it.end_pos > it.start_pos && w) {
                const uint32_t ka = ra.k0[ib + lane], kb = ra.k1[ib + lane];
                const uint2 fa = tf[ka], fb = tf[kb];
                const uint32_t ca = tf[ka + 1].x - fa.x, cb = tf[kb + 1].x - fb.x;
                const uint32_t sp = (uint32_t)it.start_pos, ep = (uint32_t)it.end_pos;
                start = fa.x + (sp > fa.y ? min(sp - fa.y, ca) : 0u);
                len = fb.x + (ep > fb.y ? min(ep - fb.y, cb) : 0u) - start;
            }
        }
        const uint32_t nu = len ? ((start & 7u) + len + (kRunUnit - 1)) / kRunUnit : 0u;
        const uint32_t incl = wave_incl_scan(nu);
        const uint32_t total = __builtin_amdgcn_readlane(incl, kWave - 1);
        auto fetch = [&](uint32_t u) {
            // the item whose units hold u
            const int r = __popcll(ballot(incl <= u));
            RunUnit x;
            x.s = __builtin_amdgcn_readlane(start, r);
            x.len = __builtin_amdgcn_readlane(len, r);
            x.w = __builtin_amdgcn_readlane(w, r);
            const uint32_t first = __builtin_amdgcn_readlane(incl - nu, r);
            x.pos = (x.s & ~7u) + (u - first) * kRunUnit + 8u * (uint32_t)lane;
            x.v = *reinterpret_cast<const uint4*>(ra.r.ids + x.pos);
            return x;
        };
        uint32_t u = turn;
        if (u < total) {
            RunUnit cur = fetch(u);
            for (;;) {
                const uint32_t un = u + kRunWaves;
                RunUnit nxt = cur;
                if (un < total)
                    nxt = fetch(un);
                // uniform: the whole unit inside its run
                const uint32_t p0 = __builtin_amdgcn_readfirstlane(cur.pos);
                if (p0 >= cur.s && p0 + kRunUnit - cur.s <= cur.len)
                    run_count8<LB, false>(cur, cnt);
                else
                    run_count8<LB, true>(cur, cnt);
                u = un;
                if (un >= total)
                    break;
                cur = nxt;
            }
        }
        // the next window starts with the wave after the one that took the last unit
        turn = (turn + kRunWaves - total % kRunWaves) % kRunWaves;
    }
    __syncthreads();
    run_select<LB>(a, s_cnt4, q, t << kRunTileLog, s_sel);
}

}  // namespace gh
