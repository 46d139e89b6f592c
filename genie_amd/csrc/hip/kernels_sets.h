// Matrix form of the set-valued batched search: the count of a (query,
// object) pair as a product over the index's most frequent keys on the matrix
// cores, plus the postings of the query's other keys scattered into LDS.
//
//     count(q, o) = sum over hot keys of w_q(k) mult_o(k)      (MFMA, i8)
//                 + sum over q's other keys of w_q(k) mult_o(k) (scatter)
//
// Token frequencies are skewed: on documents of 5-40 tokens drawn Zipf(1.05)
// from a million, the 64 most frequent keys hold 41% of the occurrences and
// 99% of the pairs' (query key, document key) matches.  A product with the 64
// hot columns costs one 16x16x64 MFMA for 256 counts whatever the queries
// name; what is left, about 0.06 additions a count, is cheap as LDS atomics
// on byte counters.
//
// Three classes of keys, fixed at index creation by list length:
//   hot   the 64 longest lists (multiplicities up to 127): a byte column each
//         of `hot`, 64 bytes per object;
//   mid   lists of at least half an id per 2,048-object tile: 16-bit ids
//         tile-major (as kernels_runs.h), a directory entry per (tile, key);
//   tail  all others: a batch's tail postings are sorted by tile once per
//         run (k_set_events), one word each.
#pragma once
#include "kernels_dense.h"
#include "kernels_runs.h"

namespace gh {

constexpr uint32_t kSmTileLog = 11;
constexpr uint32_t kSmTile = 1u << kSmTileLog;  // objects per tile
constexpr uint32_t kSmHot = 64;                 // hot keys: one K step of the i8 MFMA
constexpr uint32_t kSmHotMult = 127;            // largest multiplicity of a hot key (i8)
constexpr uint32_t kSmMaxMid = 16384;
constexpr uint32_t kSmMaxTiles = 16000;         // hot matrix below 2 GiB, tile counters of k_set_events in LDS
constexpr int kSmThreads = 512;
constexpr int kSmWaves = kSmThreads / kWave;
// Staged candidates between two flushes, a word each: count (11 bits, below
// kSetNoQuery) | query of the group << 11 | object within the flush's tiles << 16.
constexpr uint32_t kSmStage = 2048;
constexpr uint32_t kSmFlushTiles = 16;
static_assert(kSetCountPlanes == 11 && kSmFlushTiles << kSmTileLog <= 1u << 16 && kSmStage % 512 == 0, "stage words");
constexpr int kSmSlots = 2;                     // mid slots a thread keeps in registers
constexpr uint32_t kSmMidPad = 8;               // ids past the last run that a window may read

constexpr uint32_t kSmTail = 0xFFFFFFFFu;       // class of a tail key
constexpr uint64_t kSmMaxEvents = 1ull << 28;   // tail postings of a batch (1 GiB); more run on the forward lists

typedef int sm_v4i __attribute__((ext_vector_type(4)));

// One (query, mid key) pair takes `c` slots; slot j of them counts the key's
// 8-id windows j, j + c, ... of every tile.  c covers the windows that the
// key's runs usually have, so that mostly every slot is one 16-byte load.
// x: rank | query << 16 | weight << 21; y: j | c << 16.
struct SetArgs {
    const uint8_t* hot;        // [tiles * kSmTile][64] multiplicities of the hot keys
    const uint16_t* mid_ids;   // tile-major ids of the mid keys
    const uint32_t* mid_ptr;   // [n_tiles * n_mid + 1]
    uint32_t n_mid, n_tiles, n_objects;
    uint32_t G, n_queries;
    const uint8_t* wq;         // [G][32][64] weights of the hot keys
    const uint2* slots;
    const uint32_t* slot_ptr;  // [G + 1]
    const uint32_t* events;    // object in tile | query << 11 | weight << 16
    const uint32_t* ev_base;   // [G] first event of each group
    const uint32_t* ev_ptr;    // [G][n_tiles + 1]
    const uint32_t* list;      // sample: tiles of kDenseTile objects
    uint32_t n_list;
    const uint32_t* units;     // groups (x2 + half for 16-bit counters) this launch counts
    uint32_t n_units, chunks;
    const uint32_t* gthr;
    const uint32_t* redo;      // [G] groups to count again (null: every group)
    uint32_t* hist;
    const uint32_t* hshift;
    uint32_t* cand_cnt;
    const uint32_t* cand_cap;
    const uint64_t* cand_base;
    uint64_t* cand;
    uint32_t* overflow;
};

// ---- index creation --------------------------------------------------------

// gridDim.y workgroups per hot key: its column of the hot matrix (cleared before).
__global__ void __launch_bounds__(256) k_set_hot(const uint32_t* __restrict__ post,
                                                  const uint32_t* __restrict__ key_start,
                                                  const uint32_t* __restrict__ hot_keys, uint8_t* __restrict__ hot)
{
    const uint32_t j = blockIdx.x, k = hot_keys[j], s = key_start[k], e = key_start[k + 1];
    for (uint32_t p = s + blockIdx.y * blockDim.x + threadIdx.x; p < e; p += gridDim.y * blockDim.x) {
        const uint32_t o = post[p];
        if (p > s && post[p - 1] == o)
            continue;  // the object's first occurrence writes its multiplicity
        uint32_t m = 1;
        while (p + m < e && post[p + m] == o)
            ++m;
        hot[(uint64_t)o * kSmHot + j] = (uint8_t)m;
    }
}

// The tail keys' postings one list after the other (start[k + 1] = start[k] for
// the other keys): a wave per key, or every gridDim.x-th.
__global__ void __launch_bounds__(kWave) k_set_tail(const uint32_t* __restrict__ post,
                                                    const uint32_t* __restrict__ key_start,
                                                    const uint32_t* __restrict__ start, uint32_t n_keys,
                                                    uint32_t* __restrict__ out)
{
    for (uint32_t k = blockIdx.x; k < n_keys; k += gridDim.x)
        for (uint32_t i = threadIdx.x; i < start[k + 1] - start[k]; i += kWave)
            out[start[k] + i] = post[key_start[k] + i];
}

// ---- per run ---------------------------------------------------------------

// Tail pairs (key, query | weight << 5) of each group, their postings sorted
// by tile: one workgroup per group counts them per tile in LDS, lays the
// tiles out and writes one word per posting.  Two passes over lists that the
// first leaves in L2.
__global__ void __launch_bounds__(1024) k_set_events(const uint32_t* __restrict__ post,
                                                     const uint32_t* __restrict__ key_start,
                                                     const uint2* __restrict__ pairs,
                                                     const uint32_t* __restrict__ pair_ptr, uint32_t n_tiles,
                                                     const uint32_t* __restrict__ ev_base,
                                                     uint32_t* __restrict__ ev_ptr, uint32_t* __restrict__ events)
{
    __shared__ uint32_t s_cnt[kSmMaxTiles];
    __shared__ uint32_t s_w[16];
    const uint32_t g = blockIdx.x, tid = threadIdx.x, lane = lane_id(), wv = tid >> 6;
    for (uint32_t i = tid; i < n_tiles; i += 1024)
        s_cnt[i] = 0;
    __syncthreads();
    const uint32_t p0 = pair_ptr[g], p1 = pair_ptr[g + 1];
    // 16 lanes a pair: tail lists are short
    const uint32_t sub = tid & 15u;
    for (uint32_t i = p0 + (tid >> 4); i < p1; i += 64) {
        const uint32_t k = pairs[i].x;
        const uint32_t e = key_start[k + 1];
        for (uint32_t p = key_start[k] + sub; p < e; p += 16)
            atomicAdd(&s_cnt[post[p] >> kSmTileLog], 1u);
    }
    __syncthreads();
    // exclusive prefix of the tile counts, in place
    uint32_t carry = 0;
    for (uint32_t b = 0; b < n_tiles; b += 1024) {
        const uint32_t v = b + tid < n_tiles ? s_cnt[b + tid] : 0u;
        const uint32_t incl = wave_incl_scan(v);
        if (lane == kWave - 1)
            s_w[wv] = incl;
        __syncthreads();
        uint32_t off = carry, all = carry;
        for (uint32_t w = 0; w < 16; ++w) {
            off += w < wv ? s_w[w] : 0u;
            all += s_w[w];
        }
        if (b + tid < n_tiles) {
            s_cnt[b + tid] = off + incl - v;
            ev_ptr[(uint64_t)g * (n_tiles + 1) + b + tid] = off + incl - v;
        }
        carry = all;
        __syncthreads();
    }
    if (tid == 0)
        ev_ptr[(uint64_t)g * (n_tiles + 1) + n_tiles] = carry;
    uint32_t* out = events + ev_base[g];
    for (uint32_t i = p0 + (tid >> 4); i < p1; i += 64) {
        const uint2 pr = pairs[i];
        const uint32_t e = key_start[pr.x + 1];
        const uint32_t tag = (pr.y & 31u) << kSmTileLog | (pr.y >> 5) << 16;
        for (uint32_t p = key_start[pr.x] + sub; p < e; p += 16) {
            const uint32_t o = post[p];
            out[atomicAdd(&s_cnt[o >> kSmTileLog], 1u)] = (o & (kSmTile - 1u)) | tag;
        }
    }
}

// Byte (or 16-bit) counters of one tile: a row per query, padded by 16 bytes
// so that the rows of 8 queries start in different banks.  A byte counts from 0
// to the 255 that the host admits, so that no addition carries into the next
// object's; the products, whose operands are i8, read it less 128 (the top bit
// flipped).
template <bool W16>
struct SmTab {
    static constexpr uint32_t kRows = W16 ? 16u : 32u;
    static constexpr uint32_t kRow = kSmTile * (W16 ? 2u : 1u) + 16u;
    // object o of the row at byte `row` of the table (a multiple of 16)
    static __device__ __forceinline__ void add(uint8_t* tab, uint32_t row, uint32_t o, uint32_t w)
    {
        const uint32_t a = W16 ? 2u * o : o;
        atomicAdd(reinterpret_cast<uint32_t*>(tab + (row + (a & ~3u))), w << (8u * (a & 3u)));
    }
};

// The host keeps every array read this way below 2 GiB.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sm_rsrc(const void* p)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, 0x7FFFFFFF, 0x00020000);
}

// One workgroup of 512 threads counts a unit (a group of 32 queries, or half
// of one with 16-bit counters; one chunk of the tiles); two workgroups a CU,
// so that one's scatter covers the other's products.  Per tile:
//   scatter  the mid slots' windows and the tail events into the byte
//            counters: loaded during the previous tile's products;
//   products every wave takes 256 objects: per 64 objects and 16 queries, 4
//            tiles of D = hot x weights, to which the byte counters come as a
//            second product with a selection matrix (a lane's 16 bytes are the
//            B operand of 64 objects as they lie), so that no instruction
//            unpacks a counter (with a selection of K = 32, whose operand would
//            be half as wide, the chain after a K = 64 product came out wrong);
//   a lane whose largest D reaches its query's threshold has candidates.
// 2M documents of 5-40 tokens, 16,384 weighted queries: 5.95 ms for 33.6 G
// counts (the forward lists: 22.6 ms).  VALU issues in about half of the
// cycles (scatter 30%, emission 25% of it), the matrix cores in 28%; the rest
// is the latency of LDS atomics, barriers and L2 between the phases.
// A is read with object 16 (m / 4) + 4 i + m % 4 of the 64 in row m of product
// i, so that the 16 results of a lane are the 16 objects of its counter bytes.
template <bool SAMPLE, bool W16>
__global__ void __launch_bounds__(kSmThreads, 4) k_set_count(SetArgs a)
{
    using Tab = SmTab<W16>;
    constexpr int NT = W16 ? 1 : 2;  // products of 16 queries
    constexpr uint32_t HB = 256;
    __shared__ uint4 s_tab4[Tab::kRows * Tab::kRow / 16];
    __shared__ uint32_t s_hist[SAMPLE ? Tab::kRows * HB : 1];
    __shared__ uint32_t s_stage[SAMPLE ? 1 : kSmStage];
    __shared__ uint32_t s_qcnt[32], s_qbase[32], s_nhit;
    uint8_t* tab = reinterpret_cast<uint8_t*>(s_tab4);
    const uint32_t tid = threadIdx.x, lane = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ui = blockIdx.x % a.n_units, chunk = blockIdx.x / a.n_units;
    const uint32_t unit = a.units[ui];
    const uint32_t g = W16 ? unit >> 1 : unit, q0 = W16 ? (unit & 1u) * 16u : 0u;  // first query of the rows
    if (a.redo && !a.redo[g])
        return;  // the whole workgroup, before any barrier
    // this chunk's tiles: a range of the index's, or of the sample list's
    const uint32_t nt_all = SAMPLE ? a.n_list * (kDenseTile / kSmTile) : a.n_tiles;
    const uint32_t ti0 = (uint32_t)((uint64_t)nt_all * chunk / a.chunks);
    const uint32_t ti1 = (uint32_t)((uint64_t)nt_all * (chunk + 1) / a.chunks);
    auto tile_of = [&](uint32_t i) {
        if constexpr (SAMPLE)  // the second half of the index's last sample tile may lie past its end
            return min(a.list[i / (kDenseTile / kSmTile)] * (kDenseTile / kSmTile) + i % (kDenseTile / kSmTile),
                       a.n_tiles);
        else
            return i;
    };

    for (uint32_t i = tid; i < Tab::kRows * Tab::kRow / 16; i += kSmThreads)
        s_tab4[i] = make_uint4(0, 0, 0, 0);
    if (tid < 32)
        s_qcnt[tid] = 0;
    if (tid == 0)
        s_nhit = 0;
    if constexpr (SAMPLE)
        for (uint32_t i = tid; i < Tab::kRows * HB; i += kSmThreads)
            s_hist[i] = 0;

    // B operands, thresholds (or histogram shifts) of this lane's queries; the
    // products of byte counters are counts less 128, their thresholds too
    const uint32_t n = lane & 15u, quad = lane >> 4;
    constexpr int kBias = W16 ? 0 : 128;
    sm_v4i bw[NT];
    int thr[NT];
    uint32_t shift[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) {
        const uint32_t jq = q0 + 16u * i + n, q = g * 32u + jq;
        bw[i] = *reinterpret_cast<const sm_v4i*>(a.wq + ((uint64_t)g * 32u + jq) * kSmHot + 16u * quad);
        if constexpr (SAMPLE)
            shift[i] = a.hshift[min(q, a.n_queries - 1u)];
        else
            thr[i] = (q < a.n_queries ? (int)a.gthr[q] : 1 << 20) - kBias;
    }
    // selection matrices: row m of product i takes object 16 (m / 4) + 4 i + m % 4,
    // byte 4 i + m % 4 of the lanes of quad m / 4
    const int one = quad == n >> 2 ? 1 << (8 * (n & 3u)) : 0;
    const sm_v4i sel[4] = {{one, 0, 0, 0}, {0, one, 0, 0}, {0, 0, one, 0}, {0, 0, 0, one}};

    // mid slots of this thread
    const uint32_t sp0 = a.slot_ptr[g], n_slots = a.slot_ptr[g + 1] - sp0;
    uint2 slot[kSmSlots];
#pragma unroll
    for (int r = 0; r < kSmSlots; ++r) {
        const uint32_t i = tid + r * kSmThreads;
        slot[r] = i < n_slots ? a.slots[sp0 + i] : make_uint2(0, 1u << 16);
        if (((slot[r].x >> 16) & 31u) - q0 >= Tab::kRows)
            slot[r].x = 0;  // the other half's query: weight 0, no run
    }
    // loads through buffers: 32-bit offsets, the tile's part in scalar registers
    const __amdgpu_buffer_rsrc_t r_hot = sm_rsrc(a.hot), r_mid = sm_rsrc(a.mid_ids), r_ptr = sm_rsrc(a.mid_ptr),
                                 r_ev = sm_rsrc(a.events + a.ev_base[g]);
    auto run_of = [&](uint32_t rank, uint32_t t) {
        const uint32_t s0 = t * a.n_mid * 4u;
        return make_uint2(__builtin_amdgcn_raw_buffer_load_b32(r_ptr, rank * 4u, s0, 0),
                          __builtin_amdgcn_raw_buffer_load_b32(r_ptr, rank * 4u + 4u, s0, 0));
    };
    auto window = [&](uint32_t p) { return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r_mid, p * 2u, 0, 0)); };
    // adds the ids of a window (8 of them, at position p0) that lie in the run
    // [r.x, r.y), which reaches into the window: a bit each, and no branches
    auto add_window = [&](const uint4& v, uint32_t p0, const uint2& r, uint32_t sx) {
        const uint32_t x[4] = {v.x, v.y, v.z, v.w};
        const uint32_t row = (((sx >> 16) & 31u) - q0) * Tab::kRow, w = sx >> 21;
        const uint32_t lo = r.x > p0 ? r.x - p0 : 0u, hi = min(r.y - p0, 8u);
        const uint32_t in = (1u << hi) - (1u << lo);
#pragma unroll
        for (int j = 0; j < 8; ++j)
            Tab::add(tab, row, j & 1 ? x[j >> 1] >> 16 : x[j >> 1] & 0xFFFFu,
                     (uint32_t)__builtin_amdgcn_sbfe((int)in, j, 1) & w);
    };
    const uint32_t* evp = a.ev_ptr + (uint64_t)g * (a.n_tiles + 1);

    // pipeline: run and event bounds two tiles ahead, ids, events and the first
    // rows of the hot matrix one tile ahead
    uint2 run[kSmSlots], run_n[kSmSlots], eb, eb_n;
    uint4 win[kSmSlots];
    uint32_t evv = 0;
    auto load_bounds = [&](uint32_t i, uint2 (&r)[kSmSlots], uint2& e) {
        const uint32_t t = i < ti1 ? tile_of(i) : a.n_tiles;
        e = t < a.n_tiles ? make_uint2(evp[t], evp[t + 1]) : make_uint2(0, 0);
#pragma unroll
        for (int k = 0; k < kSmSlots; ++k) {
            r[k] = make_uint2(0, 0);
            if (t < a.n_tiles && slot[k].x >> 21)
                r[k] = run_of(slot[k].x & 0xFFFFu, t);
        }
    };
    auto load_ids = [&]() {  // of `run` and `eb`
#pragma unroll
        for (int k = 0; k < kSmSlots; ++k) {
            const uint32_t p = (run[k].x & ~7u) + 8u * (slot[k].y & 0xFFFFu);
            if (p < run[k].y)
                win[k] = window(p);
        }
        if (eb.x + tid < eb.y)
            evv = __builtin_amdgcn_raw_buffer_load_b32(r_ev, (eb.x + tid) * 4u, 0, 0);
    };
    // 64 objects of the hot matrix: block b of the tile's rows of this wave
    const uint32_t lane_row = (wv * 256u + 16u * (n >> 2) + (n & 3u)) * kSmHot + 16u * quad;
    auto load_hot = [&](uint32_t t, int b, sm_v4i (&ah)[4]) {
        const uint32_t s0 = min(t, a.n_tiles - 1u) * (kSmTile * kSmHot) + (uint32_t)b * (64u * kSmHot);
#pragma unroll
        for (int i = 0; i < 4; ++i)
            ah[i] = __builtin_bit_cast(sm_v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                                   r_hot, lane_row + (uint32_t)i * (4u * kSmHot), s0, 0));
    };
    sm_v4i hot[2][4];
    load_bounds(ti0, run, eb);
    load_ids();
    load_hot(tile_of(ti0), 0, hot[0]);
    load_bounds(ti0 + 1, run_n, eb_n);
    uint32_t staged_tiles = 0;
    __syncthreads();

    for (uint32_t ti = ti0; ti < ti1; ++ti) {
        const uint32_t t = tile_of(ti);
        // the slots' fields are taken apart where they are used: kept apart
        // over the loop they would spill
#pragma unroll
        for (int k = 0; k < kSmSlots; ++k)
            __asm__ volatile("" : "+v"(slot[k].x), "+v"(slot[k].y));
        // ---- scatter
#pragma unroll
        for (int k = 0; k < kSmSlots; ++k) {
            const uint32_t step = 8u * (slot[k].y >> 16), p = (run[k].x & ~7u) + 8u * (slot[k].y & 0xFFFFu);
            if (p < run[k].y)
                add_window(win[k], p, run[k], slot[k].x);
            for (uint32_t pn = p + step; pn < run[k].y; pn += step)  // a run longer than its slots, rarely
                add_window(window(pn), pn, run[k], slot[k].x);
        }
        // slots past the registers'
        for (uint32_t i = tid + kSmSlots * kSmThreads; i < n_slots && t < a.n_tiles; i += kSmThreads) {
            const uint2 d = a.slots[sp0 + i];
            if (((d.x >> 16) & 31u) - q0 >= Tab::kRows)
                continue;
            const uint2 r = run_of(d.x & 0xFFFFu, t);
            for (uint32_t p = (r.x & ~7u) + 8u * (d.y & 0xFFFFu); p < r.y; p += 8u * (d.y >> 16))
                add_window(window(p), p, r, d.x);
        }
        for (uint32_t i = eb.x + tid; i < eb.y; i += kSmThreads) {
            const uint32_t v = i == eb.x + tid ? evv : __builtin_amdgcn_raw_buffer_load_b32(r_ev, i * 4u, 0, 0);
            const uint32_t row = ((v >> kSmTileLog) & 31u) - q0;
            if (row < Tab::kRows)
                Tab::add(tab, row * Tab::kRow, v & (kSmTile - 1u), v >> 16);
        }
#pragma unroll
        for (int k = 0; k < kSmSlots; ++k)
            run[k] = run_n[k];
        eb = eb_n;
        load_ids();
        load_bounds(ti + 2, run_n, eb_n);
        __syncthreads();

        // a candidate: staged, or straight to its query's list when the stage is full
        auto emit = [&](uint32_t count, int h, uint32_t o) {
            const uint32_t x = atomicAdd(&s_nhit, 1u);
            uint32_t v = count | (q0 + 16u * h + n) << 11 | (staged_tiles << kSmTileLog | o) << 16;
            if (x < kSmStage) {
                s_stage[x] = v;
            } else {
                __asm__ volatile("" : "+v"(v));  // no address of this rare path is kept over the loop
                const uint32_t q = g * 32u + ((v >> 11) & 31u), at = atomicAdd(&a.cand_cnt[q], 1u);
                if (at < a.cand_cap[q])
                    a.cand[a.cand_base[q] + at] = make_key(count, t * kSmTile + o);
                else
                    atomicOr(a.overflow, 1u);
            }
        };
        // ---- products: objects t * kSmTile + wv * 256 + 64 b + 16 quad + 0..15 of this lane
        if (t < a.n_tiles) {  // uniform
            auto block = [&](int b, const sm_v4i (&ah)[4]) {
#pragma unroll
                for (int h = 0; h < NT; ++h) {
                    sm_v4i dd[4];
                    uint8_t* cell = tab + (16u * h + n) * Tab::kRow + (W16 ? 2u : 1u) * (wv * 256u + 64u * b + 16u * quad);
                    if constexpr (W16) {
                        uint4* c4 = reinterpret_cast<uint4*>(cell);
                        const uint4 c0 = c4[0], c1 = c4[1];
                        c4[0] = make_uint4(0, 0, 0, 0);
                        c4[1] = make_uint4(0, 0, 0, 0);
                        const uint32_t cw[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const sm_v4i ci = {(int)(cw[2 * i] & 0xFFFFu), (int)(cw[2 * i] >> 16),
                                               (int)(cw[2 * i + 1] & 0xFFFFu), (int)(cw[2 * i + 1] >> 16)};
                            dd[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[i], bw[h], ci, 0, 0, 0);
                        }
                    } else {
                        const sm_v4i cold = *reinterpret_cast<const sm_v4i*>(cell) ^ (int)0x80808080u;
                        *reinterpret_cast<sm_v4i*>(cell) = sm_v4i{0, 0, 0, 0};
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            dd[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[i], bw[h], sm_v4i{0, 0, 0, 0}, 0, 0, 0);
                            dd[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(sel[i], cold, dd[i], 0, 0, 0);
                        }
                    }
                    if constexpr (SAMPLE) {
                        // nonzero counts only (k_dense_thresh)
#pragma unroll
                        for (int i = 0; i < 4; ++i)
#pragma unroll
                            for (int r = 0; r < 4; ++r) {
                                const uint32_t c = (uint32_t)(dd[i][r] + kBias);
                                if (c)
                                    atomicAdd(&s_hist[(16u * h + n) * HB + min(c >> shift[h], HB - 1u)], 1u);
                            }
                    } else {
                        int m[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i)
                            m[i] = max(max(dd[i][0], dd[i][1]), max(dd[i][2], dd[i][3]));
                        if (ballot(max(max(m[0], m[1]), max(m[2], m[3])) >= thr[h]))
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (m[i] >= thr[h])
#pragma unroll
                                    for (int r = 0; r < 4; ++r)
                                        if (dd[i][r] >= thr[h])
                                            emit((uint32_t)(dd[i][r] + kBias), h,
                                                 wv * 256u + 64u * b + 16u * quad + 4u * i + r);
                    }
                }
            };
#pragma unroll 1
            for (int b = 0; b < 4; b += 2) {
                load_hot(t, b + 1, hot[1]);
                block(b, hot[0]);
                if (b == 0)
                    load_hot(t, 2, hot[0]);
                else
                    load_hot(ti + 1 < ti1 ? tile_of(ti + 1) : t, 0, hot[0]);
                block(b + 1, hot[1]);
            }
        }
        __syncthreads();
        if constexpr (!SAMPLE)
            // (uniform; a stage that is half full is emptied at once: where many
            // objects tie, one flush in 16 tiles left most candidates to emit's
            // atomics on the query's counter, one each: 1M documents of 1-8 of
            // 2,000 tokens, 1,024 queries of up to 8 tokens: 3,240 us a run, 620 here)
            if (++staged_tiles == kSmFlushTiles || ti + 1 == ti1 || s_nhit > kSmStage / 2) {
                // every staged candidate's rank in its query, one reservation per
                // query, then the candidates to their slots (the stage is next
                // written after the scatter's barrier)
                const uint32_t t0 = t + 1u - staged_tiles, nh = min(s_nhit, kSmStage);
                staged_tiles = 0;
                uint32_t rank[kSmStage / kSmThreads];
#pragma unroll
                for (uint32_t j = 0; j < kSmStage / kSmThreads; ++j)
                    if (j * kSmThreads + tid < nh)
                        rank[j] = atomicAdd(&s_qcnt[(s_stage[j * kSmThreads + tid] >> 11) & 31u], 1u);
                __syncthreads();
                if (tid < 32 && s_qcnt[tid])
                    s_qbase[tid] = atomicAdd(&a.cand_cnt[g * 32u + tid], s_qcnt[tid]);
                if (tid == 0)
                    s_nhit = 0;
                __syncthreads();
                if (tid < 32)
                    s_qcnt[tid] = 0;
#pragma unroll
                for (uint32_t j = 0; j < kSmStage / kSmThreads; ++j)
                    if (j * kSmThreads + tid < nh) {
                        const uint32_t v = s_stage[j * kSmThreads + tid], q = g * 32u + ((v >> 11) & 31u);
                        const uint32_t at = s_qbase[(v >> 11) & 31u] + rank[j];
                        if (at < a.cand_cap[q])
                            a.cand[a.cand_base[q] + at] = make_key(v & 2047u, t0 * kSmTile + (v >> 16));
                        else
                            atomicOr(a.overflow, 1u);
                    }
            }
    }
    if constexpr (SAMPLE) {
        for (uint32_t i = tid; i < Tab::kRows * HB; i += kSmThreads) {
            const uint32_t q = g * 32u + q0 + i / HB, v = s_hist[i];
            if (v && q < a.n_queries)
                atomicAdd(&a.hist[(uint64_t)q * kDenseBins + i % HB], v);
        }
    }
}

}  // namespace gh
