// Greedy beam search over the hybrid graph: one workgroup per query; the candidate pool, the
// query's dense row, its sparse-term tables and the fresh-neighbour list in LDS; an exact
// visited bitmap per workgroup in HBM.
#include <cmath>
#include <mutex>
#include <type_traits>

#include "apoe_internal.h"

namespace apoe {

constexpr int MAX_NEW = 64;   // fresh candidates per step: one lane each in wave 0
// Tuning constants: the measured best on MI355X.
#define APOE_SEARCH_WAVES_PER_EU 6 // plain search: 12 queries per CU fit its LDS; the other modes need more LDS per query and stay at 5 (a macro: it sits in an attribute)
constexpr int EVAL_BATCH = 3;  // candidates whose sparse parts a wave keeps in flight together
constexpr int CODE_BATCH = 3;  // rows whose codes a wave keeps in flight together
constexpr int DENSE_BATCH = 1; // dense rows a wave keeps in flight together
constexpr int MERGE_ROUNDS = 4; // 64-element rounds of the pool that the merge moves per LDS round trip
constexpr int STATS = 10;     // counters of a launch; the workspace keeps 16 words for them
constexpr int SKETCH_BATCH = 4; // sketches a wave keeps in flight together
constexpr int RING = 32;      // keyword-filter search: evicted keyword hits kept beside the pool (query.cu:18)

// What the kernel does on top of the plain beam search.
enum SearchMode { MODE_PLAIN = 0, MODE_KG = 1, MODE_KEYWORD = 2 };

// Arguments that a query needs once (when it starts or ends) stay in device memory and are read
// where they are used; the rest travels by value. Scalar registers are the scarce resource of this
// kernel: every argument held in one for the whole launch pushes loop state into vector registers.
struct SearchCold {
    SetView Q;
    const uint32_t* entry;
    uint32_t n_entry;
    float w_d, w_s, w_b;
    uint32_t q_begin;
    uint32_t* out_ids;
    float* out_dist;
    const uint32_t *q2e_off, *q2e_idx;
};

struct SearchArgs {
    CorpusView C;
    const SearchCold* cold;
    const uint32_t* graph;
    uint32_t W, degree;
    uint32_t paths;
    uint32_t cands, max_iter, q_count;
    uint32_t* bitmaps;     // one visited bitmap per workgroup
    uint32_t bitmap_words; // multiple of 4
    const SketchMeta* sketch_meta;
    const uint4* sketch;   // null: the corpus has none
    uint32_t* codes;       // of the query's dense row, 1 KB per workgroup: in device memory (it is read beside sketches, which take longer), since a
                           // kilobyte of LDS more costs long batches a resident query per CU (12 -> 11: 3 %)
    unsigned long long* work; // [0] next query, [1] expansions, [2] evaluations, [3] nnz splade, [4] nnz bm25, [5] dense rows (fp32 or half) read in the walk,
                              // [6] pool entries evaluated again in fp32, [7] their pairs, [8] sketches read, [9] pairs of the evaluations that codes left open less those that they settled
    uint32_t coded;           // 1: the records carry codes of their values and the search may ask them
    uint32_t full_eval;       // 1: read the dense row of every candidate (no bound test)
    const uint16_t* half;     // not null: the walk takes dense parts from the half-precision rows, the final pool is evaluated again in fp32
    uint32_t slots_s, slots_b, ovf_cap; // buckets of the query's SPLADE / BM25 term table, entries of the overflow list
    // knowledge graph (KG kernels only)
    const uint32_t *e2e_off, *e2e_idx, *e2d_off, *e2d_idx;
    uint32_t n_entities;
    float kg_weight;
};

// LDS carve-up shared by host (size) and device (pointers).
struct SearchLds {
    uint32_t qd, qs, stat, part, tab, ovf, pool_id, pool_dist, pool_ent, pool_hop, new_id, new_dist, new_ent, new_hop, seed_id, seed_ent, seed_dist, link, ring_id,
        ring_dist, ctl, total;
    __host__ __device__ SearchLds(uint32_t slots_s, uint32_t slots_b, uint32_t ovf_cap, uint32_t cands, int mode) {
        const bool kg = mode == MODE_KG, kwd = mode == MODE_KEYWORD;
        // fixed-size arrays first: their offsets are compile-time constants
        uint32_t o = 0;
        qd = o; o += DENSE_BYTES;       // the query's dense row, weight applied
        ctl = o; o += 16 * 4;
        qs = o; o += 4 * 4;             // scale and error of the codes of the query's dense row
        stat = o; o += (STATS + 1) / 2 * 16; // the workgroup's counters (work[1..]), sent once when it leaves; `part` is read 16 bytes at a time
        part = o; o += MAX_NEW * 16;    // of a fresh candidate: descriptor and dense norm until its wave takes them up, then its sparse sum as four
                                        // partial sums (one per 16 lanes)
        new_id = o; o += MAX_NEW * 4;
        new_dist = o; o += MAX_NEW * 4;
        new_ent = o; o += kg || kwd ? MAX_NEW * 4 : 0; // KG: linking entity; keyword search: the hit flag of a fresh candidate
        new_hop = o; o += kg ? MAX_NEW * 4 : 0;
        link = o; o += kg ? MAX_NEW * 4 : 0;
        ring_id = o; o += kwd ? RING * 4 : 0;
        ring_dist = o; o += kwd ? RING * 4 : 0;
        tab = o; o += (slots_s + slots_b) * 16; // two tables (SPLADE, BM25) of buckets of two (key, value) entries; twice as many
                                                // buckets as the longest row of the path has terms keep overflows rare
        ovf = o; o += ovf_cap * 8;              // overflow entries: up to every term of the longest query row
        pool_id = o; o += cands * 4;
        pool_dist = o; o += cands * 4;
        pool_ent = o; o += kg ? cands * 4 : 0;
        pool_hop = o; o += kg ? cands * 4 : 0;
        seed_id = o; o += kg ? (cands + MAX_NEW) * 4 : 0;
        seed_ent = o; o += kg ? (cands + MAX_NEW) * 4 : 0;
        seed_dist = o; o += kg ? (cands + MAX_NEW) * 4 : 0;
        total = o;
    }
};

enum { CTL_QUERY = 0, CTL_PARENT = 1, CTL_NNEW = 2, CTL_NSEED = 3, CTL_NOVF = 4 };

struct Pool {
    uint32_t* id;   // [cands], ascending distance
    float* dist;    // [cands]
    uint32_t* ent;  // KG only
    uint32_t* hop;  // KG only
    uint32_t cands;
};

// Keyword-filter search: pool entries that carry KW_HIT and fall off the pool. Entries are
// appended merge by merge, within one merge from the worst to the best, and slot (count % RING)
// is overwritten, so the ring holds the RING most recent ones: distances never grow along that
// sequence, which makes them the closest evicted hits (query.cu:244-248 appends in atomic order).
struct Ring {
    uint32_t* id;
    float* dist;
    uint32_t n; // appended so far (wave-uniform, wave 0)
};

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Wave 0 only: the new candidates of one expansion, lane l holds the l-th.
struct Fresh {
    float d;
    uint32_t id, ent, hop; // KG: linking entity and hop; keyword-filter search: ent != 0: holds a required keyword
    uint64_t kept;         // lanes whose candidate can enter the pool: the others (with a full pool that is most of them:
                           // everything the bound rejected, and more) are dropped
    uint32_t rank;         // of a kept candidate among the kept ones, by (distance, id); set by fresh_rank
};

template <int MODE>
__device__ __forceinline__ void fresh_load(Fresh& F, const Pool& P, const uint32_t* nid, const float* ndist, const uint32_t* nent, const uint32_t* nhop,
                                           uint32_t n) {
    const int lane = lane_id();
    F.d = INF_DIS;
    F.id = F.ent = EMPTY;
    F.hop = F.rank = 0;
    if (lane < (int)n) {
        F.d = ndist[lane];
        F.id = nid[lane];
        if (MODE == MODE_KG) { F.ent = nent[lane]; F.hop = nhop[lane]; }
        if (MODE == MODE_KEYWORD) F.ent = nent[lane];
    }
    F.kept = __ballot(lane < (int)n && F.d <= P.dist[P.cands - 1]);
}

// The kept candidate that comes first by (distance, id): its lane. F.kept must not be empty.
__device__ __forceinline__ uint32_t fresh_first(const Fresh& F) {
    const bool keep = (F.kept >> lane_id()) & 1;
    const float low = wave_min_dpp(keep ? F.d : __builtin_inff());
    uint64_t at = __ballot(keep && F.d == low);
    uint32_t best = __builtin_ctzll(at);
    for (at &= at - 1; at; at &= at - 1) { // equal distances: the smallest id
        const uint32_t i = __builtin_ctzll(at);
        if ((uint32_t)__builtin_amdgcn_readlane((int)F.id, i) < (uint32_t)__builtin_amdgcn_readlane((int)F.id, best)) best = i;
    }
    return best;
}

__device__ __forceinline__ void fresh_rank(Fresh& F) {
    for (uint64_t rest = F.kept; rest; rest &= rest - 1) { // ids are distinct
        const uint32_t i = __builtin_ctzll(rest);
        const float di = readlane_f32(F.d, i);
        const uint32_t ii = (uint32_t)__builtin_amdgcn_readlane((int)F.id, i);
        F.rank += (di < F.d) || (di == F.d && ii < F.id);
    }
}

// Wave 0 only: the first unexplored pool entry at or behind `from`.
struct Front {
    uint32_t id, slot; // id EMPTY: there is none
    float dist;
};
__device__ __forceinline__ Front pool_front(const Pool& P, uint32_t from) {
    Front f;
    f.id = EMPTY;
    f.slot = P.cands;
    f.dist = INF_DIS;
    const uint32_t lane = lane_id();
    for (uint32_t base = from & ~(uint32_t)(WAVE - 1); base < P.cands; base += WAVE) {
        const uint32_t p = base + lane;
        const uint32_t id = p < P.cands && p >= from ? P.id[p] : EMPTY;
        const float d = p < P.cands ? P.dist[p] : INF_DIS;
        const uint64_t b = __ballot((id & FLAG) == 0);
        if (b) {
            const uint32_t l = __builtin_ctzll(b);
            f.id = (uint32_t)__builtin_amdgcn_readlane((int)id, l);
            f.dist = readlane_f32(d, l);
            f.slot = base + l;
            break;
        }
    }
    return f;
}

// Wave 0 only. Merges the kept new candidates (ranked) into the sorted pool in place: a pool element keeps rank
// pos + #{new <= it}, a new element takes rank #{new before it by (distance, id)} + #{pool < it}, so on equal distance
// the new one goes first (query.cu:181-224); ranks >= cands fall off. The pool is read in groups of MERGE_ROUNDS x 64
// entries from its end, coalesced into registers; every new candidate that can enter (wave-uniform loop over the kept
// lanes) is compared with the whole group at once, which gives the group's shifts (per lane) and the candidate's own
// count of pool entries at or beyond it (population count of the compare mask). A group only writes at or above its own
// positions, into rounds that were read before; the first group whose lowest entry does not move is the last.
// The chain of a merge bounds short batches (one wave works, the others wait): a group costs one LDS round trip plus
// about twenty instructions per kept candidate. Sorting the new ones through LDS first and finding each rank by a binary
// search (one dependent LDS read per halving) took 3 900 cycles a merge at cands 128 and 8 600 at cands 1000 (one query
// per CU); this takes 1 830 and 3 360 (500 queries at cands 1000 on 100 k documents: 10.3 -> 8.0 ms).
// Returns the lowest rank a new element took (cands if none entered).
// Keyword-filter search: a candidate that holds a required keyword enters the pool with KW_HIT set on its id (ordering
// uses the plain id).
template <int MODE>
__device__ __forceinline__ uint32_t sort_merge(const Pool& P, const Fresh& F, Ring& R) {
    constexpr bool KG = MODE == MODE_KG, KWD = MODE == MODE_KEYWORD;
    const int lane = lane_id();
    const uint32_t cands = P.cands;
    const uint64_t kept = F.kept;
    if (kept == 0) return cands;
    const bool keep = (kept >> lane) & 1;
    const float d = F.d;
    uint32_t beyond = 0;   // pool entries at or beyond this lane's candidate
    uint64_t open = kept;  // candidates whose place is not found yet
    for (int top = (int)((cands - 1) & ~(uint32_t)(WAVE - 1));; top -= WAVE * MERGE_ROUNDS) {
        float v[MERGE_ROUNDS];
        uint32_t pid[MERGE_ROUNDS], pent[MERGE_ROUNDS], phop[MERGE_ROUNDS], shift[MERGE_ROUNDS];
#pragma unroll
        for (int r = 0; r < MERGE_ROUNDS; r++) {
            const int base = top - r * WAVE;
            const uint32_t p = (uint32_t)(base + lane);
            v[r] = __builtin_nanf(""); // not there: compares false with everything
            pid[r] = pent[r] = phop[r] = shift[r] = 0;
            if (base >= 0 && p < cands) {
                v[r] = P.dist[p];
                pid[r] = P.id[p];
                if (KG) { pent[r] = P.ent[p]; phop[r] = P.hop[p]; }
            }
        }
        auto place = [&](uint32_t i) { // candidate i against every entry of the group
            const float di = readlane_f32(d, i);
            uint32_t cnt = 0;
#pragma unroll
            for (int r = 0; r < MERGE_ROUNDS; r++) {
                const bool at_or_beyond = v[r] >= di;
                cnt += (uint32_t)__popcll(__ballot(at_or_beyond));
                shift[r] += at_or_beyond ? 1u : 0u;
            }
            beyond += (uint32_t)lane == i ? cnt : 0u;
        };
        const int next = top - WAVE * MERGE_ROUNDS;
        uint32_t all = 0; // candidates that go before the whole group
        if (next >= 0) {
            const uint64_t before = __ballot(((open >> lane) & 1) && readlane_f32(v[MERGE_ROUNDS - 1], 0) >= d);
            beyond += (before >> lane) & 1 ? min(cands - (uint32_t)(next + WAVE), (uint32_t)(WAVE * MERGE_ROUNDS)) : 0u;
            all = (uint32_t)__popcll(before);
#pragma unroll
            for (int r = 0; r < MERGE_ROUNDS; r++) shift[r] = all;
            open &= ~before;
            for (uint64_t rest = open; rest; rest &= rest - 1) place(__builtin_ctzll(rest));
            open = before;
        } else {
            for (uint64_t rest = open; rest; rest &= rest - 1) place(__builtin_ctzll(rest));
        }
        if (KWD && top + WAVE >= (int)cands) {
            // the pool entries that fall off all sit in the last 64 positions; lane l looks at the l-th from the end
            uint32_t n_off = 0;
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const uint32_t p = (uint32_t)(top - r * WAVE + lane);
                n_off += (uint32_t)__popcll(__ballot(shift[r] > 0 && p < cands && p + shift[r] >= cands));
            }
            uint32_t eid = EMPTY;
            float ed = 0.f;
            if ((uint32_t)lane < n_off) { eid = P.id[cands - 1 - lane]; ed = P.dist[cands - 1 - lane]; }
            const bool hit = eid != EMPTY && (eid & KW_HIT);
            const uint64_t hb = __ballot(hit);
            const uint32_t cnt = __popcll(hb), nth = __popcll(hb & ((1ull << lane) - 1));
            if (hit && nth + RING >= cnt) {
                const uint32_t slot = (R.n + nth) % RING;
                R.id[slot] = eid & ID_MASK;
                R.dist[slot] = ed;
            }
            R.n += cnt;
        }
        wave_fence();
#pragma unroll
        for (int r = 0; r < MERGE_ROUNDS; r++) {
            const uint32_t dst = (uint32_t)(top - r * WAVE + lane) + shift[r];
            if (shift[r] > 0 && dst < cands) {
                P.dist[dst] = v[r];
                P.id[dst] = pid[r];
                if (KG) { P.ent[dst] = pent[r]; P.hop[dst] = phop[r]; }
            }
        }
        wave_fence();
        if (next < 0 || all == 0) break; // none goes before the group: nothing below it moves
    }
    const uint32_t lb = cands - beyond; // #{pool < mine}
    const uint32_t at = lb + F.rank;
    if (keep && at < cands) {
        P.dist[at] = d;
        P.id[at] = KWD && F.ent ? F.id | KW_HIT : F.id;
        if (KG) { P.ent[at] = F.ent; P.hop[at] = F.hop; }
    }
    wave_fence();
    return (uint32_t)__builtin_amdgcn_readlane((int)lb, __builtin_ctzll(__ballot(keep && F.rank == 0)));
}

// A node's row (id wave-uniform) as a scalar global pointer: left alone, the compiler keeps graph + lane in a vector register
// pair for the whole launch, spills it, and wave 0 of long batches waits for the spill before it sends its loads (3 % of a
// 10 000-query batch).
typedef __attribute__((address_space(1))) const uint32_t GlobalWord;
__device__ __forceinline__ GlobalWord* graph_row(const SearchArgs& a, uint32_t id) {
    GlobalWord* row = (GlobalWord*)(a.graph + (uint64_t)uniform(id) * a.W);
    asm volatile("" : "+s"(row));
    return row;
}

// CODES: pairs are bounded by the codes of their values before they are read (figures where that is done).
template <int NW, int MODE, bool NARROW, bool HALF, bool CODES>
__global__ __launch_bounds__(NW* WAVE) __attribute__((amdgpu_waves_per_eu(MODE == MODE_PLAIN && !HALF ? APOE_SEARCH_WAVES_PER_EU : 5, 8))) void search_kernel(SearchArgs a) {
    constexpr bool KG = MODE == MODE_KG, KWD = MODE == MODE_KEYWORD;
    // Whether wave 0 asks for more than the walk may need (graph row of the first unexplored entry, descriptors of visited neighbours) to
    // have it early: one query's chain gains, a long batch, whose other queries cover the wait, pays in traffic (figures where the walk starts).
    // Knowledge-graph search gains in long batches too (ten queries a CU, a longer chain between two walks: 10 000 queries, 1 M docs,
    // cands 64 / 128 / 160: 10.55 / 18.0 / 22.4 ms ahead, 10.66 / 18.2 / 22.7 when needed).
    constexpr bool AHEAD = NW >= 4 || KG;
    a.C.narrow = NARROW ? 1u : 0u; // the pair format as a compile-time constant: no branch at the loads
    extern __shared__ __align__(16) char smem[];
    const SearchLds L(a.slots_s, a.slots_b, a.ovf_cap, a.cands, MODE);
    // not volatile (barriers separate the waves' accesses): a volatile access through a generic pointer is a flat one, which waits for every
    // load under way (one query 699 -> 663 us, 500 queries of pool 1000 8.27 -> 7.94 ms). Knowledge-graph searches gain 1 to 5 % by that on eight and sixteen
    // waves a query and lose up to 8 on four and two, most in small pools (700 queries, cands 16 / 64 / 256: 2.00 / 3.36 / 6.55 ms volatile, 2.15 / 3.54 / 6.67 not),
    // so they keep it there.
    constexpr bool FLAT = KG && NW <= 4;
    using Word = std::conditional_t<FLAT, volatile uint32_t, uint32_t>;
    using Scalar = std::conditional_t<FLAT, volatile float, float>;
    Word* ctl = reinterpret_cast<Word*>(smem + L.ctl);
    float4* qd = reinterpret_cast<float4*>(smem + L.qd);
    float* part = reinterpret_cast<float*>(smem + L.part);
    QueryTabs T;
    T.b = reinterpret_cast<uint4*>(smem + L.tab);
    T.ovf = reinterpret_cast<uint2*>(smem + L.ovf);
    T.ovf_cap = a.ovf_cap;
    T.n_ovf = const_cast<uint32_t*>(&ctl[CTL_NOVF]);
    T.mask_s = a.slots_s - 1;
    T.mask_b = a.slots_b - 1;
    Pool P;
    P.id = reinterpret_cast<uint32_t*>(smem + L.pool_id);
    P.dist = reinterpret_cast<float*>(smem + L.pool_dist);
    P.ent = reinterpret_cast<uint32_t*>(smem + L.pool_ent);
    P.hop = reinterpret_cast<uint32_t*>(smem + L.pool_hop);
    P.cands = a.cands;
    auto put_desc = [&](uint32_t pos, uint64_t desc, float dn) { // before the barrier in front of the evaluations
        reinterpret_cast<float4*>(part)[pos] = make_float4(__uint_as_float((uint32_t)desc), __uint_as_float((uint32_t)(desc >> 32)), dn, 0.f);
    };
    uint32_t* codes = a.codes + (size_t)blockIdx.x * (SKETCH_BYTES / 4);
    Scalar* qs = reinterpret_cast<Scalar*>(smem + L.qs);
    uint32_t* new_id = reinterpret_cast<uint32_t*>(smem + L.new_id);
    float* new_dist = reinterpret_cast<float*>(smem + L.new_dist);
    uint32_t* new_ent = reinterpret_cast<uint32_t*>(smem + L.new_ent);
    uint32_t* new_hop = reinterpret_cast<uint32_t*>(smem + L.new_hop);
    uint32_t* seed_id = reinterpret_cast<uint32_t*>(smem + L.seed_id);
    uint32_t* seed_ent = reinterpret_cast<uint32_t*>(smem + L.seed_ent);
    float* seed_dist = reinterpret_cast<float*>(smem + L.seed_dist);
    uint32_t* link = reinterpret_cast<uint32_t*>(smem + L.link);
    Ring R;
    R.id = reinterpret_cast<uint32_t*>(smem + L.ring_id);
    R.dist = reinterpret_cast<float*>(smem + L.ring_dist);
    R.n = 0;

    const int tid = threadIdx.x, wave = (int)uniform(tid / WAVE), lane = lane_id();
    const uint32_t cands = a.cands;
    uint32_t* bitmap = a.bitmaps + (size_t)blockIdx.x * a.bitmap_words;
    const uint64_t lane_lt = (1ull << lane) - 1;

    unsigned long long* stat = reinterpret_cast<unsigned long long*>(smem + L.stat);
    if (tid < STATS) stat[tid] = 0;
    while (true) {
        __syncthreads();
        if (tid == 0) ctl[CTL_QUERY] = (uint32_t)atomicAdd(a.work, 1ull);
        __syncthreads();
        const uint32_t qi = uniform(ctl[CTL_QUERY]);
        if (qi >= a.q_count) break;
        const uint32_t q = a.cold->q_begin + qi;

        // ---- reset per-query state ----
        {
            uint4* b4 = reinterpret_cast<uint4*>(bitmap);
            for (uint32_t i = tid; i < a.bitmap_words / 4; i += NW * WAVE) b4[i] = make_uint4(0, 0, 0, 0);
        }
        query_tabs_clear(T, tid, NW * WAVE);
        R.n = 0;
        for (uint32_t i = tid; i < cands; i += NW * WAVE) {
            P.id[i] = EMPTY;
            P.dist[i] = INF_DIS;
            if (KG) { P.ent[i] = EMPTY; P.hop[i] = 0; }
        }
        {
            const float4* src = reinterpret_cast<const float4*>(a.cold->Q.dense + (size_t)q * DIM);
            for (uint32_t i = tid; i < DIM / 4; i += NW * WAVE) {
                const float4 x = src[i];
                qd[i] = make_float4(x.x * a.cold->w_d, x.y * a.cold->w_d, x.z * a.cold->w_d, x.w * a.cold->w_d);
            }
        }
        __threadfence();
        __syncthreads();
        query_tabs_fill<NARROW, KWD>(T, a.cold->Q, q, a.cold->w_s, a.cold->w_b, a.paths & PATH_SPARSE, a.paths & PATH_BM25, tid, NW * WAVE);
        __syncthreads();
        float q_scale = 0.f, q_err = 0.f; // of the query's sketch; scale 0: not used
        const float pv_norm = pivot_dense_norm_lds(qd);
        if (a.sketch && (a.paths & PATH_DENSE)) { // every wave works out the scale and the error, all share the codes
            float4 x[NV];
            float top = 0.f, left = 0.f;
#pragma unroll
            for (int i = 0; i < NV; i++) { x[i] = qd[lane + WAVE * i]; top = fmaxf(top, max_abs4(x[i])); }
            top = -wave_min_dpp(-top);
            const float per = sketch_per(top);
            if (per > 0.f) {
                q_scale = top / 127.f;
#pragma unroll
                for (int i = 0; i < NV; i++) {
                    left += sketch_residual(x[i], per, q_scale);
                    if (wave == i % NW) codes[lane + WAVE * i] = sketch_pack(x[i], per);
                }
                q_err = 1.0001f * sqrtf(wave_sum_dpp(left));
            }
        }
        if (tid == 0) { qs[0] = q_scale; qs[1] = q_err; }
        const bool sketched = __builtin_amdgcn_readfirstlane((int)(q_scale > 0.f)) != 0;
        uint32_t st_exp = 0, st_eval = 0, st_dense = 0, st_again = 0, st_again_pairs = 0, st_sketch = 0; // wave-uniform counters of one query
        uint32_t ln_s = 0, ln_b = 0, ln_coded = 0;      // pairs read for the candidates this lane decided; of those that codes settled
        uint32_t st_reread = 0;                         // wave-uniform: pairs of the candidates that codes left open
        Front front; // wave 0: the first unexplored pool entry
        front.id = EMPTY;
        front.slot = 0;
        front.dist = INF_DIS;

        // ---- seeds ----
        if (!KG) {
            // entry points (query.cu:440-485)
            if (wave == 0) {
                uint32_t c = lane < (int)a.cold->n_entry ? a.cold->entry[lane] : EMPTY;
                bool fresh = false;
                if (c < a.C.n) {
                    const uint32_t bit = 1u << (c & 31);
                    fresh = !(atomicOr(&bitmap[c >> 5], bit) & bit);
                }
                const uint64_t b = __ballot(fresh);
                if (fresh) {
                    const uint32_t pos = __popcll(b & lane_lt);
                    new_id[pos] = c;
                    if (AHEAD) put_desc(pos, a.C.desc[c], a.C.dnorm[c]);
                }
                if (lane == 0) { ctl[CTL_NNEW] = __popcll(b); ctl[CTL_PARENT] = 0; }
            }
            __syncthreads();
        } else {
            // documents of the query's entities first, entry points only if those do not
            // fill the pool (query.cu:1577-1604); at most cands + degree seeds
            if (wave == 0) {
                const uint32_t seed_cap = cands + a.degree;
                uint32_t n_seed = 0;
                const uint32_t qe0 = uniform(a.cold->q2e_off[q]), qe1 = uniform(a.cold->q2e_off[q + 1]);
                for (uint32_t i = qe0; i < qe1; i++) {
                    const uint32_t e = uniform(a.cold->q2e_idx[i]);
                    if (e >= a.n_entities) continue;
                    const uint32_t d0 = uniform(a.e2d_off[e]), d1 = uniform(a.e2d_off[e + 1]);
                    for (uint32_t b0 = d0; b0 < d1; b0 += WAVE) {
                        const uint32_t doc = b0 + lane < d1 ? a.e2d_idx[b0 + lane] : EMPTY;
                        bool fresh = false;
                        if (doc < a.C.n) {
                            const uint32_t bit = 1u << (doc & 31);
                            fresh = !(atomicOr(&bitmap[doc >> 5], bit) & bit);
                        }
                        const uint64_t b = __ballot(fresh);
                        const uint32_t pos = n_seed + __popcll(b & lane_lt);
                        if (fresh && pos < seed_cap) { seed_id[pos] = doc; seed_ent[pos] = e; }
                        n_seed = min(seed_cap, n_seed + (uint32_t)__popcll(b));
                    }
                }
                if (n_seed < cands) {
                    const uint32_t c = lane < (int)a.cold->n_entry ? a.cold->entry[lane] : EMPTY;
                    bool fresh = false;
                    if (c < a.C.n) {
                        const uint32_t bit = 1u << (c & 31);
                        fresh = !(atomicOr(&bitmap[c >> 5], bit) & bit);
                    }
                    const uint64_t b = __ballot(fresh);
                    const uint32_t pos = n_seed + __popcll(b & lane_lt);
                    if (fresh && pos < seed_cap) { seed_id[pos] = c; seed_ent[pos] = EMPTY; }
                    n_seed = min(seed_cap, n_seed + (uint32_t)__popcll(b));
                }
                if (lane == 0) ctl[CTL_NSEED] = n_seed;
            }
            __syncthreads();
            const uint32_t n_seed = uniform(ctl[CTL_NSEED]);
            const uint32_t n_ovf_seed = uniform(ctl[CTL_NOVF]);
            for (uint32_t j = wave; j < n_seed; j += NW) {
                const uint32_t id = uniform(seed_id[j]);
                const float bonus = seed_ent[j] != EMPTY ? a.kg_weight : 0.0f; // query.cu:1637-1638
                RowLoad rl;
                RowInfo ri;
                row_issue<NARROW>(rl, ri, a.C, a.C.desc[id], true, a.paths);
                bool hit = false;
                const float acc = row_probe<NARROW, false>(a.C, rl, ri, T, n_ovf_seed, hit);
                const float ssum = (a.paths & (PATH_SPARSE | PATH_BM25)) ? wave_sum_dpp(acc) : 0.f;
                float dist = 1.0f - ssum - bonus;
                if (a.paths & PATH_DENSE) { // seeds are never dropped by the bound
                    DenseRow row;
                    dense_issue(row, ri.rec);
                    dist = 1.0f - (dense_finish_lds(row, qd, 1.0f) + ssum) - bonus;
                    st_dense++;
                }
                st_eval++;
                if (lane == 0) {
                    ln_s += (a.paths & PATH_SPARSE) ? ri.ns : 0u;
                    ln_b += (a.paths & PATH_BM25) ? ri.nb : 0u;
                    seed_dist[j] = dist;
                }
            }
            __syncthreads();
            if (wave == 0) {
                for (uint32_t b0 = 0; b0 < n_seed; b0 += WAVE) {
                    const uint32_t nb = min((uint32_t)WAVE, n_seed - b0);
                    if (lane < (int)nb) {
                        new_id[lane] = seed_id[b0 + lane];
                        new_dist[lane] = seed_dist[b0 + lane];
                        new_ent[lane] = seed_ent[b0 + lane];
                        new_hop[lane] = 0;
                    }
                    wave_fence();
                    Fresh F;
                    fresh_load<MODE>(F, P, new_id, new_dist, new_ent, new_hop, nb);
                    fresh_rank(F);
                    F.kept &= __ballot(F.rank < cands); // of more seeds than the pool holds most cannot enter, and the merge's time goes with the kept ones
                    sort_merge<MODE>(P, F, R);
                }
                front = pool_front(P, 0);
                if (lane == 0) { ctl[CTL_NNEW] = 0; ctl[CTL_PARENT] = 0; }
            }
            __syncthreads();
        }

        // The next parent is the first unexplored pool entry or a new candidate that goes before it, so it is known BEFORE
        // the merge: wave 0 starts the parent's dependent reads (graph row, visited words and, AHEAD, the descriptors) first and
        // merges while they are under way; AHEAD, the row of the first unexplored entry is requested while the candidates are
        // evaluated. At one query per compute unit the three reads were
        // 2 000 cycles of an iteration after the merge; of them 150 to 280 are left behind it. (Looking one whole expansion ahead,
        // with the visited marks taken back when a candidate overtakes: it is right for 0.55 to 0.64 of the expansions only, and
        // the marks and rows of the others cost long batches 5 %.)
        // One and two waves per query are for long batches: in plain and keyword search a row that is overtaken and the descriptors of visited neighbours are
        // traffic there, and nothing waits for them (10 000 queries, 1 M docs, cands 256 / 512: 1.921e11 -> 1.877e11 bytes and
        // 30.4 -> 30.1 ms / 55.1 -> 54.3 ms without them).
        uint32_t g_c = EMPTY, g_kw = 0; // lane l: neighbour of `front`, later of the parent; (keyword search) word l of the row's tail
        for (uint32_t it = 0; it <= a.max_iter; it++) {
            // ---- evaluate the fresh candidates: one wave per candidate ----
            const uint32_t n_new = uniform(ctl[CTL_NNEW]);
            if (uniform(ctl[CTL_PARENT]) == EMPTY) break;
            // a candidate that provably cannot enter the (full) pool is dropped after its sparse part:
            // it is reported as INF_DIS and falls off the end of the merge like any other loser
            const float thr = a.full_eval ? __builtin_inff() : P.dist[cands - 1];
            const float thr_eff = thr < INF_DIS ? thr : __builtin_inff();
            const float span = sketched ? thr_eff - P.dist[0] : __builtin_inff(); // of the pool
            const uint32_t n_ovf = uniform(ctl[CTL_NOVF]);
            // descriptors and dense norms of this wave's candidates: lane l holds candidate l's
            const bool mine = (uint32_t)lane < n_new && (uint32_t)(lane & (NW - 1)) == (uint32_t)wave;
            uint64_t my_desc = 0;
            float my_dn = 0.f;
            if (mine) {
                if (AHEAD) { // no other wave touches the slot from here to the barrier behind the evaluations
                    const float4 s4 = reinterpret_cast<const float4*>(part)[lane];
                    my_desc = (uint64_t)__float_as_uint(s4.y) << 32 | __float_as_uint(s4.x);
                    my_dn = s4.z;
                } else {
                    const uint32_t cid = new_id[lane];
                    my_desc = a.C.desc[cid];
                    my_dn = a.C.dnorm[cid];
                }
            }
            if (AHEAD && wave == 0 && front.id != EMPTY) {
                GlobalWord* row = graph_row(a, KWD ? front.id & ID_MASK : front.id);
                g_c = lane < (int)a.degree ? row[lane] : EMPTY;
                if (KWD) g_kw = lane < APOE_KW_SLOTS ? row[a.degree + lane] : 0u;
            }
            // Stage 1: the sparse parts of this wave's candidates (wave + k * NW), several rows in flight. No branch on whether a candidate
            // of the batch exists: one that does not is a row of no pairs, so the loads of the whole batch are issued back to back.
            // With codes, an upper bound of the sparse part from the terms and a byte a value instead (3 bytes a pair, not 6, CODE_BATCH rows in
            // flight); decision and sketches go by that bound, and the pairs of the few candidates that stay open come with their dense rows.
            // 10 000 queries on 1 M docs with dense neighbours at cands 80: 21.5 -> 19.5 ms (a coded row takes more vector instructions, 119 against 84 an
            // evaluation on i.i.d. rows, which then bound the batch); three or four rows in flight measure the same, and so do
            // pairs and rows of two open candidates together. Short batches, four and more waves a query, are bound by the chain of one query,
            // which a second read of the open candidates' pairs would lengthen: they read the pairs at once (with codes, dense neighbours: 1 000 queries in half precision on
            // four waves each 2.44 -> 2.51 ms, 64 queries on sixteen 1.07 -> 1.23).
            auto eval_rows = [&](auto nb, auto at) { // at(b): the b-th candidate, n_new or more: there is none
                constexpr int NB = decltype(nb)::value;
                RowLoad rl[NB];
                RowInfo ri[NB];
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const uint32_t jj = at(b);
                    row_issue<NARROW>(rl[b], ri[b], a.C, readlane64(my_desc, jj & (WAVE - 1)), jj < n_new, a.paths);
                }
                float acc[NB];
                bool hit[NB];
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    hit[b] = false;
                    acc[b] = row_probe<NARROW, KWD>(a.C, rl[b], ri[b], T, n_ovf, hit[b]);
                }
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const uint32_t jj = at(b);
                    const float rs = row_sum_dpp(acc[b]);
                    if (jj < n_new) {
                        if ((lane & 15) == 0) part[jj * 4 + (lane >> 4)] = rs;
                        if (KWD) {
                            const bool kw_hit = __ballot(hit[b]) != 0;
                            if (lane == 0) new_ent[jj] = kw_hit ? 1u : 0u;
                        }
                    }
                }
            };
            auto code_rows = [&](uint32_t j) {
                CodeLoad rl[CODE_BATCH];
#pragma unroll
                for (int b = 0; b < CODE_BATCH; b++) {
                    const uint32_t jj = j + b * NW;
                    code_issue(rl[b], a.C, readlane64(my_desc, jj & (WAVE - 1)), jj < n_new, a.paths);
                }
                float acc[CODE_BATCH];
                bool hit[CODE_BATCH];
#pragma unroll
                for (int b = 0; b < CODE_BATCH; b++) {
                    hit[b] = false;
                    acc[b] = code_probe<KWD>(a.C, rl[b], [&]() { return readlane64(my_desc, (j + b * NW) & (WAVE - 1)); }, a.paths, T, n_ovf, hit[b]);
                }
#pragma unroll
                for (int b = 0; b < CODE_BATCH; b++) {
                    const uint32_t jj = j + b * NW;
                    const float rs = row_sum_dpp(acc[b]);
                    if (jj < n_new) {
                        if ((lane & 15) == 0) part[jj * 4 + (lane >> 4)] = rs;
                        if (KWD) {
                            const bool kw_hit = __ballot(hit[b]) != 0;
                            if (lane == 0) new_ent[jj] = kw_hit ? 1u : 0u;
                        }
                    }
                }
            };
            const bool by_codes = CODES && thr_eff < __builtin_inff();
            if (CODES && by_codes) {
                for (uint32_t j = wave; j < n_new; j += NW * CODE_BATCH) code_rows(j);
            } else if (NW >= 4) { // a few rows a wave at most expansions: a row that is not there would cost issue slots of a SIMD that several waves share
                for (uint32_t j = wave; j < n_new; j += NW * EVAL_BATCH) {
                    auto at = [&](int b) { return j + b * NW; };
                    if (j + 2 * NW < n_new) eval_rows(std::integral_constant<int, 3>{}, at);
                    else if (j + NW < n_new) eval_rows(std::integral_constant<int, 2>{}, at);
                    else eval_rows(std::integral_constant<int, 1>{}, at);
                }
            } else {
                for (uint32_t j = wave; j < n_new; j += NW * EVAL_BATCH) eval_rows(std::integral_constant<int, EVAL_BATCH>{}, [&](int b) { return j + b * NW; });
            }
            wave_fence();
            // the decision for all of the wave's candidates at once, lane l for candidate l: a candidate whose
            // sparse part plus the bound of its dense part cannot reach the pool is reported as INF_DIS
            uint64_t need, asked; // bit l: candidate l still needs its dense row; its sketch comes first
            {
                bool undecided = false, wide = false;
                if (mine) {
                    float bonus = 0.f;
                    if (KG) {
                        if (new_ent[lane] != EMPTY) bonus = a.kg_weight / (float)new_hop[lane]; // query.cu:1759-1760
                    }
                    float ssum = 0.f, v = 0.f;
                    const float dub = pv_norm * my_dn; // |<query_d, doc_d>| <= |query_d| * |doc_d|
                    undecided = true;
                    wide = dub > span;
                    if (a.paths & (PATH_SPARSE | PATH_BM25)) {
                        const float4 p4 = reinterpret_cast<const float4*>(part)[lane];
                        ssum = p4.x + p4.y + p4.z + p4.w; // the order wave_sum_dpp adds its four rows in
                        v = ssum;
                        if (!(a.paths & PATH_DENSE)) {
                            v = 1.0f - ssum - bonus;
                            undecided = false;
                        } else {
                            const float lb = 1.0f - (ssum + dub) - bonus;
                            if (lb > thr_eff + 1e-5f * (fabsf(ssum) + dub + fabsf(bonus) + 1.0f)) {
                                v = INF_DIS;
                                undecided = false;
                            }
                        }
                    }
                    new_dist[lane] = v;
                    ln_s += (a.paths & PATH_SPARSE) ? desc_nnz_s(my_desc) : 0u;
                    ln_b += (a.paths & PATH_BM25) ? desc_nnz_b(my_desc) : 0u;
                }
                st_eval += __popcll(__ballot(mine));
                need = __ballot(undecided);
                asked = __ballot(undecided && wide);
            }
            wave_fence();
            // stage 2: the sketches of the survivors, SKETCH_BATCH in flight, then the same decision with the tighter bound
            // Asked are candidates whose dense part can move the distance by more than the pool spans: of those few enter the pool
            // (about span / bound of them), and a sketch that rejects saves three quarters of a row. Where the pairs decide, most
            // undecided candidates do enter, and the sketch would be a second wait for a row that is read anyway. Both sides, 10 000
            // queries on 1 M docs: dense rows with neighbours under (49, 1, 1), cands 80 (11 % of the evaluations enter): 4.1 KB of
            // dense part per evaluation -> 1.7 KB, 35.7 -> 21.6 ms; i.i.d. corpus under (1, 1, 1), cands 256 (13 % are undecided, 11 %
            // enter): asking always took 42.3 ms, this rule, which asks almost none, 39.0, no sketches 39.3.
            if (asked) {
                SketchMeta sm = {0.f, 0.f}; // of candidate l
                if ((asked >> lane) & 1) sm = a.sketch_meta[new_id[lane]];
                const uint4 u = reinterpret_cast<const uint4*>(codes)[lane];
                for (uint64_t left = asked; left;) {
                    uint4 c[SKETCH_BATCH] = {}; // set on every path: values left open would live, and spill, across the whole walk
                    uint32_t jj[SKETCH_BATCH];
#pragma unroll
                    for (int b = 0; b < SKETCH_BATCH; b++) {
                        jj[b] = EMPTY;
                        if (left) {
                            jj[b] = __builtin_ctzll(left);
                            left &= left - 1;
                            c[b] = a.sketch[(size_t)uniform(new_id[jj[b]]) * (SKETCH_BYTES / 16) + lane];
                        }
                    }
#pragma unroll
                    for (int b = 0; b < SKETCH_BATCH; b++) {
                        if (jj[b] != EMPTY) {
                            const float dot = sketch_dot(c[b], u);
                            if (lane == 0) part[jj[b] * 4] = dot;
                        }
                    }
                }
                st_sketch += __popcll(asked);
                wave_fence();
                bool far = false;
                if ((asked >> lane) & 1) {
                    float bonus = 0.f;
                    if (KG) {
                        if (new_ent[lane] != EMPTY) bonus = a.kg_weight / (float)new_hop[lane];
                    }
                    const float ssum = new_dist[lane], dub = pv_norm * my_dn;
                    float most = part[lane * 4] * (qs[0] * sm.scale) + pv_norm * sm.err + qs[1] * (my_dn + sm.err);
                    if (HALF) most += pv_norm * (4.9e-4f * my_dn + 1.1e-6f); // the walk's rows are rounded to half precision
                    const float lb = 1.0f - (ssum + most) - bonus;
                    far = lb > thr_eff + 1e-5f * (fabsf(ssum) + dub + fabsf(bonus) + 1.0f);
                    if (far) new_dist[lane] = INF_DIS;
                }
                need &= ~__ballot(far);
                wave_fence();
            }
            if (CODES && by_codes && mine && !((need >> lane) & 1))
                ln_coded += ((a.paths & PATH_SPARSE) ? desc_nnz_s(my_desc) : 0u) + ((a.paths & PATH_BM25) ? desc_nnz_b(my_desc) : 0u);
            // stage 3: the dense rows of the survivors, DENSE_BATCH rows in flight (two of the half-precision rows); behind codes the pairs with them
            st_dense += __popcll(need);
            while (HALF && !CODES && need) {
                DenseRowHalf row[2];
                uint32_t jj[2];
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    jj[b] = EMPTY;
                    if (need) {
                        jj[b] = __builtin_ctzll(need);
                        need &= need - 1;
                        dense_issue_half(row[b], a.half + (size_t)uniform(new_id[jj[b]]) * DIM);
                    }
                }
#pragma unroll
                for (int b = 0; b < 2; b++) {
                    if (jj[b] != EMPTY) {
                        const float dsum = dense_finish_lds_half(row[b], qd, 1.0f);
                        if (lane == 0) new_dist[jj[b]] = 1.0f - (dsum + new_dist[jj[b]]) - 0.f;
                    }
                }
            }
            while (!HALF && !CODES && need) {
                DenseRow row[DENSE_BATCH];
                uint32_t jj[DENSE_BATCH];
#pragma unroll
                for (int b = 0; b < DENSE_BATCH; b++) {
                    jj[b] = EMPTY;
                    if (need) {
                        jj[b] = __builtin_ctzll(need);
                        need &= need - 1;
                        dense_issue(row[b], a.C.recs + desc_off(readlane64(my_desc, jj[b])) * 16);
                    }
                }
#pragma unroll
                for (int b = 0; b < DENSE_BATCH; b++) {
                    if (jj[b] != EMPTY) {
                        float bonus = 0.f;
                        if (KG) {
                            if (new_ent[jj[b]] != EMPTY) bonus = a.kg_weight / (float)new_hop[jj[b]];
                        }
                        const float dsum = dense_finish_lds(row[b], qd, 1.0f);
                        if (lane == 0) new_dist[jj[b]] = 1.0f - (dsum + new_dist[jj[b]]) - bonus;
                    }
                }
            }
            constexpr int ROWS = HALF ? 2 : DENSE_BATCH;
            while (CODES && need) {
                std::conditional_t<HALF, DenseRowHalf, DenseRow> row[ROWS] = {}; // set on every path, as the sketches
                RowLoad rl[ROWS] = {};
                RowInfo ri[ROWS] = {};
                uint32_t jj[ROWS];
#pragma unroll
                for (int b = 0; b < ROWS; b++) {
                    jj[b] = EMPTY;
                    if (need) {
                        jj[b] = __builtin_ctzll(need);
                        need &= need - 1;
                        const uint64_t desc = readlane64(my_desc, jj[b]);
                        if (by_codes) {
                            row_issue<NARROW>(rl[b], ri[b], a.C, desc, true, a.paths);
                            st_reread += (uint32_t)ri[b].n;
                        }
                        if constexpr (HALF) dense_issue_half(row[b], a.half + (size_t)uniform(new_id[jj[b]]) * DIM);
                        else dense_issue(row[b], a.C.recs + desc_off(desc) * 16);
                    }
                }
#pragma unroll
                for (int b = 0; b < ROWS; b++) {
                    if (jj[b] != EMPTY) {
                        float bonus = 0.f;
                        if (KG) {
                            if (new_ent[jj[b]] != EMPTY) bonus = a.kg_weight / (float)new_hop[jj[b]];
                        }
                        float ssum, dsum;
                        if (by_codes) {
                            bool hit = false; // known from the codes already
                            ssum = wave_sum_dpp(row_probe<NARROW, KWD>(a.C, rl[b], ri[b], T, n_ovf, hit));
                        } else ssum = new_dist[jj[b]];
                        if constexpr (HALF) dsum = dense_finish_lds_half(row[b], qd, 1.0f);
                        else dsum = dense_finish_lds(row[b], qd, 1.0f);
                        if (lane == 0) new_dist[jj[b]] = 1.0f - (dsum + ssum) - bonus;
                    }
                }
            }
            __syncthreads();
            // ---- wave 0: merge, pick the next parent, fetch its neighbours ----
            if (wave == 0) {
                Fresh F;
                fresh_load<MODE>(F, P, new_id, new_dist, new_ent, new_hop, n_new);
                uint32_t parent = EMPTY, n_next = 0;
                bool overtaken = false; // the parent is a new candidate (on equal distance the new one goes first)
                if (it < a.max_iter) {
                    parent = front.id;
                    if (F.kept) {
                        const uint32_t l = fresh_first(F);
                        if (parent == EMPTY || readlane_f32(F.d, l) <= front.dist) {
                            overtaken = true;
                            parent = (uint32_t)__builtin_amdgcn_readlane((int)F.id, l);
                        }
                    }
                    if (KWD && parent != EMPTY) parent &= ID_MASK;
                }
                if (parent != EMPTY && (overtaken || !AHEAD)) {
                    GlobalWord* row = graph_row(a, parent);
                    g_c = lane < (int)a.degree ? row[lane] : EMPTY;
                    if (KWD) g_kw = lane < APOE_KW_SLOTS ? row[a.degree + lane] : 0u;
                }
                fresh_rank(F);
                bool fresh = false;
                uint64_t g_desc = 0;
                float g_dn = 0.f;
                if (parent != EMPTY && g_c < a.C.n) {
                    const uint32_t bit = 1u << (g_c & 31);
                    fresh = !(atomicOr(&bitmap[g_c >> 5], bit) & bit);
                    if (AHEAD) {
                        g_desc = a.C.desc[g_c];
                        g_dn = a.C.dnorm[g_c];
                    }
                }
                const uint32_t lowest = sort_merge<MODE>(P, F, R);
                if (parent != EMPTY) {
                    const uint32_t slot = overtaken ? lowest : front.slot; // nothing new goes before an entry that was not overtaken
                    uint32_t p_ent = EMPTY, p_hop = 0;
                    if (KG) { p_ent = P.ent[slot]; p_hop = P.hop[slot]; }
                    if (lane == 0) P.id[slot] |= FLAG;
                    wave_fence();
                    front = pool_front(P, slot + 1);
                    st_exp++;
                    uint32_t c = g_c;
                    bool alive = fresh;
                    uint32_t ent = EMPTY;
                    if (KWD) {
                        // slots whose graph neighbour was already visited (or invalid) are recycled with
                        // the parent's keyword edges: the t-th such slot takes keyword edge t
                        // (query.cu:1397-1409; which slot gets which edge does not matter)
                        const bool dup = lane < (int)a.degree && !fresh;
                        const uint32_t t = __popcll(__ballot(dup) & lane_lt);
                        const uint32_t n_kw = min(uniform(g_kw), (uint32_t)APOE_KW_SLOTS - 1u);
                        const uint32_t c2 = __shfl(g_kw, (int)min(t + 1u, (uint32_t)APOE_KW_SLOTS - 1u), WAVE);
                        if (dup && t < n_kw) {
                            if (c2 < a.C.n) {
                                const uint32_t bit = 1u << (c2 & 31);
                                if (!(atomicOr(&bitmap[c2 >> 5], bit) & bit)) { c = c2; alive = true; }
                            }
                        }
                    }
                    if (KG) {
                        // logical edges: parent's entity -> neighbour entity -> document
                        if (p_hop < 3 && p_ent < a.n_entities) {
                            uint32_t* slot_id = seed_id; // scratch, free after seeding
                            uint32_t* prop = seed_ent;
                            const uint32_t e0 = uniform(a.e2e_off[p_ent]), e1 = uniform(a.e2e_off[p_ent + 1]);
                            slot_id[lane] = fresh ? c : EMPTY;
                            link[lane] = EMPTY;
                            wave_fence();
                            // (i) a fresh graph neighbour that is also a logical neighbour is
                            //     tagged with the first linking entity (query.cu:1699-1715)
                            for (uint32_t jb = e0; jb < e1; jb += WAVE) {
                                const uint32_t j = jb + lane;
                                if (j < e1) {
                                    const uint32_t e2 = a.e2e_idx[j];
                                    if (e2 < a.n_entities) {
                                        for (uint32_t k = a.e2d_off[e2]; k < a.e2d_off[e2 + 1]; k++) {
                                            const uint32_t doc = a.e2d_idx[k];
                                            for (uint32_t t = 0; t < a.degree; t++)
                                                if (slot_id[t] == doc) atomicMin(&link[t], j - e0);
                                        }
                                    }
                                }
                            }
                            wave_fence();
                            if (fresh && link[lane] != EMPTY) ent = a.e2e_idx[e0 + link[lane]];
                            // (ii) slots whose graph neighbour was already visited (or invalid) are
                            //      recycled: the t-th such slot takes the first unvisited document
                            //      of the t-th neighbour entity (query.cu:1718-1735). A document
                            //      claimed by several slots in one round goes to the lowest slot;
                            //      the others move on to their next document.
                            const bool recyc = lane < (int)a.degree && !fresh;
                            const uint64_t rb = __ballot(recyc);
                            const uint32_t t = __popcll(rb & lane_lt);
                            bool unresolved = recyc && t < e1 - e0;
                            uint32_t e2 = EMPTY, k = 0, k1 = 0;
                            if (unresolved) {
                                e2 = a.e2e_idx[e0 + t];
                                if (e2 < a.n_entities) { k = a.e2d_off[e2]; k1 = a.e2d_off[e2 + 1]; }
                                else unresolved = false;
                            }
                            while (__any(unresolved)) {
                                uint32_t doc = EMPTY;
                                if (unresolved) {
                                    while (k < k1) {
                                        const uint32_t x = a.e2d_idx[k];
                                        if (x != parent && x < a.C.n) {
                                            const uint32_t word = __hip_atomic_load(&bitmap[x >> 5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                                            if (!(word & (1u << (x & 31)))) { doc = x; break; }
                                        }
                                        k++;
                                    }
                                    if (doc == EMPTY) unresolved = false;
                                }
                                prop[lane] = doc;
                                wave_fence();
                                if (unresolved) {
                                    bool lose = false;
                                    for (int l = 0; l < lane; l++) lose |= prop[l] == doc;
                                    if (lose) k++;
                                    else {
                                        atomicOr(&bitmap[doc >> 5], 1u << (doc & 31));
                                        c = doc;
                                        ent = e2;
                                        alive = true;
                                        unresolved = false;
                                    }
                                }
                                wave_fence();
                                __threadfence();
                            }
                        }
                    }
                    const uint64_t b = __ballot(alive);
                    if (alive) {
                        const uint32_t pos = __popcll(b & lane_lt);
                        new_id[pos] = c;
                        if (AHEAD && (KG || KWD) && !fresh) { // not a graph neighbour: recycled through a keyword or logical edge
                            g_desc = a.C.desc[c];
                            g_dn = a.C.dnorm[c];
                        }
                        if (AHEAD) put_desc(pos, g_desc, g_dn);
                        if (KG) { new_ent[pos] = ent; new_hop[pos] = p_hop + 1; }
                    }
                    n_next = __popcll(b);
                }
                if (lane == 0) { ctl[CTL_PARENT] = parent; ctl[CTL_NNEW] = n_next; }
            }
            __syncthreads();
        }
        // ---- half-precision walk: every pool entry again with its fp32 row, then the pool in order again ----
        if (HALF) {
            __syncthreads();
            const uint32_t n_ovf = uniform(ctl[CTL_NOVF]);
            for (uint32_t e = wave; e < cands; e += NW) {
                const uint32_t id = uniform(P.id[e]) & ~FLAG;
                if (id >= a.C.n) continue; // empty slot
                RowLoad rl;
                RowInfo ri;
                row_issue<NARROW>(rl, ri, a.C, a.C.desc[id], true, a.paths);
                bool hit = false;
                const float acc = row_probe<NARROW, false>(a.C, rl, ri, T, n_ovf, hit);
                const float ssum = (a.paths & (PATH_SPARSE | PATH_BM25)) ? wave_sum_dpp(acc) : 0.f;
                // the same expressions as in the walk, so an entry gets the bits the default search gives it
                float dist = 1.0f - ssum - 0.f;
                if (a.paths & PATH_DENSE) {
                    DenseRow row;
                    dense_issue(row, ri.rec);
                    dist = 1.0f - (dense_finish_lds(row, qd, 1.0f) + ssum) - 0.f;
                }
                if (lane == 0) P.dist[e] = dist;
                st_again++;
                st_again_pairs += ri.n;
            }
            __syncthreads();
            if (wave == 0) {
                // nearly sorted already: odd-even transposition until a double pass moves nothing (stable)
                bool moved = true;
                while (moved) {
                    moved = false;
                    for (uint32_t phase = 0; phase < 2; phase++) {
                        bool sw = false;
                        for (uint32_t i = phase + 2 * lane; i + 1 < cands; i += 2 * WAVE) {
                            const float d0 = P.dist[i], d1 = P.dist[i + 1];
                            if (d1 < d0) {
                                const uint32_t i0 = P.id[i], i1 = P.id[i + 1];
                                P.dist[i] = d1;
                                P.dist[i + 1] = d0;
                                P.id[i] = i1;
                                P.id[i + 1] = i0;
                                sw = true;
                            }
                        }
                        wave_fence();
                        moved |= __any(sw) != 0;
                    }
                }
            }
            __syncthreads();
        }
        // ---- results (query.cu:566-569) ----
        if (!KWD) {
            for (uint32_t i = tid; i < cands; i += NW * WAVE) {
                a.cold->out_ids[(size_t)qi * cands + i] = P.id[i] & ~FLAG;
                a.cold->out_dist[(size_t)qi * cands + i] = P.dist[i];
            }
        } else if (wave == 0) {
            // pool entries that hold a required keyword, in pool order, then the evicted hits by
            // (distance, id); the rest of the row is empty (query.cu:1464-1481)
            uint32_t* oid = a.cold->out_ids + (size_t)qi * cands;
            float* od = a.cold->out_dist + (size_t)qi * cands;
            uint32_t kn = 0;
            for (uint32_t base = 0; base < cands; base += WAVE) {
                const uint32_t id = base + lane < cands ? P.id[base + lane] : EMPTY;
                const bool hit = id != EMPTY && (id & KW_HIT);
                const uint64_t hb = __ballot(hit);
                if (hit) {
                    const uint32_t pos = kn + __popcll(hb & lane_lt);
                    oid[pos] = id & ID_MASK;
                    od[pos] = P.dist[base + lane];
                }
                kn += __popcll(hb);
            }
            const uint32_t m = min(R.n, (uint32_t)RING);
            if ((uint32_t)lane < m) {
                const float d = R.dist[lane];
                const uint32_t id = R.id[lane];
                uint32_t rank = 0;
                for (uint32_t i = 0; i < m; i++) {
                    const float di = R.dist[i];
                    const uint32_t ii = R.id[i];
                    rank += (di < d) || (di == d && ii < id);
                }
                if (kn + rank < cands) { oid[kn + rank] = id; od[kn + rank] = d; }
            }
            for (uint32_t i = kn + m + lane; i < cands; i += WAVE) { oid[i] = EMPTY & ~FLAG; od[i] = INF_DIS; }
        }
        uint32_t st_ns = ln_s, st_nb = ln_b;
#pragma unroll
        for (int o = WAVE / 2; o > 0; o >>= 1) {
            st_ns += __shfl_xor(st_ns, o, WAVE);
            st_nb += __shfl_xor(st_nb, o, WAVE);
            if (CODES) ln_coded += __shfl_xor(ln_coded, o, WAVE);
        }
        if (lane == 0) { // summed in LDS over the workgroup's queries: seven atomics per query on one memory line would queue up
            if (st_exp) atomicAdd(stat + 1, (unsigned long long)st_exp);
            if (st_eval) atomicAdd(stat + 2, (unsigned long long)st_eval);
            if (st_ns) atomicAdd(stat + 3, (unsigned long long)st_ns);
            if (st_nb) atomicAdd(stat + 4, (unsigned long long)st_nb);
            if (st_dense) atomicAdd(stat + 5, (unsigned long long)st_dense);
            if (st_again) atomicAdd(stat + 6, (unsigned long long)st_again);
            if (st_again_pairs) atomicAdd(stat + 7, (unsigned long long)st_again_pairs);
            if (st_sketch) atomicAdd(stat + 8, (unsigned long long)st_sketch);
            if (CODES) atomicAdd(stat + 9, (unsigned long long)st_reread - ln_coded);
        }
    }
    __syncthreads();
    if (tid >= 1 && tid < STATS && stat[tid]) atomicAdd(a.work + tid, stat[tid]);
}

// Counters and once-per-query arguments of a launch, written on the stream (no host copy from a stack frame,
// no memset node for a caller that records the stream).
__global__ void search_setup_kernel(unsigned long long* work, SearchCold* dst, SearchCold cold) {
    if (threadIdx.x < STATS) work[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) *dst = cold;
}

// Workspace of apoe_search_noalloc: counters, once-per-query arguments and the visited bitmaps of as many workgroups as fit
// APOE_NOALLOC_WS_BYTES; behind them the query codes of as many workgroups as a GPU of 256 CUs holds (32 waves a CU), so that
// the codes take no bitmap's place. One copy per GPU, held until the process ends; every call on a GPU uses it, so calls
// that overlap on one GPU race. Host code never uses the array's name as an address: the device address is
// asked for once per device (search_static_workspace) and kept.
constexpr uint32_t NOALLOC_CODES = 256 * 32;
static __device__ __align__(256) unsigned char search_scratch[APOE_NOALLOC_WS_BYTES + NOALLOC_CODES * SKETCH_BYTES];

constexpr int MAX_DEVICES = 64;
static std::mutex scratch_mutex;
static char* scratch_ptr[MAX_DEVICES]; // per device: address of search_scratch on that GPU, null until asked for

int search_static_workspace(int device, char** out) {
    APOE_REQUIRE(device >= 0 && device < MAX_DEVICES, "device %d outside [0,%d)", device, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[device]) {
        APOE_HIP(hipSetDevice(device));
        void* p = nullptr;
        APOE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(search_scratch)));
        APOE_REQUIRE(p != nullptr, "no device address for the static search workspace on device %d", device);
        scratch_ptr[device] = static_cast<char*>(p);
    }
    *out = scratch_ptr[device];
    return APOE_OK;
}

template <int NW, int MODE, bool NARROW, bool HALF = false, bool CODES = false>
static int launch_format(apoe_ctx* ctx, const SearchArgs& a, uint32_t grid, size_t lds, int* per_cu) {
    if constexpr (MODE == MODE_PLAIN && !HALF && !CODES) {
        if (a.half) return launch_format<NW, MODE, NARROW, true>(ctx, a, grid, lds, per_cu);
    }
    if constexpr (NARROW && NW <= 2 && !CODES) {
        if (a.coded) return launch_format<NW, MODE, NARROW, HALF, true>(ctx, a, grid, lds, per_cu);
    }
    const void* fn = reinterpret_cast<const void*>(&search_kernel<NW, MODE, NARROW, HALF, CODES>);
    APOE_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    if (per_cu) { // occupancy query only
        APOE_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, fn, NW * WAVE, lds));
        return APOE_OK;
    }
    search_kernel<NW, MODE, NARROW, HALF, CODES><<<grid, NW * WAVE, lds, ctx->stream>>>(a);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

template <int NW, int MODE>
static int launch_variant(apoe_ctx* ctx, const SearchArgs& a, uint32_t grid, size_t lds, int* per_cu) {
    return a.C.narrow ? launch_format<NW, MODE, true>(ctx, a, grid, lds, per_cu) : launch_format<NW, MODE, false>(ctx, a, grid, lds, per_cu);
}

template <int MODE>
static int launch_shape(apoe_ctx* ctx, int nw, const SearchArgs& a, uint32_t grid, size_t lds, int* per_cu) {
    switch (nw) {
        case 1: return launch_variant<1, MODE>(ctx, a, grid, lds, per_cu);
        case 4: return launch_variant<4, MODE>(ctx, a, grid, lds, per_cu);
        case 8: return launch_variant<8, MODE>(ctx, a, grid, lds, per_cu);
        case 16: return launch_variant<16, MODE>(ctx, a, grid, lds, per_cu);
        default: return launch_variant<2, MODE>(ctx, a, grid, lds, per_cu);
    }
}

static int launch_mode(apoe_ctx* ctx, int mode, int nw, const SearchArgs& a, uint32_t grid, size_t lds, int* per_cu) {
    switch (mode) {
        case MODE_KG: return launch_shape<MODE_KG>(ctx, nw, a, grid, lds, per_cu);
        case MODE_KEYWORD: return launch_shape<MODE_KEYWORD>(ctx, nw, a, grid, lds, per_cu);
        default: return launch_shape<MODE_PLAIN>(ctx, nw, a, grid, lds, per_cu);
    }
}

// static_ws: null, or the device address of this GPU's search_scratch: then nothing is allocated, the grid is cut to
// the bitmaps that fit, and a call without `stats` returns with the work still running on the context's stream.
// Whether a search asks the codes. They pay where the dense part decides, so that pairs settle little and memory bounds a long batch; elsewhere pairs settle
// what the looser bound leaves open, and their kernels, which take more vector instructions a row, are the slower ones. What decides is estimated from the
// corpus: the dense part of a score reaches w_dense |q_d| |d_d|, the sparse part at most w |q_s| |d_s| a path, with the documents' mean squared norms (a query's
// dense row is as long as a document's; its pairs are as long as a document's, but fewer). Time without codes / with codes, 10 000 queries on 1 M docs,
// cands 64 ... 256, by the ratio of the two, on lists of near rows and on a built index:
//   plain    i.i.d. 0.014: 0.97-1.05  0.03: 0.98-1.03  0.08: 0.96-1.03  0.17: 1.07-1.12  0.4: 1.10-1.11  1.5: 1.08   dense neighbours 0.09: 0.93-0.96  0.18: 1.00-1.07
//            0.36: 1.10-1.13  2.2: 1.08-1.14
//   half     0.014: 0.90-0.97  0.03: 0.87-0.95  0.08: 0.87-1.02  0.17: 1.01-1.08  1.5: 0.99-1.06;  0.09: 0.88-0.93  0.18: 0.99-1.05  0.36: 1.09-1.11
//   keyword  0.014: 0.91-0.98  0.03: 0.86-0.99  0.08: 0.89-0.97  0.17: 0.96-1.07  1.5: 0.97-1.04;  0.09: 0.93-0.94  0.18: 1.00-1.04  0.36: 1.06-1.08  2.2: 1.07-1.08
// The line lies at an eighth. A linking entity's bonus is a third part: where it exceeds the dense part, the pool holds linked documents, no sketch is asked and the
// pairs of most others are read twice (bonus 40; dense part 8 and 16 with dense neighbours 0.91, 49: 1.07-1.09, 100 on i.i.d. rows 1.03-1.08). Pairs alone never
// ask them (SPLADE, cands 256: 24.5 ms without, 25.8 with). Rows longer than the loads of a batch (192 pairs) read their rest one chunk after the other: 10 000 queries
// on 200 000 docs with dense neighbours, time without / with codes by the pairs of an average row, cands 16 ... 200: plain 180: 1.04-1.11, 240: 1.03-1.06,
// 300-360: 0.99-1.02, 420-480: 0.98-1.01, 660: 0.95; half 180: 1.02-1.03, 240: 0.96-0.98, 300: 0.95-0.97; keyword 180: 0.99-1.02, 240: 0.95-0.97. The lines lie at
// 192 and, for plain searches, 320 pairs. The codes are kernels of their own: with both ways in one, spilled registers cost searches without codes 3 %.
static bool codes_pay(const apoe_corpus* c, const apoe_queries* q, const apoe_search_params* p, uint32_t q_count, uint32_t paths, bool kg, bool plain) {
    if (!(paths & PATH_DENSE) || !(paths & (PATH_SPARSE | PATH_BM25))) return false;
    const uint64_t read = (paths & PATH_SPARSE ? c->pairs_s : 0) + (paths & PATH_BM25 ? c->total_pairs - c->pairs_s : 0);
    if (read > (plain ? 320ull : 3ull * WAVE) * c->n) return false;
    auto part = [&](float w, double mean_sq, uint64_t pairs, uint64_t q_pairs) { // of a path with that many pairs in all documents and in the batch
        return pairs ? fabs((double)w) * mean_sq * sqrt((double)q_pairs / q_count / ((double)pairs / c->n)) : 0.0;
    };
    const uint32_t q0 = p->q_begin, q1 = q0 + q_count;
    const double dense = (double)p->w_dense * c->mean_sq[0];
    const double sparse = (paths & PATH_SPARSE ? part(p->w_sparse, c->mean_sq[1], c->pairs_s, q->h_s_off[q1] - q->h_s_off[q0]) : 0.0) +
                          (paths & PATH_BM25 ? part(p->w_bm25, c->mean_sq[2], c->total_pairs - c->pairs_s, q->h_b_off[q1] - q->h_b_off[q0]) : 0.0);
    return dense >= sparse / 8 && (!kg || dense >= p->kg_weight);
}

int launch_search(apoe_ctx* ctx, const apoe_corpus* c, const apoe_queries* q, const apoe_graph* g, const apoe_kg* kg,
                  const apoe_search_params* p, uint32_t* out_ids_dev, float* out_dist_dev, apoe_search_stats* stats, char* static_ws) {
    APOE_REQUIRE(p->cands >= 1 && p->cands <= APOE_MAX_CANDS, "cands must be in 1..%d, got %u", APOE_MAX_CANDS, p->cands);
    APOE_REQUIRE(g->width > APOE_KW_SLOTS && g->width - APOE_KW_SLOTS <= MAX_NEW, "graph degree must be in 1..64, got width %u", g->width);
    APOE_REQUIRE(g->n == c->n, "graph has %u nodes but the corpus has %u documents", g->n, c->n);
    APOE_REQUIRE(p->q_begin <= q->n, "q_begin %u beyond %u queries", p->q_begin, q->n);
    const uint32_t q_count = p->q_count ? p->q_count : q->n - p->q_begin;
    APOE_REQUIRE(q_count <= q->n - p->q_begin, "query range of %u from %u beyond %u queries", q_count, p->q_begin, q->n);
    if (stats) *stats = apoe_search_stats{};
    if (q_count == 0) return APOE_OK;

    SearchArgs a{};
    SearchCold cold{};
    a.C = c->view();
    cold.Q = q->view();
    a.graph = g->rows.p;
    a.W = g->width;
    a.degree = g->width - APOE_KW_SLOTS;
    cold.entry = g->entry.p;
    cold.n_entry = std::min<uint32_t>(g->n_entry, MAX_NEW);
    cold.w_d = p->w_dense;
    cold.w_s = p->w_sparse;
    cold.w_b = p->w_bm25;
    a.paths = (!(p->w_dense < 1e-5f) ? PATH_DENSE : 0) | (!(p->w_sparse < 1e-5f) ? PATH_SPARSE : 0) | (!(p->w_bm25 < 1e-5f) ? PATH_BM25 : 0);
    a.cands = p->cands;
    a.max_iter = p->max_iter ? p->max_iter : 1000;
    cold.q_begin = p->q_begin;
    a.q_count = q_count;
    cold.out_ids = out_ids_dev;
    cold.out_dist = out_dist_dev;
    a.slots_s = next_pow2(std::max(16u, 2 * q->max_nnz_s));
    a.slots_b = next_pow2(std::max(16u, 2 * q->max_nnz_b));
    a.ovf_cap = (q->max_nnz + 7u) & ~7u;
    a.kg_weight = p->kg_weight;
    a.full_eval = (p->variant & 0x100u) ? 1u : 0u;
    a.half = nullptr;
    a.sketch_meta = c->sketch_meta.p;
    a.sketch = reinterpret_cast<const uint4*>(c->sketch.p);
    if (p->variant & 0x200u) {
        APOE_REQUIRE(c->half.p != nullptr, "variant 0x200 needs the half-precision rows: call apoe_corpus_make_half_rows first");
        APOE_REQUIRE(kg == nullptr && !p->keyword_filter, "variant 0x200 (half-precision rows) is for the plain search only");
        a.half = c->half.p;
    }

    const bool use_kg = kg != nullptr;
    const bool use_kw = p->keyword_filter != 0;
    APOE_REQUIRE(!(use_kg && use_kw), "keyword-filter search cannot be combined with a knowledge graph");
    const int mode = use_kg ? MODE_KG : use_kw ? MODE_KEYWORD : MODE_PLAIN;
    if (use_kw) {
        APOE_REQUIRE(c->n < (1u << 30), "keyword-filter search keeps two flag bits on a document id: %u documents are too many", c->n);
        a.paths = PATH_DENSE | PATH_SPARSE | PATH_BM25; // query.cu:2005-2007: always the three-path loop
    }
    a.coded = c->coded && !a.full_eval && codes_pay(c, q, p, q_count, a.paths, use_kg, mode == MODE_PLAIN && !a.half) ? 1u : 0u;
    if (use_kg) {
        APOE_REQUIRE(kg->n_queries >= p->q_begin + q_count, "knowledge graph holds entities for %u queries, %u needed", kg->n_queries, p->q_begin + q_count);
        a.e2e_off = kg->e2e_off.p;
        a.e2e_idx = kg->e2e_idx.p;
        a.e2d_off = kg->e2d_off.p;
        a.e2d_idx = kg->e2d_idx.p;
        cold.q2e_off = kg->q2e_off.p;
        cold.q2e_idx = kg->q2e_idx.p;
        a.n_entities = kg->n_entities;
    }
    const SearchLds L(a.slots_s, a.slots_b, a.ovf_cap, a.cands, mode);
    // 64 KB; the fixed arrays were 224 bytes longer when that line was drawn, and the query rows that are served do not depend on their length
    APOE_REQUIRE(L.total <= 64 * 1024 - 224, "search needs %u bytes of LDS (query rows with up to %u sparse terms)", L.total, q->max_nnz);

    a.bitmap_words = ((c->n + 31) / 32 + 3) & ~3u;
    // workspace: [counters: 16 x u64][once-per-query arguments][visited bitmaps][codes of the queries' dense rows]
    const size_t cold_at = 16 * sizeof(unsigned long long), bitmaps_at = (cold_at + sizeof(SearchCold) + 255) & ~(size_t)255;
    const size_t bitmap_bytes = (size_t)a.bitmap_words * sizeof(uint32_t);
    size_t fit = SIZE_MAX; // workgroups whose visited bitmaps fit the workspace
    if (static_ws) {
        fit = std::min<size_t>((APOE_NOALLOC_WS_BYTES - bitmaps_at) / bitmap_bytes, NOALLOC_CODES);
        APOE_REQUIRE(fit >= 1, "the static workspace of %u bytes holds no visited bitmap of %zu bytes", (unsigned)APOE_NOALLOC_WS_BYTES, bitmap_bytes);
    }

    // Launch shape (waves per query). 1, 2, 3, 4, 5: one, four, eight, two, sixteen waves, as the caller says. 0, the default:
    //  * a batch that is resident all at once is bound by the time of ONE query, and that falls with the waves it has
    //    (128 queries, 1 M docs, cands 256: 4.5 / 3.0 / 2.2 ms with 4 / 8 / 16 waves): sixteen waves while every query has a
    //    CU of its own (256 queries: 2.30 ms against 3.10 with eight; 300: 3.38 against 3.10), eight while all queries still fit
    //    the machine that way (768 at 3 per CU: 3.74 against 5.09 with four; 1 024: 5.28 against 5.18), else four while they fit
    //    (1 536: 6.0 against 8.9 with two); four also for batches of up to two rounds of the two-wave grid (6 144 queries),
    //    whose second round ends sooner that way (4 096: 13.6 against 15.4 ms, 6 144: 21.1 against 22.6, at cands 64 7.0 against 7.6);
    //  * a longer batch is bound by the memory system and runs best with two waves per query and as many queries as fit
    //    (12 per CU) - unless the pool is so large that LDS leaves room for at most 9 queries on a CU: then four waves
    //    per query keep twice the loads in flight (10 000 queries, 1 M docs, four against two waves: 98.0 against 105.6 ms
    //    at cands 1024, where 9 queries fit, 185.6 against 248.7 at 2048; knowledge-graph search: 32.8 against 34.6 ms at
    //    cands 256, where 9 fit, 25.9 against 25.5 at 192, where 10 fit, 129.7 against 184.5 at 1024; the keyword search
    //    measures the same or worse with four up to cands 768 and stays at two). Plain searches where 10 to 12 queries fit
    //    measure 1 to 7 % less with four waves as well; the line is one for both modes.
    int nw = 2;
    const uint32_t shape = p->variant & 0xFFu;
    if (shape == 1) nw = 1;
    else if (shape == 2) nw = 4;
    else if (shape == 3) nw = 8;
    else if (shape == 5) nw = 16;
    else APOE_REQUIRE(shape == 0 || shape == 4, "launch shape %u is not one of 0 (default), 1, 2, 3, 4, 5 (one, four, eight, two, sixteen waves per query)", shape);
    auto resident_per_cu = [&](int waves, int* out) -> int {
        *out = 1;
        APOE_TRY(launch_mode(ctx, mode, waves, a, 0, L.total, out));
        if (*out < 1) *out = 1;
        return APOE_OK;
    };
    int per_cu = 1;
    if (shape == 0) {
        const size_t at_once = std::min<size_t>(q_count, fit); // queries in flight if every one of them had a workgroup
        int pc16 = 1, pc8 = 1, pc4 = 1;
        APOE_TRY(resident_per_cu(16, &pc16));
        APOE_TRY(resident_per_cu(8, &pc8));
        APOE_TRY(resident_per_cu(4, &pc4));
        APOE_TRY(resident_per_cu(2, &per_cu));
        if (at_once <= (size_t)pc16 * ctx->num_cus) { nw = 16; per_cu = pc16; }
        else if (at_once <= (size_t)pc8 * ctx->num_cus) { nw = 8; per_cu = pc8; }
        else if (at_once <= (size_t)pc4 * ctx->num_cus || at_once <= 2 * (size_t)per_cu * ctx->num_cus) { nw = 4; per_cu = pc4; }
        else if (per_cu <= 9 && mode != MODE_KEYWORD && pc4 * 4 > per_cu * 2) { nw = 4; per_cu = pc4; }
    } else {
        APOE_TRY(resident_per_cu(nw, &per_cu));
    }
    // persistent grid: as many workgroups as can be resident, never more than queries or bitmaps
    const uint32_t grid = (uint32_t)std::min<size_t>(std::min<size_t>(q_count, fit), (size_t)per_cu * (size_t)ctx->num_cus);
    char* ws = static_ws;
    if (!static_ws) APOE_TRY(ctx->search_workspace(bitmaps_at + (size_t)grid * (bitmap_bytes + SKETCH_BYTES), &ws));
    unsigned long long* work = reinterpret_cast<unsigned long long*>(ws);
    search_setup_kernel<<<1, WAVE, 0, ctx->stream>>>(work, reinterpret_cast<SearchCold*>(ws + cold_at), cold);
    APOE_HIP(hipGetLastError());
    a.cold = reinterpret_cast<const SearchCold*>(ws + cold_at);
    a.bitmaps = reinterpret_cast<uint32_t*>(ws + bitmaps_at);
    a.codes = reinterpret_cast<uint32_t*>(static_ws ? static_ws + APOE_NOALLOC_WS_BYTES : ws + bitmaps_at + (size_t)grid * bitmap_bytes);
    a.work = work;

    if (static_ws && !stats) return launch_mode(ctx, mode, nw, a, grid, L.total, nullptr);
    float ms = 0.f;
    APOE_TRY(timed(ctx, &ms, [&]() { return launch_mode(ctx, mode, nw, a, grid, L.total, nullptr); }));
    APOE_HIP(hipStreamSynchronize(ctx->stream));
    if (stats) {
        unsigned long long h[STATS];
        APOE_HIP(hipMemcpy(h, work, sizeof(h), hipMemcpyDeviceToHost));
        stats->kernel_ms = ms;
        stats->expansions = h[1];
        stats->evaluations = h[2];
        stats->nnz_sparse = h[3];
        stats->nnz_bm25 = h[4];
        stats->dense_rows = h[5];
        // dense rows and sketches actually needed (a sketch with its scale and error) + pairs + descriptor and dense norm (12 B per evaluation)
        uint64_t bytes = h[5] * (uint64_t)(a.half ? DENSE_BYTES / 2 : DENSE_BYTES) + h[8] * (uint64_t)(SKETCH_BYTES + sizeof(SketchMeta));
        bytes += (c->narrow ? 6 : 8) * (h[3] + h[4]) + 12 * h[2];
        bytes += 3 * h[9]; // codes are three bytes a pair with their terms: instead of the pair, or beside it where it was read after all
        bytes += h[6] * (uint64_t)(DENSE_BYTES + 8) + (c->narrow ? 6 : 8) * h[7]; // the pool evaluated again in fp32
        bytes += h[1] * 4ull * a.W;
        uint64_t qbytes = (uint64_t)q_count * DENSE_BYTES + 8 * (q->h_s_off[p->q_begin + q_count] - q->h_s_off[p->q_begin]) +
                          8 * (q->h_b_off[p->q_begin + q_count] - q->h_b_off[p->q_begin]);
        bytes += qbytes + (uint64_t)q_count * a.cands * 8;
        stats->algo_bytes = bytes;
    }
    return APOE_OK;
}

} // namespace apoe
