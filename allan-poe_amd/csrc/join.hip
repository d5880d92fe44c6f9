// NN-Descent step as a local join around the picked neighbour.
//
// The reference's step (index.cu:156-376) lets node u meet the forward list N(v) and the reverse list R(v) of
// each neighbour v it picks: one pivot against many rows, every row gathered for one evaluation. Here the same
// pairs are formed the other way round: all pickers of one v are the ROWS of a tile (32 at a time), N(v) and R(v)
// are its COLUMNS (up to 128), every row of the tile is gathered once and meets every column:
//   dense part   32 x 128 x 1024 contraction on the matrix cores (fp32 MFMA 16x16x4; the waves take the
//                16-column blocks that exist x equal parts of the dimensions)
//   sparse part  eight picker rows at a time in an LDS rank table that the column rows probe (apoe_ranktab.h)
//   insertion    a pair closer than the row's last list entry (and not in that list) is offered to the row node
//                with a 64-bit atomicMin on slot hash(id) of its proposal row: (distance, id), the smallest wins;
//                in symmetric mode the pair is offered to the column node as well (both endpoints, as the classic
//                NN-Descent join does; the reference's step updates u only)
// and a second kernel merges every node's proposals into its sorted list (wave-level rank merge, new before old
// on equal distance, index.cu:333-351) and registers the entries that are new in a list with their nodes' reverse
// lists (slot = registrations so far, modulo K; every registration a 64-bit atomicMin, so beyond K the closer entry
// of a slot stays, index.cu:362-372). Lists are read as the step found them, proposals are minima under a total
// order, and the bits of a distance do not depend on which of a node's pickers share a tile (tile_dense; in the wide pair
// format the last bit may, where two terms of a group sit on one table slot), so the lists a step leaves do not depend on the
// order in which pickers arrive and tiles run. The reverse lists are append-only
// over the steps: a node that later drops v stays in R(v) (a stale column costs one evaluation and can never enter a
// list wrongly: its distance is computed again), and while a list has fewer than K registrations its content does
// not depend on the order either; beyond K, which entries share a slot follows the arrival order of the counter.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <type_traits>

#include "apoe_gram.h"
#include "apoe_internal.h"
#include "apoe_ranktab.h"

namespace apoe {

constexpr int JT_ROWS = 32;
constexpr int JT_COLS = 128;
// A tile is a chain of short phases (queue, ids, pairs and table builds, probes, dense rows, proposals) with barriers between
// them: one phase waits for memory, the next for LDS or the vector units. Two workgroups of eight waves per CU, each with half
// of the CU's LDS and registers, cover each other's waits; at most a hundred columns meet four to eight pickers in an average
// tile, so neither workgroup lacks work. Builds of ten steps against one workgroup of sixteen waves (wide pairs: of eight) with the
// columns' pairs in registers: 100 000 docs K = 64 145.2 -> 113.3 ms, 30 011 docs K = 128 97.3 -> 76.7 ms, 20 000 docs wide 54.5 ->
// 37.4 ms, 300 000 docs of the i.i.d. corpus 299 -> 254 ms. A corpus whose longest row does not fit the table of the smaller LDS takes one
// workgroup of sixteen waves per CU (tile_shape), and so does one whose rows are long (join_shape, gram_tiles_pair).
constexpr int JT_PAIR_THREADS = 512, JT_SOLO_THREADS = 1024;
constexpr int JT_STRIDE = JT_COLS + 1;
constexpr int JT_STAGE_DIMS = 256; // the picker rows are staged at least this many dimensions at a time
constexpr int JT_SEEN = 512; // slots of the id set that removes repeated columns
// The kernels below are built for lists of KK = 64 and KK = 128 entries (index.cu:6 has K 64; a degree above 32 needs
// 2 * degree <= K there, index.cu:702). A node has 2 * KK proposal slots: two proposals of one step whose ids hash to one
// slot are one proposal, the closer one. With KK = 128 the columns of a picked node (its list and its reverse list, up to
// 256) are two tiles: the list, then what the reverse list adds to it.
constexpr int JOIN_PICKS = 4; // index.cu:157,171-181
constexpr int JOIN_COUNT_PARTS = 256, JOIN_COUNT_AT = 8; // partial insertion counters in the step's work array, one per 64-byte line, from word 8

__device__ __forceinline__ uint32_t prop_slot(uint32_t id, uint32_t P) { return (uint32_t)(mix64(id) >> 40) & (P - 1); }

__device__ __forceinline__ float join_key_dist(unsigned long long key) {
    uint32_t u = (uint32_t)(key >> 32);
    u ^= (u >> 31) ? 0x80000000u : 0xFFFFFFFFu;
    return __uint_as_float(u);
}

// One wave per node: the picking rule of the expansion step (group g takes the first unsampled slot >= g; none
// left: slot 0 again), the picked neighbours counted per target.
template <uint32_t KK>
__global__ __launch_bounds__(256) void join_pick_kernel(uint32_t n, uint32_t* ids, uint32_t* picks, uint32_t* pick_cnt) {
    constexpr int KL = KK / WAVE; // list entries per lane: entry e sits in register e / 64 of lane e % 64
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const uint32_t u = blockIdx.x * 4 + wave;
    if (u >= n) return;
    const size_t base = (size_t)u * KK;
    uint32_t own[KL];
    uint64_t m0[KL];
#pragma unroll
    for (int k = 0; k < KL; k++) {
        own[k] = ids[base + k * WAVE + lane];
        m0[k] = __ballot(!(own[k] & FLAG));
    }
    uint32_t slot[JOIN_PICKS], mine = EMPTY; // everything here is wave-uniform except `mine`: lane g keeps the g-th pick
#pragma unroll
    for (int g = 0; g < JOIN_PICKS; g++) {
        uint32_t s = 0;
        bool found = false;
#pragma unroll
        for (int k = 0; k < KL; k++) {
            const uint64_t a = k == 0 ? m0[0] & ~((1ull << g) - 1) : m0[k];
            if (!found && a) {
                s = k * WAVE + __ffsll((unsigned long long)a) - 1;
                m0[k] &= ~(1ull << (s % WAVE));
                if ((uint32_t)lane == s % WAVE) ids[base + s] = own[k] | FLAG;
                found = true;
            }
        }
        slot[g] = s;
        bool dup = false;
#pragma unroll
        for (int t = 0; t < g; t++) dup |= slot[t] == s;
        uint32_t v = 0;
#pragma unroll
        for (int k = 0; k < KL; k++)
            if (s / WAVE == (uint32_t)k) v = (uint32_t)__builtin_amdgcn_readlane((int)own[k], s % WAVE) & ~FLAG;
        if (dup || v >= n) v = EMPTY;
        if (lane == g) mine = v;
    }
    if (lane < JOIN_PICKS) {
        picks[(size_t)u * JOIN_PICKS + lane] = mine;
        if (mine != EMPTY) atomicAdd(&pick_cnt[mine], 1u);
    }
}

__global__ __launch_bounds__(256) void join_tile_count_kernel(uint32_t n, uint32_t halves, const uint32_t* pick_cnt, uint32_t* tile_cnt) {
    const uint32_t v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v < n) tile_cnt[v] = (pick_cnt[v] + JT_ROWS - 1) / JT_ROWS * halves;
    if (v == n) tile_cnt[v] = 0;
}

// The pickers of every v side by side, and the node of every tile.
__global__ __launch_bounds__(256) void join_fill_kernel(uint32_t n, uint32_t halves, const uint32_t* picks, const uint32_t* pick_off, const uint32_t* tile_off,
                                                        uint32_t* pick_fill, uint32_t* pick_src, uint32_t* tile_v) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (uint64_t)n * JOIN_PICKS) return;
    const uint32_t v = picks[t];
    if (v == EMPTY) return;
    const uint32_t k = atomicAdd(&pick_fill[v], 1u);
    pick_src[pick_off[v] + k] = (uint32_t)(t / JOIN_PICKS);
    if (k % JT_ROWS == 0)
        for (uint32_t h = 0; h < halves; h++) tile_v[tile_off[v] + k / JT_ROWS * halves + h] = v;
}

struct JoinArgs {
    CorpusView C;
    float dense_mul;
    uint32_t n, P, symmetric;
    const uint32_t* ids;
    const float* dist;
    const unsigned long long* rev;
    const uint32_t *pick_off, *pick_src, *tile_off, *tile_v;
    unsigned long long* prop;
    unsigned long long* work; // [0] next tile, [1] pairs evaluated, [2] dense rows read, [3] a row did not fit the table, [5] rows whose pairs were read
    uint32_t index_bits, slot_cap, span;
    const SketchMeta* sketch_meta;
    const uint4* sketch; // null: every dense row is read
};

// The table region holds the staged sketches of the picker rows, then the rank table of the sparse part, then the staged dense rows.
struct JoinLds {
    uint32_t G, rowptr, rownnz, row_id, row_worst, col_id, col_worst, listed, seen, seen_col, scan, ctl, tab, tab_bytes, total;
    __host__ __device__ JoinLds(uint32_t index_bits, uint32_t slot_cap, bool narrow) {
        uint32_t o = 0;
        G = o; o += JT_ROWS * JT_STRIDE * 4;
        o = (o + 7) & ~7u;
        rowptr = o; o += (JT_ROWS + JT_COLS) * 8;
        rownnz = o; o += (JT_ROWS + JT_COLS) * 4;
        row_id = o; o += JT_ROWS * 4;
        row_worst = o; o += JT_ROWS * 4;
        col_id = o; o += JT_COLS * 4;
        col_worst = o; o += JT_COLS * 4;
        listed = o; o += JT_COLS * 4;
        seen = o; o += JT_SEEN * 4;
        seen_col = o; o += JT_SEEN;
        scan = o; o += 20 * 4;
        ctl = o; o += 8 * 4;
        o = (o + 15) & ~15u;
        tab = o;
        const uint32_t table = (RankTabLds(index_bits, slot_cap, narrow).total + 15) & ~15u, least = JT_ROWS * JT_STAGE_DIMS * 4;
        tab_bytes = table > least ? table : least;
        o += tab_bytes;
        total = o;
    }
};

// Dense part of a tile on v_mfma_f32_16x16x4_f32. A wave owns 16 columns and a range of 16-float blocks of the
// dimensions; the picker rows come from LDS (`A`: row r, float4 c of the staged dimensions at A[r * row4 + (c ^ (r & 7))] -- the
// swizzle spreads the sixteen rows of a read over the banks without padding), the column rows straight from memory (`pb`: the
// lane's column at the first staged dimension). Lane (j, g), j = lane % 16, g = lane / 16, supplies float4 number 4 b + g of block
// b for row j (A operand) and for column j (B operand): the four multiplies of a block take one component each, so k-slot g of
// multiply c stands for dimension 16 b + 4 g + c on both sides. RING column blocks are in flight ahead of the one being
// multiplied (a ring of registers, filled by join_ring, refilled as it is consumed). Rows 16..31 of the tile take a second accumulator fed from the
// same column registers, and only when the tile has them: a tile of at most 16 rows costs half the matrix time.
// Result: lane (j, g) holds row 4 g + e (+ 16), column j in acc0[e] (acc1[e]).
typedef float floatx4 __attribute__((ext_vector_type(4)));
template <int RING>
__device__ __forceinline__ void join_ring(float4 (&ring)[RING], const float4* pb, int b_begin) {
#pragma unroll
    for (int u = 0; u < RING; u++) ring[u] = pb[4 * (b_begin + u)];
}
template <int RING>
__device__ __forceinline__ void join_dense16(float4 (&ring)[RING], const float4* A, uint32_t row4, uint32_t nr, const float4* pb, int lane, int b_begin, int b_end,
                                             floatx4& acc0, floatx4& acc1) {
    const int j = lane & 15, g = lane >> 4;
    const uint32_t i0 = min((uint32_t)j, nr - 1), i1 = min(16u + (uint32_t)j, nr - 1);
    const float4* a0 = A + i0 * row4;
    const float4* a1 = A + i1 * row4;
    const uint32_t s0 = i0 & 7, s1 = i1 & 7;
    const bool two = nr > 16; // wave-uniform
#pragma unroll 1
    for (int b = b_begin; b < b_end; b += RING) {
        const bool more = b + RING < b_end;
#pragma unroll
        for (int u = 0; u < RING; u++) {
            const float4 bv = ring[u];
            if (more) ring[u] = pb[4 * (b + u + RING)];
            const uint32_t c = 4u * (uint32_t)(b + u) + (uint32_t)g;
            const float4 av = a0[c ^ s0];
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, bv.x, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, bv.y, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, bv.z, acc0, 0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, bv.w, acc0, 0, 0, 0);
            if (two) {
                const float4 aw = a1[c ^ s1];
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(aw.x, bv.x, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(aw.y, bv.y, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(aw.z, bv.z, acc1, 0, 0, 0);
                acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(aw.w, bv.w, acc1, 0, 0, 0);
            }
        }
    }
}

// The pairs of row or column i (wave-uniform) of a tile.
template <bool NARROW>
__device__ __forceinline__ Pairs tile_pairs(const char* recs, const unsigned long long* rowptr, const uint32_t* rownnz, uint32_t i) {
    const unsigned long long at = rowptr[i];
    Pairs p;
    p.base = recs + ((unsigned long long)uniform((uint32_t)(at >> 32)) << 32 | uniform((uint32_t)at));
    const uint32_t w = uniform(rownnz[i]);
    p.nnz = w & 0xFFFFu;
    p.ns = w >> 16;
    p.narrow = NARROW ? 1u : 0u;
    return p;
}

// Sparse part of a tile: G[r * JT_STRIDE + c] = <row r, column c>_sparse for the R rows and M columns whose record addresses and
// shapes `rowptr` / `rownnz` hold (rows at [0, JT_ROWS), columns at [JT_ROWS, JT_ROWS + JT_COLS): gram_rows_gather). Groups of
// eight rows in the rank table, every column probes it once per group. All threads of the workgroup call it after a barrier behind
// those arrays; it ends with a barrier. `unfit` = counter of rows whose terms did not fit the table.
// The pairs of a group's rows are requested while the group before it is probed, those of a wave's columns TILE_AHEAD columns ahead
// (a tile of the join has one group in most cases: with the columns held in registers for all groups a wave needs 96 of them and a CU holds
// one workgroup only; HOLD does that for the full tiles of a Gram matrix where it is so: K = 128 prune of 12 000 docs, 360 terms a row 17.7 -> 16.5 ms). A group of at most four pivots (an average tile of a 100 000-document build has five) reads one plane of
// the table; with the rows' lists looked up among the columns instead of sorted and searched, the tenth step of that build
// went from 6.33 to 5.91 ms.
// `meanwhile` runs once the first loads are on their way; it may use the table region and has to leave it behind a barrier.
template <bool NARROW, int NT, bool HOLD, typename Meanwhile>
__device__ __forceinline__ void tile_sparse(const char* recs, const RankTab& T, float* G, const unsigned long long* rowptr, const uint32_t* rownnz, uint32_t* scan, uint32_t R,
                                            uint32_t M, unsigned long long* unfit, int tid, int wave, int lane, Meanwhile meanwhile) {
    constexpr int NW = NT / WAVE, TILE_AHEAD = HOLD ? JT_COLS / NW : NARROW ? 3 : 2;
    constexpr int BATCH = HOLD && NW == 8 ? 2 : 1; // columns a wave probes together: with two waves per SIMD one at a time leaves waits uncovered
    static_assert(NW >= RT_T, "a wave per pivot of a group");
    auto row_pairs = [&](uint32_t i) { return tile_pairs<NARROW>(recs, rowptr, rownnz, i); };
    auto col_pairs = [&](uint32_t b) { return tile_pairs<NARROW>(recs, rowptr, rownnz, JT_ROWS + b); };
    // a group's pivots, one per wave (as the prune holds its rows): a build hands every wave its own row's pairs, four to a lane
    RtRow<NARROW> pv;
    uint32_t pv_shape = 0;
    auto pivots_load = [&](uint32_t first) {
        pv_shape = 0;
        if (wave < RT_T && first + wave < R) {
            pv_shape = uniform(rownnz[first + wave]);
            rt_row_load(pv, row_pairs(first + wave), lane);
        }
    };
    // the wave's columns wave, wave + NW, ...; shapes (nnz | ns << 16) are wave-uniform. Slot s holds columns wave + (s + k * TILE_AHEAD) * NW
    RtRow<NARROW> col[TILE_AHEAD];
    uint32_t col_shape[TILE_AHEAD];
    auto col_load = [&](int s, uint32_t b) {
        col_shape[s] = uniform(rownnz[JT_ROWS + b]);
        rt_row_load(col[s], col_pairs(b), lane);
    };
    pivots_load(0);
#pragma unroll
    for (int s = 0; s < TILE_AHEAD; s++) {
        col_shape[s] = 0;
        if (wave + s * NW < (int)M) col_load(s, wave + s * NW);
    }
    meanwhile();
    uint32_t a0 = 0;
    while (a0 < R) {
        uint32_t nt = min((uint32_t)RT_T, R - a0);
        uint32_t built;
        while (true) {
            built = ranktab_build_rows<NARROW>(T, pv, pv_shape, (uint32_t)wave < nt, wave, row_pairs(min(a0 + wave, R - 1)), scan, tid, NT, nt > 4 ? 2 : 1);
            if (built != EMPTY || nt == 1) break;
            nt = (nt + 1) / 2; // the registers hold the first pivots of the group whatever nt is
        }
        const uint32_t a1 = a0 + nt;
        if (a1 < R) pivots_load(a1);
        if (built == EMPTY) { // one row alone does not fit: its sparse part is missing, the host is told
            if (tid == 0) atomicAdd(unfit, 1ull);
            for (uint32_t c = tid; c < M; c += NT) G[a0 * JT_STRIDE + c] = 0.f;
            a0 = a1;
            continue;
        }
        const uint32_t n_ovf = NARROW ? 0u : uniform(min(scan[16], (uint32_t)RT_OVF));
        auto probe = [&](auto pivots) {
            constexpr int NP = decltype(pivots)::value;
            for (uint32_t b0 = wave; b0 < M; b0 += TILE_AHEAD * NW) {
#pragma unroll
                for (int s = 0; s < TILE_AHEAD; s += BATCH) {
                    const uint32_t b = b0 + s * NW;
                    if (b < M) { // wave-uniform; a second column that is not there has no pairs
                        float acc[BATCH][NP];
                        RtRow<NARROW> rows[BATCH];
                        uint32_t shape[BATCH];
#pragma unroll
                        for (int k = 0; k < BATCH; k++) {
                            rows[k] = col[s + k];
                            shape[k] = col_shape[s + k];
                            if constexpr (HOLD) { // what follows from a row is worked out where it is used, not kept for all groups
                                rows[k].touch();
                                asm volatile("" : "+s"(shape[k]));
                            }
                        }
                        if constexpr (!HOLD) {
                            const uint32_t next = b + TILE_AHEAD * NW;
                            if (next < M) col_load(s, next);
                            else if (a1 < R) col_load(s, wave + s * NW); // the first of the slot again, for the next group
                        }
#pragma unroll
                        for (int k = 0; k < BATCH; k++)
#pragma unroll
                            for (int t = 0; t < NP; t++) acc[k][t] = 0.f;
                        ranktab_probe_rows<NARROW, BATCH, NP>(T, rows, shape, [&](int k) { return col_pairs(b + k * NW); }, n_ovf, acc, lane);
#pragma unroll
                        for (int k = 0; k < BATCH; k++) {
                            const uint32_t at = b + k * NW;
                            if (k > 0 && at >= M) continue;
                            uint32_t t;
                            if constexpr (NP == 4) {
                                const float z = wave_sum4_dpp(acc[k], lane, &t);
                                if (lane < 4 && t < nt) G[(a0 + t) * JT_STRIDE + at] = z;
                            } else {
                                const float z = wave_sum_1x8(acc[k], lane, &t);
                                if ((lane & 15) < 4 && lane < 32 && t < nt) G[(a0 + t) * JT_STRIDE + at] = z;
                            }
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0); // one batch at a time: the scheduler must not pile up the reads of all of them
                }
            }
        };
        if (nt > 4) probe(std::integral_constant<int, RT_T>{});
        else probe(std::integral_constant<int, 4>{});
        a0 = a1;
        __syncthreads();
    }
}

// Dense part of a tile: adds dense_mul * <row r, column c>_dense to G for the R rows and the M columns c = cols[0 .. M) (null: 0 .. M). The waves share the 16-column
// blocks that exist (8, 4, 2 or 1 by the number of columns) and, for each block, equal parts of the dimensions: no wave idles
// when a tile has few columns. The picker rows are staged in `stage`, all dimensions at once if they fit, else a half or a quarter
// at a time. Partial tiles are added into G in a fixed order, a barrier between them. All threads of the workgroup call it after a barrier; it ends with a
// barrier.
// How the dimensions are split into partial sums follows from split_rows (staging) and split_cols (parts) alone. A node whose pickers fill
// several tiles gives JT_ROWS and all its columns: which pickers are this tile's, and so R and the columns they leave open, is up to the order of
// their arrival, and the sums must not be. That leaves waves idle where few columns are left (last step, K = 128, 200 000 docs 15.7 -> 16.4 ms;
// K = 64, 1 M docs 58.3 -> 58.7); a node of one tile has the same R and columns in every run and splits by them.
template <int NT>
__device__ __forceinline__ void tile_dense(const char* recs, float dense_mul, char* stage, uint32_t stage_bytes, float* G, const unsigned long long* rowptr, const uint32_t* cols,
                                           uint32_t R, uint32_t M, uint32_t split_rows, uint32_t split_cols, int tid, int wave, int lane) {
    constexpr int NW = NT / WAVE;
    constexpr int RING = 8; // column blocks a wave has in flight: 128 KB per CU
    static_assert(DIM == 4 * JT_STAGE_DIMS, "a row is staged whole, in halves or in quarters");
    const uint32_t nblk = split_cols <= 16 ? 1u : split_cols <= 32 ? 2u : split_cols <= 64 ? 4u : 8u, parts = (uint32_t)NW / nblk;
    const uint32_t blk = (uint32_t)wave % nblk, part = (uint32_t)wave / nblk;
    const bool active = blk * 16 < M;
    const uint32_t fit = stage_bytes / (4 * split_rows);
    const uint32_t dims = fit >= DIM ? (uint32_t)DIM : fit >= DIM / 2 ? (uint32_t)DIM / 2 : (uint32_t)DIM / 4;
    const uint32_t per = dims / 16 / parts; // 16-float blocks of the staged dimensions per part: 64 ... 1
    float4* A = reinterpret_cast<float4*>(stage);
    const uint32_t row4 = dims / 4;
    uint32_t jcol = min(blk * 16 + (uint32_t)(lane & 15), M - 1);
    if (cols) jcol = cols[jcol];
    const float4* pb = reinterpret_cast<const float4*>(recs + rowptr[JT_ROWS + jcol] - DENSE_BYTES) + (lane >> 4);
    floatx4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t d4 = 0; d4 < DIM / 4; d4 += row4) {
        const int b0 = (int)(part * per), b1 = b0 + (int)per;
        float4 ring[RING] = {}; // the first blocks are requested before the rows are staged
        if (active) {
            if (per >= (uint32_t)RING) join_ring<RING>(ring, pb + d4, b0);
            else if (per >= 4) join_ring<4>(reinterpret_cast<float4(&)[4]>(ring), pb + d4, b0);
            else join_ring<1>(reinterpret_cast<float4(&)[1]>(ring), pb + d4, b0);
        }
        if (d4) __syncthreads();
#pragma unroll 4
        for (uint32_t i = tid; i < R * row4; i += NT) {
            const uint32_t r = i / row4, c = i % row4;
            A[r * row4 + (c ^ (r & 7))] = reinterpret_cast<const float4*>(recs + rowptr[r] - DENSE_BYTES)[d4 + c];
        }
        __syncthreads();
        if (active) {
            if (per >= (uint32_t)RING) join_dense16<RING>(ring, A, row4, R, pb + d4, lane, b0, b1, acc0, acc1);
            else if (per >= 4) join_dense16<4>(reinterpret_cast<float4(&)[4]>(ring), A, row4, R, pb + d4, lane, b0, b1, acc0, acc1);
            else join_dense16<1>(reinterpret_cast<float4(&)[1]>(ring), A, row4, R, pb + d4, lane, b0, b1, acc0, acc1);
        }
    }
    for (uint32_t ph = 0; ph < parts; ph++) {
        if (active && part == ph && blk * 16 + (uint32_t)(lane & 15) < M) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float* at = &G[(4 * (lane >> 4) + e) * JT_STRIDE + jcol];
                *at += dense_mul * acc0[e];
                if (R > 16) at[16 * JT_STRIDE] += dense_mul * acc1[e];
            }
        }
        __syncthreads();
    }
}

// Which pairs of a tile can still matter, from the 8-bit sketches of the dense rows (apoe_device.h). Before the sparse part:
// tile_sketch, upper bounds of the dense parts; the code products of a 16 x 16 block are sixteen v_mfma_i32_16x16x64_i8 (exact; a
// wave takes 16 columns), lane (j, g), j = lane % 16, g = lane / 16, supplies the sixteen codes 64 b + 16 g .. of block b for row j
// and for column j, and holds row 4 g + e (+ 16), column j of the result: the bounds stay in its registers, two to a word and
// rounded up to bf16 (they are 0.8 off under dense_mul 49 and rows of norm 1 anyway). Behind the sparse part: tile_undecided, bit r
// of colmask[c] = the distance of row r and column c may lie below row_worst[r], colkeep[c] = some row's may lie below col_worst[c].
// All threads call either after a barrier; either ends with one.
typedef int intx4 __attribute__((ext_vector_type(4)));
struct TileSketch {
    uint32_t colmask[JT_COLS], colkeep[JT_COLS], cols[JT_COLS];
    float scale[JT_ROWS], err[JT_ROWS], norm[JT_ROWS];
};
struct TileBound {
    uint32_t two[4]; // [e]: rows 4 g + e (low half) and 16 + 4 g + e
};
__device__ __forceinline__ uint32_t bf16_at_least(float x) { // the smallest bf16 not below x, as bits; a NaN may become an infinity
    const uint32_t b = __float_as_uint(x);
    return (b >> 31 ? b : b + 0xFFFFu) >> 16;
}
template <int NT>
__device__ __forceinline__ void tile_sketch(const SketchMeta* meta, const uint4* sketch, const float* dnorm, float dense_mul, uint4* stage,
                                            const uint32_t* row_id, const uint32_t* col_id, TileSketch* S, TileBound& bound, uint32_t R, uint32_t M, int tid,
                                            int wave, int lane) {
    constexpr uint32_t ROW16 = SKETCH_BYTES / 16;
    constexpr int BLOCKS = SKETCH_BYTES / 64, RING = 8;
    static_assert(NT / WAVE >= JT_COLS / 16, "a wave per block of columns");
    const int j = lane & 15, g = lane >> 4;
    const uint32_t cid = col_id[min((uint32_t)(wave * 16 + j), M - 1)];
    const bool active = wave * 16 < (int)M; // wave-uniform
    uint4 ring[RING] = {};
    SketchMeta cm = {0.f, 0.f};
    float cn = 0.f;
    const uint4* pc = sketch + (size_t)cid * ROW16 + g;
    if (active) {
#pragma unroll
        for (int u = 0; u < RING; u++) ring[u] = pc[4 * u];
        cm = meta[cid];
        cn = dnorm[cid];
    }
    for (uint32_t i = tid; i < R * ROW16; i += NT) {
        const uint32_t r = i / ROW16, k = i % ROW16;
        stage[r * ROW16 + (k ^ (r & 7))] = sketch[(size_t)row_id[r] * ROW16 + k];
    }
    if ((uint32_t)tid < R) {
        const SketchMeta m = meta[row_id[tid]];
        S->scale[tid] = m.scale;
        S->err[tid] = m.err;
        S->norm[tid] = dnorm[row_id[tid]];
    }
    if (tid < JT_COLS) S->colmask[tid] = S->colkeep[tid] = 0;
    __syncthreads();
    if (active) {
        const uint32_t i0 = min((uint32_t)j, R - 1), i1 = min(16u + (uint32_t)j, R - 1);
        const uint4 *a0 = stage + i0 * ROW16, *a1 = stage + i1 * ROW16;
        const uint32_t s0 = i0 & 7, s1 = i1 & 7;
        const bool two = R > 16;
        intx4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
#pragma unroll 1
        for (int b = 0; b < BLOCKS; b += RING) {
            const bool more = b + RING < BLOCKS;
#pragma unroll
            for (int u = 0; u < RING; u++) {
                const intx4 bv = __builtin_bit_cast(intx4, ring[u]);
                if (more) ring[u] = pc[4 * (b + u + RING)];
                const uint32_t k = 4u * (uint32_t)(b + u) + (uint32_t)g;
                acc0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(intx4, a0[k ^ s0]), bv, acc0, 0, 0, 0);
                if (two) acc1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(intx4, a1[k ^ s1]), bv, acc1, 0, 0, 0);
            }
        }
        auto most = [&](uint32_t r, int dot) { // with room for the rounding of the exact dense part
            const float rn = S->norm[r], re = S->err[r];
            return dense_mul * ((float)dot * (S->scale[r] * cm.scale) + (rn * cm.err + re * (cn + cm.err))) + 1e-5f * (dense_mul * rn * cn + 1.0f);
        };
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const uint32_t r = min((uint32_t)(4 * g + e), R - 1);
            bound.two[e] = bf16_at_least(most(r, acc0[e]));
            if (two) bound.two[e] |= bf16_at_least(most(min(r + 16u, R - 1), acc1[e])) << 16;
        }
    }
    __syncthreads();
}
__device__ __forceinline__ void tile_undecided(const TileBound& bound, const float* G, const float* row_worst, const float* col_worst, const uint32_t* listed,
                                               TileSketch* S, uint32_t R, uint32_t M, int wave, int lane) {
    const uint32_t c = (uint32_t)(wave * 16 + (lane & 15));
    if (c < M) {
        const float cw = col_worst[c];
        uint32_t mask = 0, keep = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t r = 16 * h + 4 * (lane >> 4) + e;
                if (r < R) {
                    const float s = G[r * JT_STRIDE + c], least = 1.0f - (s + __uint_as_float(h ? bound.two[e] & 0xFFFF0000u : bound.two[e] << 16)) - 1e-5f * fabsf(s);
                    mask |= (least >= row_worst[r] ? 0u : 1u) << r; // not a number: undecided
                    keep |= least >= cw ? 0u : 1u;
                }
            }
        }
        mask &= ~listed[c];
        if (mask) atomicOr(&S->colmask[c], mask);
        if (keep) S->colkeep[c] = 1u;
    }
    __syncthreads();
}

// Slot of an id in a tile's id set, its own or the free one where it belongs.
__device__ __forceinline__ uint32_t tile_set_find(const uint32_t* set, uint32_t id) {
    uint32_t h = term_hash(id, JT_SEEN - 1);
    while (set[h] != id && set[h] != EMPTY) h = (h + 1) & (JT_SEEN - 1);
    return h;
}

template <bool NARROW, uint32_t KK, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void join_tile_kernel(JoinArgs a) {
    constexpr uint32_t HALVES = KK / 64; // tiles per block of picker rows
    constexpr int NW = NT / WAVE;
    a.C.narrow = NARROW ? 1u : 0u;
    extern __shared__ __align__(16) char smem[];
    const JoinLds L(a.index_bits, a.slot_cap, NARROW);
    const RankTab T = ranktab_at(smem + L.tab, a.index_bits, a.slot_cap, a.span, NARROW);
    float* G = reinterpret_cast<float*>(smem + L.G);
    unsigned long long* rowptr = reinterpret_cast<unsigned long long*>(smem + L.rowptr);
    uint32_t* rownnz = reinterpret_cast<uint32_t*>(smem + L.rownnz);
    uint32_t* row_id = reinterpret_cast<uint32_t*>(smem + L.row_id);
    uint32_t* col_id = reinterpret_cast<uint32_t*>(smem + L.col_id);
    float* row_worst = reinterpret_cast<float*>(smem + L.row_worst);
    float* col_worst = reinterpret_cast<float*>(smem + L.col_worst);
    uint32_t* listed = reinterpret_cast<uint32_t*>(smem + L.listed); // bit r of [c]: column c is in the list of row r, or r itself
    uint32_t* seen = reinterpret_cast<uint32_t*>(smem + L.seen); // the columns' ids as a set ...
    uint8_t* seen_col = reinterpret_cast<uint8_t*>(smem + L.seen_col); // ... and their numbers; NO_COL: not a column of this tile
    constexpr uint8_t NO_COL = 0xFF;
    uint32_t* scan = reinterpret_cast<uint32_t*>(smem + L.scan);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(smem + L.ctl); // [0] tile, [1] columns, [4] columns whose dense rows are read; [2], [3], [5] counts (below)
    TileSketch* S = reinterpret_cast<TileSketch*>(seen); // once the rows' lists are looked up
    static_assert(sizeof(TileSketch) <= JT_SEEN * 4, "the id set's bytes hold what the sketches tell");

    const int wave = (int)uniform(threadIdx.x / WAVE);
    const uint32_t n_tiles = a.tile_off[a.n];

    if (threadIdx.x == 0) { ctl[2] = 0; ctl[3] = 0; ctl[5] = 0; } // pairs evaluated, dense rows and rows of pairs read by this workgroup's tiles
    while (true) {
        // opaque to the compiler: what follows from a thread's number is worked out where a tile needs it, not once for all tiles and spilled
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int lane = tid & (WAVE - 1);
        __syncthreads();
        if (tid == 0) { ctl[0] = (uint32_t)atomicAdd(a.work, 1ull); ctl[1] = 0; }
        for (uint32_t i = tid; i < JT_SEEN; i += NT) seen[i] = EMPTY;
        if (tid < JT_COLS) listed[tid] = 0;
        __syncthreads();
        const uint32_t tile = uniform(ctl[0]);
        if (tile >= n_tiles) break;
        const uint32_t v = uniform(a.tile_v[tile]);
        const uint32_t p0 = uniform(a.pick_off[v]), cnt = uniform(a.pick_off[v + 1]) - p0;
        const uint32_t local = tile - uniform(a.tile_off[v]);
        const uint32_t r0 = local / HALVES * JT_ROWS, half = local % HALVES;
        const uint32_t R = min((uint32_t)JT_ROWS, cnt - r0);

        // rows: pickers of v; columns: N(v) and R(v) without repeats
        if (tid < JT_ROWS) {
            const uint32_t u = (uint32_t)tid < R ? a.pick_src[p0 + r0 + tid] : EMPTY;
            row_id[tid] = u;
            row_worst[tid] = u != EMPTY ? a.dist[(size_t)u * KK + KK - 1] : -INF_DIS;
        }
        auto column = [&](uint32_t id, bool wanted) { // an id met for the first time
            if (id >= a.n) return;
            uint32_t h = term_hash(id, JT_SEEN - 1);
            while (true) {
                const uint32_t old = atomicCAS(&seen[h], EMPTY, id);
                if (old == id) return;
                if (old == EMPTY) break;
                h = (h + 1) & (JT_SEEN - 1);
            }
            uint32_t at = NO_COL;
            if (wanted) {
                at = atomicAdd(&ctl[1], 1u);
                col_id[at] = id;
            }
            seen_col[h] = (uint8_t)at;
        };
        if (HALVES == 1) {
            if (tid < 2 * (int)KK) column(tid < (int)KK ? a.ids[(size_t)v * KK + tid] & ~FLAG : (uint32_t)a.rev[(size_t)v * KK + (tid - KK)], true);
        } else {
            // first tile: the list of v without repeats; second tile: what the reverse list adds to it
            uint32_t rc = EMPTY;
            if (tid < (int)KK) {
                if (half == 1) rc = (uint32_t)a.rev[(size_t)v * KK + tid];
                column(a.ids[(size_t)v * KK + tid] & ~FLAG, half == 0);
            }
            if (half == 1) {
                __syncthreads();
                column(rc, true);
            }
        }
        __syncthreads();
        const uint32_t M = uniform(ctl[1]);
        if (M == 0) continue;
        if ((uint32_t)tid < M) col_worst[tid] = a.symmetric ? a.dist[(size_t)col_id[tid] * KK + KK - 1] : -INF_DIS;
        gram_rows_gather(a.C, row_id, R, rowptr, rownnz, tid, NT);
        gram_rows_gather(a.C, col_id, M, rowptr + JT_ROWS, rownnz + JT_ROWS, tid, NT);
        // which columns the rows list already (they are never offered): wave w looks the entries of rows w, w + NW, ... up among the columns
        {
            constexpr int KL = KK / WAVE;
            uint32_t own[JT_ROWS / NW][KL];
#pragma unroll
            for (int k = 0; k < JT_ROWS / NW; k++) {
                const uint32_t r = wave + k * NW;
#pragma unroll
                for (int l = 0; l < KL; l++) own[k][l] = r < R ? a.ids[(size_t)row_id[r] * KK + l * WAVE + lane] & ~FLAG : EMPTY;
            }
#pragma unroll
            for (int k = 0; k < JT_ROWS / NW; k++) {
                const uint32_t r = wave + k * NW;
                auto mark = [&](uint32_t id) {
                    const uint32_t h = tile_set_find(seen, id);
                    if (seen[h] == id && seen_col[h] != NO_COL) atomicOr(&listed[seen_col[h]], 1u << r);
                };
                if (r < R) { // wave-uniform
#pragma unroll
                    for (int l = 0; l < KL; l++)
                        if (own[k][l] < a.n) mark(own[k][l]);
                    if (lane == 0) mark(row_id[r]);
                }
            }
        }
        __syncthreads();
        // Once the lists have settled, the sketches (1 KB a row) tell for most columns that no exact distance of theirs can matter, or only
        // to rows that list them already: those columns' dense rows (4 KB) are not read. A step asks them when few pairs of the step
        // before entered a list (join_step_finish).
        const bool settled = a.sketch != nullptr;
        TileBound bound = {};
        tile_sparse<NARROW, NT, false>(a.C.recs, T, G, rowptr, rownnz, scan, R, M, a.work + 3, tid, wave, lane, [&]() {
            if (settled)
                tile_sketch<NT>(a.sketch_meta, a.sketch, a.C.dnorm, a.dense_mul, reinterpret_cast<uint4*>(smem + L.tab), row_id, col_id, S, bound, R, M, tid,
                                wave, lane);
        });
        const uint32_t* cols = nullptr;
        uint32_t Mc = M;
        if (settled) {
            tile_undecided(bound, G, row_worst, col_worst, listed, S, R, M, wave, lane);
            if (wave == 0) {
                uint32_t n = 0;
#pragma unroll
                for (int k = 0; k < JT_COLS / WAVE; k++) {
                    const uint32_t c = k * WAVE + lane;
                    const bool keep = c < M && (S->colmask[c] | S->colkeep[c]) != 0;
                    const uint64_t b = __ballot(keep);
                    if (keep) S->cols[n + __popcll(b & ((1ull << lane) - 1))] = c;
                    n += __popcll(b);
                }
                if (lane == 0) ctl[4] = n;
            }
            __syncthreads();
            cols = S->cols;
            Mc = uniform(ctl[4]);
        }
        if (Mc) tile_dense<NT>(a.C.recs, a.dense_mul, smem + L.tab, L.tab_bytes, G, rowptr, cols, R, Mc, cnt > JT_ROWS ? (uint32_t)JT_ROWS : R, cnt > JT_ROWS ? M : Mc, tid, wave, lane);
        // proposals
        for (uint32_t p = tid; p < R * Mc; p += NT) {
            const uint32_t r = p / Mc, c = cols ? cols[p % Mc] : p % Mc;
            const uint32_t uid = row_id[r], cid = col_id[c];
            if (uid == cid) continue;
            const float d = 1.0f - G[r * JT_STRIDE + c];
            if (d < row_worst[r] && !((listed[c] >> r) & 1u)) atomicMin(&a.prop[(size_t)uid * a.P + prop_slot(cid, a.P)], dist_id_key(d, cid));
            if (d < col_worst[c]) atomicMin(&a.prop[(size_t)cid * a.P + prop_slot(uid, a.P)], dist_id_key(d, uid));
        }
        if (tid == 0) { // summed here, sent once when the workgroup leaves: a million atomics on one address per step would queue up
            ctl[2] += R * M;
            ctl[3] += Mc ? R + Mc : 0;
            ctl[5] += R + M;
            if (ctl[2] >= 0x40000000u) { atomicAdd(a.work + 1, (unsigned long long)ctl[2]); ctl[2] = 0; }
        }
    }
    if (threadIdx.x == 0) {
        atomicAdd(a.work + 1, (unsigned long long)ctl[2]);
        atomicAdd(a.work + 2, (unsigned long long)ctl[3]);
        atomicAdd(a.work + 5, (unsigned long long)ctl[5]);
    }
}

// One wave per node: its proposals (2 * KK slots, PL per lane) merged into its list (KL entries per lane: entry e in register
// e / 64 of lane e % 64); the entries that are new in the list register with their nodes' reverse lists (index.cu:362-372
// registers every entry of a changed list and starts the reverse lists again with every step; the join keeps them over the
// steps, so an entry registers once, when it enters). Proposal slots are left empty.
template <uint32_t KK>
__global__ __launch_bounds__(256) void join_apply_kernel(uint32_t n, uint32_t* ids, float* dist, unsigned long long* prop, unsigned long long* rev,
                                                         uint32_t* rev_cnt, unsigned long long* inserted) {
    constexpr int KL = KK / WAVE, PL = 2 * KL;
    constexpr uint32_t P = 2 * KK;
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const uint32_t u = blockIdx.x * 4 + wave;
    if (u >= n) return;
    const size_t base = (size_t)u * KK, pbase = (size_t)u * P;
    unsigned long long key[PL];
    bool some = false;
#pragma unroll
    for (int s = 0; s < PL; s++) {
        key[s] = prop[pbase + s * WAVE + lane];
        some |= key[s] != ~0ull;
    }
    if (__ballot(some) == 0) return;
#pragma unroll
    for (int s = 0; s < PL; s++) prop[pbase + s * WAVE + lane] = ~0ull;
    uint32_t own_id[KL];
    float own_d[KL];
#pragma unroll
    for (int k = 0; k < KL; k++) {
        own_id[k] = ids[base + k * WAVE + lane];
        own_d[k] = dist[base + k * WAVE + lane];
    }
    // a proposal counts if it names another node that is not in the list yet (one id always hashes to one slot: no repeats among them)
    bool valid[PL];
    float d[PL];
#pragma unroll
    for (int s = 0; s < PL; s++) {
        const uint32_t c = (uint32_t)key[s];
        valid[s] = key[s] != ~0ull && c != u && c < n;
        d[s] = join_key_dist(key[s]);
    }
#pragma unroll
    for (int k = 0; k < KL; k++) {
        for (uint32_t i = 0; i < WAVE; i++) {
            const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)own_id[k], i) & ~FLAG;
#pragma unroll
            for (int s = 0; s < PL; s++) valid[s] = valid[s] && x != (uint32_t)key[s];
        }
    }
    uint64_t nb[PL], any = 0;
#pragma unroll
    for (int s = 0; s < PL; s++) { nb[s] = __ballot(valid[s]); any |= nb[s]; }
    if (any == 0) return;
    // new: rank among the new ones by (distance, id), plus the old entries strictly closer (new first on ties)
    uint32_t rank_new[PL], le_old[KL];
#pragma unroll
    for (int s = 0; s < PL; s++) rank_new[s] = 0;
#pragma unroll
    for (int k = 0; k < KL; k++) le_old[k] = 0;
#pragma unroll
    for (int t = 0; t < PL; t++) {
        for (uint64_t rest = nb[t]; rest; rest &= rest - 1) {
            const unsigned long long ki = readlane64(key[t], (uint32_t)__builtin_ctzll(rest));
#pragma unroll
            for (int s = 0; s < PL; s++) rank_new[s] += ki < key[s];
#pragma unroll
            for (int k = 0; k < KL; k++) le_old[k] += join_key_dist(ki) <= own_d[k]; // old entry: new ones at or below its distance go first
        }
    }
#pragma unroll
    for (int k = 0; k < KL; k++) {
        for (uint32_t i = 0; i < WAVE; i++) {
            const float di = readlane_f32(own_d[k], i);
#pragma unroll
            for (int s = 0; s < PL; s++) rank_new[s] += di < d[s];
        }
    }
    bool new_in[PL];
    uint32_t n_ins = 0;
#pragma unroll
    for (int s = 0; s < PL; s++) {
        new_in[s] = valid[s] && rank_new[s] < KK;
        n_ins += __popcll(__ballot(new_in[s]));
    }
    if (n_ins == 0) return;
#pragma unroll
    for (int k = 0; k < KL; k++) {
        const uint32_t rank_old = (uint32_t)(k * WAVE + lane) + le_old[k];
        if (rank_old < KK) { ids[base + rank_old] = own_id[k]; dist[base + rank_old] = own_d[k]; }
    }
#pragma unroll
    for (int s = 0; s < PL; s++) {
        if (new_in[s]) { ids[base + rank_new[s]] = (uint32_t)key[s]; dist[base + rank_new[s]] = d[s]; }
    }
    if (lane == 0) atomicAdd(inserted + (blockIdx.x % JOIN_COUNT_PARTS) * 8, (unsigned long long)n_ins); // one address for every node would serialise a million atomics
    // reverse registration of the new entries: (distance, u) in one word, slot count % K keeps the closer one beyond K
    auto reg = [&](uint32_t e, float dv) {
        const uint32_t v = e & ~FLAG;
        if (v >= n) return;
        const uint32_t slot = atomicAdd(&rev_cnt[v], 1u);
        const unsigned long long k = dist_id_key(dv, u);
        // every registration is a minimum (the lists start at ~0 and the join never starts them again): a store into a slot
        // that a later registration of the same step has already reached through its wrap-around could undo that one
        atomicMin(rev + (size_t)v * KK + (slot % KK), k);
    };
#pragma unroll
    for (int s = 0; s < PL; s++) {
        if (new_in[s]) reg((uint32_t)key[s], d[s]);
    }
}

// work[4] = entries that entered a list in this step, beside the pairs for the host. settled: the step asked the sketches, one for every
// row and column of a tile.
__global__ static void join_account_kernel(unsigned long long* work, unsigned long long* counter, uint32_t settled) {
    counter[KC_EVALUATIONS] += work[1];
    counter[KC_DENSE_ROWS] += work[2];
    counter[KC_JOIN_EVALUATIONS] += work[1];
    counter[KC_JOIN_PAIR_ROWS] += work[5];
    if (settled) counter[KC_SKETCHES] += work[5];
    unsigned long long inserted = 0; // the partial counts of join_apply_kernel
    for (int p = 0; p < JOIN_COUNT_PARTS; p++) inserted += work[JOIN_COUNT_AT + p * 8];
    counter[KC_INSERTED] = inserted;
    work[4] = inserted;
}

__global__ __launch_bounds__(256) static void fill_u64_kernel(unsigned long long* p, uint64_t count, unsigned long long v) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < count; t += (uint64_t)gridDim.x * blockDim.x) p[t] = v;
}
__global__ __launch_bounds__(256) static void fill_u32_kernel2(uint32_t* p, uint64_t count, uint32_t v) {
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < count; t += (uint64_t)gridDim.x * blockDim.x) p[t] = v;
}

// ---- hybrid Gram matrices of whole neighbour lists, tile by tile (the prune of lists longer than 64 entries) ----
//
// For node u = nodes[node0 + q] the valid entries of its list (distance below INF_DIS, a document, not u itself),
// in list order, are the rows and columns of a Gram matrix of at most 128 x 128. Tile t computes rows
// [32 t, 32 t + 32) against the columns [32 t, m): the upper triangle, diagonal blocks whole. The products go to
// gram[q * 128 * 128 + i * 128 + j] for i <= j (entries below the diagonal of a diagonal block are
// written too). Same tile body as the local join: every row of a tile is gathered once, dense part on the matrix cores,
// sparse part through the rank table.
constexpr uint32_t GT_MAX = 128;                 // longest list
struct GramTileArgs {
    CorpusView C;
    float dense_mul;
    uint32_t K, node0, n_nodes;
    const uint32_t* nodes; // node q of the batch is nodes[node0 + q]
    const uint32_t* ids;
    const float* dist;
    float* gram;
    unsigned long long* work; // [0] next tile, [3] a row did not fit the table
    uint32_t index_bits, slot_cap, span;
};

template <bool NARROW, int NT, bool HOLD>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(HOLD ? NT / 256 : 4, HOLD ? NT / 256 : 4))) void gram_tile_kernel(GramTileArgs a) {
    a.C.narrow = NARROW ? 1u : 0u;
    extern __shared__ __align__(16) char smem[];
    const JoinLds L(a.index_bits, a.slot_cap, NARROW);
    const RankTab T = ranktab_at(smem + L.tab, a.index_bits, a.slot_cap, a.span, NARROW);
    float* G = reinterpret_cast<float*>(smem + L.G);
    unsigned long long* rowptr = reinterpret_cast<unsigned long long*>(smem + L.rowptr);
    uint32_t* rownnz = reinterpret_cast<uint32_t*>(smem + L.rownnz);
    uint32_t* row_id = reinterpret_cast<uint32_t*>(smem + L.row_id);
    uint32_t* col_id = reinterpret_cast<uint32_t*>(smem + L.col_id);
    uint32_t* valid = reinterpret_cast<uint32_t*>(smem + L.seen); // the node's valid list entries, in list order
    uint32_t* scan = reinterpret_cast<uint32_t*>(smem + L.scan);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(smem + L.ctl); // [0] tile, [1] valid entries
    static_assert(JT_SEEN >= (int)GT_MAX, "the id set's words hold a whole list");
    const int wave = (int)uniform(threadIdx.x / WAVE);
    while (true) { // a workgroup takes a node and runs its tiles one after the other: the columns of a tile are the rows and columns of the next
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid)); // as in join_tile_kernel
        const int lane = tid & (WAVE - 1);
        const uint64_t lane_lt = (1ull << lane) - 1;
        __syncthreads();
        if (tid == 0) ctl[0] = (uint32_t)atomicAdd(a.work, 1ull);
        __syncthreads();
        const uint32_t slot = uniform(ctl[0]);
        if (slot >= a.n_nodes) break;
        const uint32_t u = uniform(a.nodes[a.node0 + slot]);
        if (wave == 0) {
            const size_t base = (size_t)u * a.K;
            uint32_t m = 0;
            for (uint32_t b0 = 0; b0 < a.K; b0 += WAVE) {
                const uint32_t v = (a.ids[base + b0 + lane] & ~FLAG);
                const float dv = a.dist[base + b0 + lane];
                const bool ok = dv < INF_DIS && v < a.C.n && v != u;
                const uint64_t b = __ballot(ok);
                if (ok) valid[m + __popcll(b & lane_lt)] = v;
                m += __popcll(b);
            }
            if (lane == 0) ctl[1] = m;
        }
        __syncthreads();
        const uint32_t m = uniform(ctl[1]);
        float* out = a.gram + (size_t)slot * GT_MAX * GT_MAX;
        for (uint32_t r0 = 0; r0 < m; r0 += JT_ROWS) {
            const uint32_t R = min((uint32_t)JT_ROWS, m - r0), M = m - r0;
            if ((uint32_t)tid < R) row_id[tid] = valid[r0 + tid];
            if ((uint32_t)tid < M) col_id[tid] = valid[r0 + tid];
            __syncthreads();
            gram_rows_gather(a.C, row_id, R, rowptr, rownnz, tid, NT);
            gram_rows_gather(a.C, col_id, M, rowptr + JT_ROWS, rownnz + JT_ROWS, tid, NT);
            __syncthreads();
            tile_sparse<NARROW, NT, HOLD>(a.C.recs, T, G, rowptr, rownnz, scan, R, M, a.work + 3, tid, wave, lane, [] {});
            tile_dense<NT>(a.C.recs, a.dense_mul, smem + L.tab, L.tab_bytes, G, rowptr, nullptr, R, M, R, M, tid, wave, lane);
            for (uint32_t p = tid; p < R * M; p += NT) {
                const uint32_t r = p / M, c = p % M;
                out[(size_t)(r0 + r) * GT_MAX + r0 + c] = G[r * JT_STRIDE + c];
            }
            __syncthreads(); // G and the id arrays are rewritten by the next tile
        }
    }
}

// Table of a tile, and whether two workgroups share a CU (`pair`, where a row fits the table beside half of the LDS). The table then takes as many slots
// as fit, up to eight rows of the longest kind: an average group of eight rows of 180 terms has 1 000 distinct ones, 1 332 slots fit beside a
// bitmap for a vocabulary of 32 768. A group that exceeds them is done in halves; a corpus with a single row that does would lose that row, so it takes
// the whole LDS.
struct TileShape {
    uint32_t index_bits, slot_cap, span, lds;
    bool pair;
};
static TileShape tile_shape(const apoe_ctx* ctx, const apoe_corpus* c, bool pair) {
    TileShape s;
    s.span = next_pow2(std::max(c->max_term + 1, 1024u));
    s.index_bits = c->narrow ? 2 * s.span : 65536u;
    const uint32_t longest = c->max_nnz_s + c->max_nnz_b, want = std::max<uint32_t>((RT_T * longest + 63) & ~63u, 256u);
    const uint32_t half = (uint32_t)(ctx->lds_per_block / 2), floor_slots = std::max(longest, 256u);
    s.slot_cap = want;
    while (s.slot_cap > floor_slots && JoinLds(s.index_bits, s.slot_cap, c->narrow).total > half) s.slot_cap -= 64;
    s.pair = pair && s.slot_cap >= floor_slots && JoinLds(s.index_bits, s.slot_cap, c->narrow).total <= half;
    if (!s.pair) s.slot_cap = std::min<uint32_t>(want, (uint32_t)APOE_JOIN_MAX_ROW_TERMS);
    s.lds = JoinLds(s.index_bits, s.slot_cap, c->narrow).total;
    return s;
}
// Of the join: also one workgroup for a narrow corpus of whose average rows the smaller table holds fewer than four: its groups
// are pairs and single rows, each a build and a probe of every column. Eight steps on 12 000 docs, K = 64, two workgroups / one, by rows that the
// smaller table holds: vocabulary 32 768 (1 332 slots) 7.6 rows 8.8 / 11.6 ms, 4.2 11.5 / 13.3, 4.0 10.7 / 10.4, 3.9 16.3 / 14.6, 3.1 18.5 / 16.7,
// 1.6 74.7 / 45.3; 65 536 (820 slots) 4.7 10.6 / 12.1, 4.1 12.2 / 12.1, 3.6 12.6 / 12.0, 3.1 17.6 / 13.3. Wide corpora, whose builds and probes
// wait longer, gain from the second workgroup at any length (7.5 rows 16.0 / 20.8 ms, 1.6 198 / 235).
static TileShape join_shape(const apoe_ctx* ctx, const apoe_corpus* c) {
    const TileShape s = tile_shape(ctx, c, true);
    return s.pair && c->narrow && (uint64_t)s.slot_cap * c->n < 4 * c->total_pairs ? tile_shape(ctx, c, false) : s;
}

// A persistent grid of tile workgroups.
template <typename Args>
static int launch_tiles(apoe_ctx* ctx, void (*kernel)(Args), const TileShape& shape, int threads, const Args& a) {
    APOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)shape.lds));
    int per_cu = 1;
    APOE_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), threads, shape.lds));
    kernel<<<(uint32_t)std::max(per_cu, 1) * (uint32_t)ctx->num_cus, threads, shape.lds, ctx->stream>>>(a);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

int join_alloc(apoe_knn* g) {
    const size_t n = g->n;
    APOE_TRY(g->picks.alloc(n * JOIN_PICKS));
    APOE_TRY(g->pick_cnt.alloc(n + 1));
    APOE_TRY(g->pick_off.alloc(n + 1));
    APOE_TRY(g->pick_fill.alloc(n + 1));
    APOE_TRY(g->pick_src.alloc(n * JOIN_PICKS));
    APOE_TRY(g->tile_cnt.alloc(n + 1));
    APOE_TRY(g->tile_off.alloc(n + 1));
    const size_t halves = g->K / 64, P = 2 * (size_t)g->K;
    APOE_TRY(g->tile_v.alloc((n + n * JOIN_PICKS / JT_ROWS + 1) * halves));
    APOE_TRY(g->prop.alloc(n * P));
    APOE_TRY(g->join_work.alloc(JOIN_COUNT_AT + JOIN_COUNT_PARTS * 8));
    size_t temp_bytes = 0;
    APOE_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, temp_bytes, g->pick_cnt.p, g->pick_off.p, (int)(n + 1), g->ctx->stream));
    APOE_TRY(g->scan_tmp.alloc(temp_bytes));
    fill_u64_kernel<<<1024, 256, 0, g->ctx->stream>>>(g->prop.p, (uint64_t)n * P, ~0ull);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

int launch_nnd_join_iterate(apoe_knn* g) {
    apoe_ctx* ctx = g->ctx;
    hipStream_t st = ctx->stream;
    const uint32_t n = g->n;
    APOE_REQUIRE(g->K == 64 || g->K == 128, "the local-join step is built for K = 64 and K = 128 lists, this handle has K = %u", g->K);
    const bool k128 = g->K == 128;
    const uint32_t halves = g->K / 64;
    if (!g->prop.p) APOE_TRY(join_alloc(g));
    const TileShape shape = join_shape(ctx, g->corpus);
    APOE_REQUIRE(shape.lds <= ctx->lds_per_block, "the local-join tile needs %u bytes of LDS, a workgroup may have %zu", shape.lds, ctx->lds_per_block);

    APOE_HIP(hipMemsetAsync(g->counter.p, 0, sizeof(unsigned long long), st)); // the inserted entries; the counts behind them run over the build
    fill_u32_kernel2<<<1024, 256, 0, st>>>(g->pick_cnt.p, (uint64_t)n + 1, 0u);
    fill_u32_kernel2<<<1024, 256, 0, st>>>(g->pick_fill.p, (uint64_t)n + 1, 0u);
    fill_u64_kernel<<<8, 256, 0, st>>>(g->join_work.p, JOIN_COUNT_AT + JOIN_COUNT_PARTS * 8, 0ull);
    if (k128) join_pick_kernel<128><<<(n + 3) / 4, 256, 0, st>>>(n, g->ids.p, g->picks.p, g->pick_cnt.p);
    else join_pick_kernel<64><<<(n + 3) / 4, 256, 0, st>>>(n, g->ids.p, g->picks.p, g->pick_cnt.p);
    APOE_HIP(hipGetLastError());
    join_tile_count_kernel<<<(n + 256) / 256, 256, 0, st>>>(n, halves, g->pick_cnt.p, g->tile_cnt.p);
    APOE_HIP(hipGetLastError());
    size_t temp_bytes = g->scan_tmp.n;
    APOE_HIP(hipcub::DeviceScan::ExclusiveSum(g->scan_tmp.p, temp_bytes, g->pick_cnt.p, g->pick_off.p, (int)(n + 1), st));
    temp_bytes = g->scan_tmp.n;
    APOE_HIP(hipcub::DeviceScan::ExclusiveSum(g->scan_tmp.p, temp_bytes, g->tile_cnt.p, g->tile_off.p, (int)(n + 1), st));
    const uint64_t total = (uint64_t)n * JOIN_PICKS;
    join_fill_kernel<<<(uint32_t)((total + 255) / 256), 256, 0, st>>>(n, halves, g->picks.p, g->pick_off.p, g->tile_off.p, g->pick_fill.p, g->pick_src.p, g->tile_v.p);
    APOE_HIP(hipGetLastError());

    JoinArgs a{};
    a.C = g->corpus->view();
    a.dense_mul = g->dense_scale * g->dense_scale;
    a.n = n;
    a.P = 2 * g->K;
    a.symmetric = g->join_symmetric ? 1u : 0u;
    a.ids = g->ids.p;
    a.dist = g->dist.p;
    a.rev = g->rev.p;
    a.pick_off = g->pick_off.p;
    a.pick_src = g->pick_src.p;
    a.tile_off = g->tile_off.p;
    a.tile_v = g->tile_v.p;
    a.prop = g->prop.p;
    a.work = g->join_work.p;
    a.index_bits = shape.index_bits;
    a.slot_cap = shape.slot_cap;
    a.span = shape.span;
    a.sketch_meta = g->corpus->sketch_meta.p;
    a.sketch = g->settled ? reinterpret_cast<const uint4*>(g->corpus->sketch.p) : nullptr;
    const bool narrow = g->corpus->narrow;
    auto kernel_of = [&](auto threads) {
        constexpr int NT = decltype(threads)::value;
        return k128 ? (narrow ? &join_tile_kernel<true, 128, NT> : &join_tile_kernel<false, 128, NT>)
                    : (narrow ? &join_tile_kernel<true, 64, NT> : &join_tile_kernel<false, 64, NT>);
    };
    if (shape.pair) APOE_TRY(launch_tiles(ctx, kernel_of(std::integral_constant<int, JT_PAIR_THREADS>{}), shape, JT_PAIR_THREADS, a));
    else APOE_TRY(launch_tiles(ctx, kernel_of(std::integral_constant<int, JT_SOLO_THREADS>{}), shape, JT_SOLO_THREADS, a));
    if (k128) join_apply_kernel<128><<<(n + 3) / 4, 256, 0, st>>>(n, g->ids.p, g->dist.p, g->prop.p, g->rev.p, g->rev_cnt.p, g->join_work.p + JOIN_COUNT_AT);
    else join_apply_kernel<64><<<(n + 3) / 4, 256, 0, st>>>(n, g->ids.p, g->dist.p, g->prop.p, g->rev.p, g->rev_cnt.p, g->join_work.p + JOIN_COUNT_AT);
    APOE_HIP(hipGetLastError());
    join_account_kernel<<<1, 1, 0, st>>>(g->join_work.p, g->counter.p, a.sketch != nullptr);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// Whether two workgroups of the Gram tiles share a CU. Their tiles are full: a column is probed once for every eight rows, or for every four or two where the
// terms of eight exceed the table, and rows of one length may do either. So the terms of a few nodes' rows are counted; a probe costs a fifth more for every
// overflow entry (wide pairs: a term whose bit another one of the group has). Narrow corpora take two workgroups where that does not cost more than an eighth more
// with their smaller table than with the whole LDS. Wide ones, whose builds and probes wait longer, up to twice as much, or half more where rows exceed the
// registers (their tails are read again by every probe). K = 128 prune of 12 000 docs, every node open, ms with two workgroups / one, by the terms a row and their vocabulary:
//   narrow: 180 of the synthetic corpora 10.8 / 12.1; uniform 180 of 30 000 14.1 / 12.0, 260 of 2 000 17.4 / 13.5; 360 of 2 000 23.1 / 16.0; 860 of 30 000 200 / 106
//   wide:   180 25.5 / 41.8; 180 of 30 000 35.6 / 85.4; 860 of 30 000 508 / 1027; few terms a bit: 180 of 2 000 17.0 / 20.1, 260 of 2 000 22.5 / 25.0, 360 of 2 000
//           45.2 / 32.9, 460 of 3 000 66.1 / 61.0, 560 of 1 500 82.9 / 48.9
constexpr uint32_t GRAM_SAMPLE = 64; // nodes
constexpr uint32_t GRAM_COUNTED = 3072; // terms: more than any table holds
struct GramSample {
    uint32_t terms[4], shared[4]; // distinct terms of the first one, two, four and eight rows of a node, and how many of them find their bit taken
};
template <bool NARROW>
__global__ __launch_bounds__(256) void gram_sample_kernel(GramTileArgs a, GramSample* out) {
    constexpr uint32_t SLOTS = 4096;
    static_assert(GRAM_COUNTED + 256 < SLOTS, "a free slot is left whatever the threads insert at once");
    __shared__ uint32_t keys[SLOTS], bits[NARROW ? 1 : 65536 / 32], rows[RT_T], rows_n, n_terms, n_shared;
    const uint32_t u = a.nodes[(uint64_t)blockIdx.x * a.n_nodes / gridDim.x];
    RankTab T{};
    T.index_bits = a.index_bits;
    T.span = a.span;
    for (uint32_t i = threadIdx.x; i < SLOTS; i += 256) keys[i] = EMPTY;
    for (uint32_t i = threadIdx.x; i < (NARROW ? 0u : a.index_bits / 32); i += 256) bits[i] = 0;
    if (threadIdx.x == 0) {
        uint32_t m = 0;
        for (uint32_t i = 0; i < a.K && m < (uint32_t)RT_T; i++) {
            const uint32_t v = a.ids[(size_t)u * a.K + i] & ~FLAG;
            if (a.dist[(size_t)u * a.K + i] < INF_DIS && v < a.C.n && v != u) rows[m++] = v;
        }
        rows_n = m;
        n_terms = n_shared = 0;
    }
    __syncthreads();
    for (uint32_t r = 0; r < (uint32_t)RT_T; r++) {
        if (r < rows_n) {
            const uint64_t d = a.C.desc[rows[r]];
            const Pairs sp = record_pairs(a.C, d);
            for (uint32_t j = threadIdx.x; j < sp.nnz && __hip_atomic_load(&n_terms, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < GRAM_COUNTED; j += 256) {
                const uint32_t raw = sp.raw(j).x, idx = ranktab_index<NARROW>(T, raw, j >= sp.ns), key = NARROW ? idx : raw;
                uint32_t h = term_hash(key, SLOTS - 1);
                while (true) {
                    const uint32_t old = atomicCAS(&keys[h], EMPTY, key);
                    if (old == key) break;
                    if (old == EMPTY) {
                        atomicAdd(&n_terms, 1u);
                        if (!NARROW && (atomicOr(&bits[idx >> 5], 1u << (idx & 31)) >> (idx & 31) & 1u)) atomicAdd(&n_shared, 1u);
                        break;
                    }
                    h = (h + 1) & (SLOTS - 1);
                }
            }
        }
        __syncthreads();
        if (threadIdx.x == 0 && (r & (r + 1)) == 0) {
            out[blockIdx.x].terms[__popc(r)] = n_terms;
            out[blockIdx.x].shared[__popc(r)] = n_shared;
        }
        __syncthreads();
    }
}
int gram_tiles_pair(apoe_knn* g, const uint32_t* nodes, uint32_t n_nodes, bool* pair) {
    apoe_ctx* ctx = g->ctx;
    const TileShape two = tile_shape(ctx, g->corpus, true), one = tile_shape(ctx, g->corpus, false);
    *pair = two.pair;
    if (!two.pair) return APOE_OK;
    if (!g->join_work.p) APOE_TRY(g->join_work.alloc(JOIN_COUNT_AT + JOIN_COUNT_PARTS * 8));
    GramTileArgs a{};
    a.C = g->corpus->view();
    a.K = g->K;
    a.n_nodes = n_nodes;
    a.nodes = nodes;
    a.ids = g->ids.p;
    a.dist = g->dist.p;
    a.index_bits = two.index_bits;
    a.span = two.span;
    const uint32_t sample = std::min(n_nodes, GRAM_SAMPLE);
    static_assert(JOIN_COUNT_PARTS * 8 * sizeof(unsigned long long) >= GRAM_SAMPLE * sizeof(GramSample), "the step's partial counters hold the sample");
    GramSample *out = reinterpret_cast<GramSample*>(g->join_work.p + JOIN_COUNT_AT), h[GRAM_SAMPLE];
    if (g->corpus->narrow) gram_sample_kernel<true><<<sample, 256, 0, ctx->stream>>>(a, out);
    else gram_sample_kernel<false><<<sample, 256, 0, ctx->stream>>>(a, out);
    APOE_HIP(hipGetLastError());
    APOE_HIP(hipMemcpyAsync(h, out, sample * sizeof(GramSample), hipMemcpyDeviceToHost, ctx->stream));
    APOE_HIP(hipStreamSynchronize(ctx->stream));
    auto cost = [&](uint32_t slots) { // of a column's probes by eight rows, in fifths of a probe, summed over the sample
        uint64_t sum = 0;
        for (uint32_t i = 0; i < sample; i++) {
            int t = 3;
            while (t > 0 && (h[i].terms[t] > slots || h[i].shared[t] > (uint32_t)RT_OVF)) t--;
            sum += (8u >> t) * (5ull + h[i].shared[t]);
        }
        return sum;
    };
    const uint64_t c2 = cost(two.slot_cap), c1 = cost(one.slot_cap);
    const bool window = g->corpus->total_pairs <= (uint64_t)RT_CHUNKS * WAVE * g->corpus->n;
    *pair = g->corpus->narrow ? 8 * c2 <= 9 * c1 : window ? c2 <= 2 * c1 : 2 * c2 <= 3 * c1;
    return APOE_OK;
}

// Gram matrices (upper triangles) of the lists of nodes[node0 .. node0 + n_nodes) (pair: gram_tiles_pair) into gram[n_nodes][128][128]. *unfit = rows
// whose sparse terms did not fit the tile's table (their products lack the sparse part: the caller must not use the result).
int launch_gram_tiles(apoe_knn* g, const uint32_t* nodes, uint32_t node0, uint32_t n_nodes, bool pair, float* gram, unsigned long long* unfit) {
    apoe_ctx* ctx = g->ctx;
    hipStream_t st = ctx->stream;
    APOE_REQUIRE(g->K <= GT_MAX, "Gram tiles are built for lists of at most %u entries", GT_MAX);
    if (!g->join_work.p) APOE_TRY(g->join_work.alloc(JOIN_COUNT_AT + JOIN_COUNT_PARTS * 8));
    const TileShape shape = tile_shape(ctx, g->corpus, pair);
    APOE_REQUIRE(shape.lds <= ctx->lds_per_block, "a Gram tile needs %u bytes of LDS, a workgroup may have %zu", shape.lds, ctx->lds_per_block);
    fill_u64_kernel<<<1, 64, 0, st>>>(g->join_work.p, 8, 0ull);
    APOE_HIP(hipGetLastError());
    GramTileArgs a{};
    a.C = g->corpus->view();
    a.dense_mul = g->dense_scale * g->dense_scale;
    a.K = g->K;
    a.nodes = nodes;
    a.node0 = node0;
    a.n_nodes = n_nodes;
    a.ids = g->ids.p;
    a.dist = g->dist.p;
    a.gram = gram;
    a.work = g->join_work.p;
    a.index_bits = shape.index_bits;
    a.slot_cap = shape.slot_cap;
    a.span = shape.span;
    if (shape.pair) APOE_TRY(launch_tiles(ctx, g->corpus->narrow ? &gram_tile_kernel<true, JT_PAIR_THREADS, false> : &gram_tile_kernel<false, JT_PAIR_THREADS, false>, shape, JT_PAIR_THREADS, a));
    else if (g->corpus->narrow) APOE_TRY(launch_tiles(ctx, &gram_tile_kernel<true, JT_SOLO_THREADS, true>, shape, JT_SOLO_THREADS, a));
    else APOE_TRY(launch_tiles(ctx, &gram_tile_kernel<false, JT_PAIR_THREADS, true>, shape, JT_PAIR_THREADS, a));
    if (unfit) {
        unsigned long long h[4] = {0, 0, 0, 0};
        APOE_HIP(hipMemcpyAsync(h, g->join_work.p, sizeof(h), hipMemcpyDeviceToHost, st));
        APOE_HIP(hipStreamSynchronize(st));
        *unfit = h[3];
    }
    return APOE_OK;
}

// Whether launch_gram_tiles can serve this handle: lists of at most 128 entries, rows that fit a tile's table, LDS for a tile.
bool gram_tiles_fit(const apoe_knn* g) {
    if (g->K > GT_MAX || g->corpus->max_nnz_s + g->corpus->max_nnz_b > (uint32_t)APOE_JOIN_MAX_ROW_TERMS) return false;
    return tile_shape(g->ctx, g->corpus, false).lds <= g->ctx->lds_per_block;
}

// How many rows did not fit the table in the last step (waits for it). Notes whether the lists have settled: less than a twelfth
// of the step's pairs entered a list. Milliseconds of a step that reads every dense row and of one that asks the sketches first, by the
// share of the step before: 100 000 docs K = 64 0.10: 10.0 / 10.6, 0.09: 8.9 / 9.1, 0.08: 7.9 / 7.8, 0.065: 7.25 / 6.85, 0.005: 7.3 / 5.9;
// 30 011 docs K = 128 0.10: 5.65 / 5.76, 0.09: 4.9 / 4.7, 0.06: 4.3 / 4.0, 0.002: 4.3 / 3.6.
int join_step_finish(apoe_knn* g, unsigned long long* unfit) {
    unsigned long long h[5] = {0, 0, 0, 0, 0};
    APOE_HIP(hipMemcpy(h, g->join_work.p, sizeof(h), hipMemcpyDeviceToHost));
    *unfit = h[3];
    g->settled = h[4] * 12 < h[1];
    return APOE_OK;
}

} // namespace apoe
