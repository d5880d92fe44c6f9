// RNG-IP joint pruning with keyword-aware neighbour recycling, and the final row
// assembly with reverse edges. One workgroup (4 waves) per node for the prune, one
// wave per node for the assembly.
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <memory>

#include "apoe_gram.h"
#include <cmath>

#include "apoe_internal.h"
#include "apoe_ranktab.h"

namespace apoe {

constexpr int PR_THREADS = 256;
constexpr uint32_t ALL_PATHS = PATH_DENSE | PATH_SPARSE | PATH_BM25;

__device__ __forceinline__ void wave_fence_lds() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

struct PruneLds {
    uint32_t tab, idmap, uset, nb_id, nb_dist, det, cid, cdet, sel_id, sel_det, sel_live, sel_kw, o_fwd, o_det, o_kw, ctl, total;
    __host__ __device__ PruneLds(uint32_t term_slots, uint32_t uset_slots, uint32_t map_slots, uint32_t K) {
        uint32_t o = 0;
        tab = o; o += term_slots * 8;
        idmap = o; o += map_slots * 8;
        uset = o; o += uset_slots * 4;
        nb_id = o; o += K * 4;
        nb_dist = o; o += K * 4;
        det = o; o += K * 4;
        cid = o; o += K * 4;
        cdet = o; o += K * 4;
        sel_id = o; o += K * 4;
        sel_det = o; o += K * 4;
        sel_live = o; o += K * 4;
        sel_kw = o; o += K * 4;
        o_fwd = o; o += K * 4;
        o_det = o; o += K * 4;
        o_kw = o; o += (1 + APOE_KW_CAND) * 4;
        ctl = o; o += 16 * 4;
        total = o;
    }
};

enum { PC_M = 0, PC_NSEL = 1, PC_REJECT = 2, PC_ALLFLAG = 3, PC_CNT = 4, PC_FAIL = 5, PC_OPEN = 6, PC_STILL_OPEN = 7, PC_TABLE = 8 };

// What a node leaves to another form of the prune: a pair that bounds do not settle, or a neighbour whose norm is not finite. The gathered forms
// multiply a value by zero where a row lacks its term, which an infinite one does not survive; the table-probing kernel multiplies hits only.
enum { NODE_SETTLED = 0, NODE_OPEN = 1, NODE_TABLE = 2 };

// allan_poe (index.cu:539-714) for node u = blockIdx.x (nodes: the list's entry there):
//  (a) detour counts over u's sorted list; (b) order by (detour, rank);
//  (c) sequential RNG-IP selection: candidate c is the pivot, each live selected s is
//      evaluated against it by one wave; norm[c] < <c,s> rejects c, norm[s] < <c,s>
//      tombstones s; (d) c carries the keyword flag when every live s it met has a
//      BM25 term that u holds and c lacks; (e) first `d` live selected go to the
//      forward row, flagged live ones beyond become keyword-edge candidates.
__global__ __launch_bounds__(PR_THREADS) void prune_kernel(CorpusView C, float dense_mul, const float* __restrict__ norms, uint32_t K,
                                                           const uint32_t* __restrict__ ids, const float* __restrict__ dist, uint32_t d,
                                                           const uint32_t* __restrict__ nodes, uint32_t* fwd, uint32_t* det_out, uint32_t* cnt_out,
                                                           uint32_t* kw_out, uint32_t term_slots, uint32_t uset_slots, uint32_t map_slots) {
    extern __shared__ __align__(16) char smem[];
    const PruneLds L(term_slots, uset_slots, map_slots, K);
    uint2* tab = reinterpret_cast<uint2*>(smem + L.tab);
    uint2* idmap = reinterpret_cast<uint2*>(smem + L.idmap);
    uint32_t* uset = reinterpret_cast<uint32_t*>(smem + L.uset);
    uint32_t* nb_id = reinterpret_cast<uint32_t*>(smem + L.nb_id);
    float* nb_dist = reinterpret_cast<float*>(smem + L.nb_dist);
    uint32_t* det = reinterpret_cast<uint32_t*>(smem + L.det);
    uint32_t* cid = reinterpret_cast<uint32_t*>(smem + L.cid);
    uint32_t* cdet = reinterpret_cast<uint32_t*>(smem + L.cdet);
    uint32_t* sel_id = reinterpret_cast<uint32_t*>(smem + L.sel_id);
    uint32_t* sel_det = reinterpret_cast<uint32_t*>(smem + L.sel_det);
    volatile uint32_t* sel_live = reinterpret_cast<volatile uint32_t*>(smem + L.sel_live);
    uint32_t* sel_kw = reinterpret_cast<uint32_t*>(smem + L.sel_kw);
    uint32_t* o_fwd = reinterpret_cast<uint32_t*>(smem + L.o_fwd);
    uint32_t* o_det = reinterpret_cast<uint32_t*>(smem + L.o_det);
    uint32_t* o_kw = reinterpret_cast<uint32_t*>(smem + L.o_kw);
    volatile uint32_t* ctl = reinterpret_cast<volatile uint32_t*>(smem + L.ctl);

    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id();
    const uint32_t u = nodes ? nodes[blockIdx.x] : blockIdx.x, tmask = term_slots - 1, umask = uset_slots - 1, mmask = map_slots - 1;
    const size_t base = (size_t)u * K;
    const uint64_t lane_lt = (1ull << lane) - 1;

    for (uint32_t i = tid; i < map_slots; i += PR_THREADS) idmap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < uset_slots; i += PR_THREADS) uset[i] = EMPTY;
    for (uint32_t i = tid; i < K; i += PR_THREADS) det[i] = 0;
    if (tid < 16) ctl[tid] = 0;
    __syncthreads();

    // valid list entries, in list order
    if (wave == 0) {
        uint32_t m = 0;
        for (uint32_t b0 = 0; b0 < K; b0 += WAVE) {
            const uint32_t v = ids[base + b0 + lane] & ~FLAG;
            const float dv = dist[base + b0 + lane];
            const bool ok = dv < INF_DIS && v < C.n && v != u;
            const uint64_t b = __ballot(ok);
            if (ok) {
                const uint32_t pos = m + __popcll(b & lane_lt);
                nb_id[pos] = v;
                nb_dist[pos] = dv;
            }
            m += __popcll(b);
        }
        if (lane == 0) ctl[PC_M] = m;
    }
    {   // u's BM25 terms
        const uint64_t du = C.desc[u];
        const Pairs sp = record_pairs(C, du);
        const uint32_t ns = desc_nnz_s(du), nb = desc_nnz_b(du);
        for (uint32_t j = tid; j < nb; j += PR_THREADS) {
            const uint32_t key = sp.key(ns + j);
            uint32_t h = term_hash(key, umask);
            while (true) {
                const uint32_t old = atomicCAS(&uset[h], EMPTY, key);
                if (old == EMPTY || old == key) break;
                h = (h + 1) & umask;
            }
        }
    }
    __syncthreads();
    const uint32_t m = ctl[PC_M];

    // (a) detour counts
    for (uint32_t i = tid; i < m; i += PR_THREADS) {
        const uint32_t key = nb_id[i];
        uint32_t h = term_hash(key, mmask);
        while (true) {
            const uint32_t old = atomicCAS(&idmap[h].x, EMPTY, key);
            if (old == EMPTY) { idmap[h].y = i; break; }
            if (old == key) break;
            h = (h + 1) & mmask;
        }
    }
    __syncthreads();
    for (uint32_t t = tid; t < m * K; t += PR_THREADS) {
        const uint32_t r = t / K, j = t % K;
        const size_t at = (size_t)nb_id[r] * K + j;
        const uint32_t x = ids[at] & ~FLAG;
        const float dx = dist[at];
        uint32_t h = term_hash(x, mmask);
        while (true) {
            const uint2 e = idmap[h];
            if (e.x == x) {
                if (e.y > r && dx < nb_dist[e.y]) atomicAdd(&det[e.y], 1u);
                break;
            }
            if (e.x == EMPTY) break;
            h = (h + 1) & mmask;
        }
    }
    __syncthreads();
    // (b) stable order by detour count
    for (uint32_t i = tid; i < m; i += PR_THREADS) {
        const uint32_t key = (det[i] << 16) | i;
        uint32_t r = 0;
        for (uint32_t j = 0; j < m; j++) r += ((det[j] << 16) | j) < key;
        cid[r] = nb_id[i];
        cdet[r] = det[i];
    }
    if (tid == 0 && m > 0) ctl[PC_ALLFLAG] = 1;
    __syncthreads();
    if (tid == 0 && m > 0) {
        sel_id[0] = cid[0];
        sel_det[0] = cdet[0];
        sel_live[0] = 1;
        sel_kw[0] = 0;
        ctl[PC_NSEL] = 1;
    }
    __syncthreads();

    // (c)+(d) sequential selection
    for (uint32_t t = 1; t < m; t++) {
        const uint32_t c = cid[t];
        term_table_clear(tab, term_slots, tid, PR_THREADS);
        __syncthreads();
        const uint64_t dc = C.desc[c];
        const char* rec = C.recs + desc_off(dc) * 16;
        PivotDense pv;
        pivot_dense_load(pv, reinterpret_cast<const float*>(rec), 1.0f);
        pivot_terms_from_record(tab, tmask, record_pairs(C, dc), tid, PR_THREADS);
        __syncthreads();
        const uint32_t n_sel = ctl[PC_NSEL];
        const float norm_c = norms[c];
        for (uint32_t i = wave; i < n_sel; i += PR_THREADS / WAVE) {
            if (!sel_live[i]) continue;
            const uint32_t s = uniform(sel_id[i]);
            bool kwf = false;
            EvalOut e = eval_wave<true>(C, s, pv, tab, tmask, ALL_PATHS, dense_mul, uset, umask, &kwf);
            if (lane == 0) {
                if (norm_c < e.ip) ctl[PC_REJECT] = 1;
                if (norms[s] < e.ip) sel_live[i] = 0;
                if (!kwf) ctl[PC_ALLFLAG] = 0;
            }
        }
        __syncthreads();
        if (tid == 0) {
            if (!ctl[PC_REJECT]) {
                sel_id[n_sel] = c;
                sel_det[n_sel] = cdet[t];
                sel_live[n_sel] = 1;
                sel_kw[n_sel] = ctl[PC_ALLFLAG];
                ctl[PC_NSEL] = n_sel + 1;
            }
            ctl[PC_REJECT] = 0;
            ctl[PC_ALLFLAG] = 1;
        }
        __syncthreads();
    }

    // (e) emit
    if (tid == 0) {
        const uint32_t n_sel = ctl[PC_NSEL];
        uint32_t cnt = 0, nkw = 0;
        for (uint32_t i = 0; i < n_sel; i++) {
            if (!sel_live[i]) continue;
            if (cnt < d) { o_fwd[cnt] = sel_id[i]; o_det[cnt] = sel_det[i]; cnt++; }
            else if (sel_kw[i] && nkw < APOE_KW_CAND) { o_kw[1 + nkw] = sel_id[i]; nkw++; }
        }
        for (uint32_t t = 0; t < m && cnt < d; t++) {
            const uint32_t c = cid[t];
            bool present = false;
            for (uint32_t j = 0; j < cnt; j++) present |= o_fwd[j] == c;
            if (!present) { o_fwd[cnt] = c; o_det[cnt] = cdet[t]; cnt++; }
        }
        ctl[PC_CNT] = cnt;
        for (; cnt < d; cnt++) { o_fwd[cnt] = u; o_det[cnt] = EMPTY; }
        o_kw[0] = nkw;
        for (uint32_t j = nkw; j < APOE_KW_CAND; j++) o_kw[1 + j] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < d; i += PR_THREADS) {
        fwd[(size_t)u * d + i] = o_fwd[i];
        det_out[(size_t)u * d + i] = o_det[i];
    }
    for (uint32_t i = tid; i < 1 + APOE_KW_CAND; i += PR_THREADS) kw_out[(size_t)u * (1 + APOE_KW_CAND) + i] = o_kw[i];
    if (tid == 0) cnt_out[u] = ctl[PC_CNT];
}

// ---- keys in an LDS map of (key, value) words, open addressing ----

__device__ __forceinline__ void lds_map_insert(uint2* map, uint32_t mask, uint32_t key, uint32_t val) { // a key that is there keeps its value
    uint32_t h = term_hash(key, mask);
    while (true) {
        const uint32_t old = atomicCAS(&map[h].x, EMPTY, key);
        if (old == EMPTY) { map[h].y = val; return; }
        if (old == key) return;
        h = (h + 1) & mask;
    }
}
// The entries of N keys (EMPTY: none): e[k].x == key[k] where it is found. The first slots of all keys are read before any is
// compared, then the second ones of those that met another key, and so on: as many LDS round trips as the longest chain, not N times that.
template <int N>
__device__ __forceinline__ void lds_map_find(const uint2* map, uint32_t mask, const uint32_t (&key)[N], uint2 (&e)[N]) {
    uint32_t h[N];
#pragma unroll
    for (int k = 0; k < N; k++) {
        h[k] = term_hash(key[k], mask);
        e[k] = map[h[k]];
    }
    while (true) {
        bool more = false;
#pragma unroll
        for (int k = 0; k < N; k++) {
            const bool go = e[k].x != key[k] && e[k].x != EMPTY && key[k] != EMPTY;
            h[k] = (h[k] + 1) & mask;
            if (go) e[k] = map[h[k]];
            more |= go;
        }
        if (__ballot(more) == 0) break;
    }
}

// ---- the prune where bounds settle it ----
//
// The selection (below) asks of two neighbours c and s of a node only whether <c, s> exceeds either one's norm. |<c, s>_dense - the
// product of the sketches| has a bound (apoe_device.h), |<c, s>_sparse| is at most the product of the two sparse norms; on a corpus
// whose dense rows have neighbours that answers all pairs of most nodes (100 000 docs, dense_mul 49: 86 of 100), and neither a dense row nor a
// pair of terms but the keys of the BM25 terms is read. A node with an open pair sets open[u] = NODE_OPEN, one with a norm that is not finite NODE_TABLE, and
// leaves nothing else.
// Small in LDS and registers, so that many nodes share a CU: it is a chain of short phases (five nodes of 64 rows a CU;
// 100 000 docs 3.8 ms, with the 14 000 open nodes behind it 6.0 ms, where Gram matrices and selection took 25.4; 30 011 docs K = 128 28.9 -> 10.4 ms).
template <uint32_t K>
struct BoundLds {
    uint32_t stage, row, F, above, below, rowptr, rownnz, idmap, umap, R, nb_id, nb_dist, nrm, det, order, o_fwd, o_det, o_kw, ctl, total;
    __host__ __device__ BoundLds(uint32_t umap_slots, uint32_t map_slots, uint32_t words) {
        uint32_t o = 0;
        // the sketches, a quarter of the dimensions at a time; then what the later phases need
        stage = o;
        idmap = o; o += map_slots * 8;
        umap = o; o += umap_slots * 8;
        R = o; o += K * words * 4;
        o = (o + 7) & ~7u;
        F = o; o += K * (K / 8);
        if (o < K * (SKETCH_BYTES / 4)) o = K * (SKETCH_BYTES / 4);
        row = o; o += K * 16;
        above = o; o += K * (K / 8);
        below = o; o += K * (K / 8);
        rowptr = o; o += K * 8;
        rownnz = o; o += K * 4;
        nb_id = o; o += K * 4;
        nb_dist = o; o += K * 4;
        nrm = o; o += K * 4;
        det = o; o += K * 4;
        order = o; o += K * 4;
        o_fwd = o; o += WAVE * 4;
        o_det = o; o += WAVE * 4;
        o_kw = o; o += (1 + APOE_KW_CAND) * 4;
        ctl = o; o += 16 * 4;
        total = o;
    }
};
typedef int intx4 __attribute__((ext_vector_type(4)));
template <uint32_t K, bool NARROW>
__global__ __launch_bounds__(K * 4) __attribute__((amdgpu_waves_per_eu(4, 8))) void prune_bound_kernel(CorpusView C, float dense_mul, const float* __restrict__ norms,
                                                               const uint32_t* __restrict__ ids, const float* __restrict__ dist, uint32_t d, uint32_t* fwd,
                                                               uint32_t* det_out, uint32_t* cnt_out, uint32_t* kw_out, uint32_t umap_slots, uint32_t map_slots,
                                                               uint32_t words, const SketchMeta* __restrict__ sketch_meta, const uint4* __restrict__ sketch,
                                                               uint32_t* open) {
    constexpr int NT = K * 4, NWAVES = NT / WAVE, KL = K / WAVE;
    constexpr int OWN = K / NWAVES; // rows a wave looks after: wave, wave + NWAVES, ...
    static_assert(OWN == 16, "two batches of eight rows");
    C.narrow = NARROW ? 1u : 0u;
    extern __shared__ __align__(16) char smem[];
    const BoundLds<K> L(umap_slots, map_slots, words);
    intx4* stage = reinterpret_cast<intx4*>(smem + L.stage);
    uint2* idmap = reinterpret_cast<uint2*>(smem + L.idmap);
    uint2* umap = reinterpret_cast<uint2*>(smem + L.umap);
    uint32_t* R = reinterpret_cast<uint32_t*>(smem + L.R);
    uint64_t* F = reinterpret_cast<uint64_t*>(smem + L.F); // [K][KL], as above and below
    uint64_t* above = reinterpret_cast<uint64_t*>(smem + L.above);
    uint64_t* below = reinterpret_cast<uint64_t*>(smem + L.below);
    float4* row = reinterpret_cast<float4*>(smem + L.row); // dense norm, scale and error of the sketch, bound of the norm of the sparse part
    unsigned long long* rowptr = reinterpret_cast<unsigned long long*>(smem + L.rowptr);
    uint32_t* rownnz = reinterpret_cast<uint32_t*>(smem + L.rownnz);
    uint32_t* nb_id = reinterpret_cast<uint32_t*>(smem + L.nb_id);
    float* nb_dist = reinterpret_cast<float*>(smem + L.nb_dist);
    float* nrm = reinterpret_cast<float*>(smem + L.nrm);
    uint32_t* det = reinterpret_cast<uint32_t*>(smem + L.det);
    uint32_t* order = reinterpret_cast<uint32_t*>(smem + L.order);
    uint32_t* o_fwd = reinterpret_cast<uint32_t*>(smem + L.o_fwd);
    uint32_t* o_det = reinterpret_cast<uint32_t*>(smem + L.o_det);
    uint32_t* o_kw = reinterpret_cast<uint32_t*>(smem + L.o_kw);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(smem + L.ctl);

    const int tid = threadIdx.x, wave = (int)uniform(tid / WAVE), lane = lane_id();
    const uint32_t u = blockIdx.x, umask = umap_slots - 1, mmask = map_slots - 1;
    const size_t base = (size_t)u * K;
    const uint64_t lane_lt = (1ull << lane) - 1;

    for (uint32_t i = tid; i < K * KL; i += NT) above[i] = below[i] = 0;
    for (uint32_t i = tid; i < K; i += NT) det[i] = 0;
    if (tid < 16) ctl[tid] = 0;
    // valid list entries, in list order
    if (wave == 0) {
        uint32_t m = 0;
#pragma unroll
        for (int q = 0; q < KL; q++) {
            const uint32_t v = ids[base + q * WAVE + lane] & ~FLAG;
            const float dv = dist[base + q * WAVE + lane];
            const bool ok = dv < INF_DIS && v < C.n && v != u;
            const uint64_t b = __ballot(ok);
            if (ok) {
                const uint32_t pos = m + __popcll(b & lane_lt);
                nb_id[pos] = v;
                nb_dist[pos] = dv;
            }
            m += __popcll(b);
        }
        if (lane == 0) ctl[PC_M] = m;
    }
    __syncthreads();
    const uint32_t m = uniform(ctl[PC_M]);
    // the code products of all pairs: 16 x 16 blocks (bi <= bj), dealt out to the waves; a quarter of the dimensions is staged while the
    // next one is on its way. Lane (j, g), j = lane % 16, g = lane / 16, supplies codes 64 b + 16 g .. of row j of a block and holds row 4 g + e, column j
    constexpr int NB = K / 16, BLOCKS = NB * (NB + 1) / 2, PER = (BLOCKS + NWAVES - 1) / NWAVES;
    constexpr uint32_t UNITS = SKETCH_BYTES / 4 / 16; // 16-byte units of a row in a quarter
    const int j = lane & 15, g = lane >> 4;
    uint32_t bi[PER], bj[PER]; // wave-uniform; bj = NB: none
    intx4 acc[PER];
#pragma unroll
    for (int q = 0; q < PER; q++) {
        uint32_t t = wave + q * NWAVES, i = 0;
        while (i < NB && t >= NB - i) { t -= NB - i; i++; }
        bi[q] = uniform(i);
        bj[q] = uniform(i < NB ? i + t : (uint32_t)NB);
        acc[q] = intx4{0, 0, 0, 0};
    }
    if (m > 0) {
        constexpr int LOADS = K * UNITS / NT;
        const intx4* from[LOADS]; // rows that are not there: the last one again
        intx4 ahead[LOADS];
#pragma unroll
        for (int k = 0; k < LOADS; k++) {
            const uint32_t i = tid + k * NT;
            from[k] = reinterpret_cast<const intx4*>(sketch) + (size_t)nb_id[min(i / UNITS, m - 1)] * (SKETCH_BYTES / 16) + i % UNITS;
            ahead[k] = from[k][0];
        }
        if (tid < (int)m) { // meanwhile: what the tests and the later phases need of a row
            const uint32_t v = nb_id[tid];
            const uint64_t desc = C.desc[v];
            const float nv = norms[v], dn = C.dnorm[v];
            const SketchMeta sm = sketch_meta[v];
            nrm[tid] = nv;
            if (!(nv < __builtin_inff())) ctl[PC_OPEN] = ctl[PC_TABLE] = 1;
            // what the hybrid norm leaves to the sparse part, with room for the rounding of both norms
            row[tid] = make_float4(dn, sm.scale, sm.err, sqrtf(fmaxf(nv - dense_mul * dn * dn, 0.f) + 1e-5f * (nv + dense_mul * dn * dn)));
            rowptr[tid] = desc_off(desc) * 16 + DENSE_BYTES;
            rownnz[tid] = (desc_nnz_s(desc) + desc_nnz_b(desc)) | (desc_nnz_s(desc) << 16);
        }
        // On a corpus whose pairs decide, the longest rows sit in every list, and next to a shorter one the product of the sparse norms tells
        // nothing: if even the largest dense part cannot take a pair out of reach of the smaller norm, the node is open without a look at
        // the sketches (100 000 i.i.d. docs, where all are: 0.2 ms instead of 3.5).
        __syncthreads();
        if (wave == 0) {
            float longest = 0.f, top_dense = 0.f;
#pragma unroll
            for (int q = 0; q < KL; q++) {
                const float4 x = q * WAVE + (uint32_t)lane < m ? row[q * WAVE + lane] : make_float4(0.f, 0.f, 0.f, 0.f);
                longest = fmaxf(longest, x.w);
                top_dense = fmaxf(top_dense, x.x);
            }
            longest = -wave_min_dpp(-longest);
            top_dense = -wave_min_dpp(-top_dense);
#pragma unroll
            for (int q = 0; q < KL; q++) {
                const uint32_t i = q * WAVE + lane;
                // the row of the longest sparse part is not compared with itself
                const float dense = i < m ? row[i].x : 0.f;
                if (i < m && row[i].w < longest && longest * row[i].w - dense_mul * dense * top_dense > nrm[i]) ctl[PC_OPEN] = 1;
            }
        }
        __syncthreads();
        if (uniform(ctl[PC_OPEN])) {
            if (tid == 0) open[u] = ctl[PC_TABLE] ? NODE_TABLE : NODE_OPEN;
            return;
        }
#pragma unroll 1
        for (uint32_t quarter = 0; quarter < 4; quarter++) {
            if (quarter) __syncthreads();
#pragma unroll
            for (int k = 0; k < LOADS; k++) {
                const uint32_t i = tid + k * NT, r = i / UNITS, c = i % UNITS;
                stage[r * UNITS + (c ^ (r & (UNITS - 1)))] = ahead[k];
            }
            __syncthreads();
            if (quarter < 3) {
#pragma unroll
                for (int k = 0; k < LOADS; k++) ahead[k] = from[k][(quarter + 1) * UNITS];
            }
#pragma unroll
            for (int q = 0; q < PER; q++) {
                if (16 * bj[q] < m) { // wave-uniform; a block that is not there starts at K >= m
                    const uint32_t ra = min(16 * bi[q] + (uint32_t)j, m - 1), rb = min(16 * bj[q] + (uint32_t)j, m - 1);
#pragma unroll
                    for (int k = 0; k < (int)UNITS / 4; k++) {
                        const uint32_t c = 4 * k + g;
                        const intx4 a = stage[ra * UNITS + (c ^ (ra & (UNITS - 1)))], b = stage[rb * UNITS + (c ^ (rb & (UNITS - 1)))];
                        acc[q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, acc[q], 0, 0, 0);
                    }
                }
            }
        }
    }
    bool undecided = false;
#pragma unroll
    for (int q = 0; q < PER; q++) {
        if (16 * bj[q] < m) {
            const uint32_t c = 16 * bj[q] + j;
            const float4 rc = c < m ? row[c] : make_float4(0.f, 0.f, 0.f, 0.f);
            const float nc = c < m ? nrm[c] : 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const uint32_t r = 16 * bi[q] + 4 * g + e;
                if (r < c && c < m) {
                    const float4 rr = row[r];
                    const float nr = nrm[r];
                    const float p = dense_mul * ((float)acc[q][e] * (rr.y * rc.y));
                    const float off = dense_mul * (rr.x * rc.z + rr.z * (rc.x + rc.z)) + rr.w * rc.w + 1e-5f * (dense_mul * rr.x * rc.x + rr.w * rc.w + 1.0f);
                    undecided |= !(fabsf(p - nr) > off && fabsf(p - nc) > off); // not a number: open
                    auto set = [&](uint64_t* masks, uint32_t of, uint32_t bit) { atomicOr(reinterpret_cast<uint32_t*>(masks) + of * (2 * KL) + (bit >> 5), 1u << (bit & 31)); };
                    if (nr < p) { set(above, r, c); set(below, c, r); }
                    if (nc < p) { set(above, c, r); set(below, r, c); }
                }
            }
        }
    }
    if (undecided) ctl[PC_OPEN] = 1;
    __syncthreads();
    if (uniform(ctl[PC_OPEN])) {
        if (tid == 0) open[u] = NODE_OPEN;
        return;
    }
    // the staged sketches make room
    for (uint32_t i = tid; i < map_slots; i += NT) idmap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < umap_slots; i += NT) umap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < K * words; i += NT) R[i] = 0;
    __syncthreads();
    if (tid < (int)m) lds_map_insert(idmap, mmask, nb_id[tid], tid);
    {   // u's BM25 terms -> index
        const uint64_t du = C.desc[u];
        const Pairs sp = record_pairs(C, du);
        const uint32_t ns = desc_nnz_s(du), nb = desc_nnz_b(du);
        for (uint32_t i = tid; i < nb; i += NT) lds_map_insert(umap, umask, sp.key(ns + i), i);
    }
    __syncthreads();
    // (a) detour counts, eight list entries of a thread at a time
#pragma unroll 1
    for (uint32_t t0 = 0; t0 < m * K; t0 += 8 * NT) {
        uint32_t xs[8];
        float dxs[8];
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t t = t0 + tid + k * NT;
            xs[k] = EMPTY;
            dxs[k] = 0.f;
            if (t < m * K) {
                const size_t at = (size_t)nb_id[t / K] * K + t % K;
                xs[k] = ids[at] & ~FLAG;
                dxs[k] = dist[at];
            }
        }
        uint2 e[8];
        lds_map_find(idmap, mmask, xs, e);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t r = (t0 + tid + k * NT) / K;
            if (xs[k] != EMPTY && e[k].x == xs[k] && e[k].y > r && dxs[k] < nb_dist[e[k].y]) atomicAdd(&det[e[k].y], 1u);
        }
    }
    // R[r] = bits of u's BM25 terms that row r holds too: one wave per row, the first 64 BM25 terms of eight rows at a time
#pragma unroll 1
    for (int half = 0; half < 2; half++) {
        uint32_t key[8], nbs[8];
        auto row_pairs = [&](uint32_t r) {
            Pairs sp = gram_row(C, rowptr, rownnz, r);
            sp.narrow = NARROW ? 1u : 0u;
            return sp;
        };
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t r = wave + NWAVES * (8 * half + k);
            nbs[k] = 0;
            key[k] = EMPTY;
            if (r < m) { // wave-uniform
                const Pairs sp = row_pairs(r);
                nbs[k] = uniform(sp.nnz - sp.ns);
                if ((uint32_t)lane < nbs[k]) key[k] = sp.raw(sp.ns + lane).x; // the path bit follows where the key is used
            }
        }
        uint2 e[8];
#pragma unroll
        for (int k = 0; k < 8; k++) key[k] |= BM25_BIT;
        lds_map_find(umap, umask, key, e);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            const uint32_t r = wave + NWAVES * (8 * half + k);
            if (key[k] != EMPTY && e[k].x == key[k]) atomicOr(&R[r * words + (e[k].y >> 5)], 1u << (e[k].y & 31));
            if (nbs[k] > WAVE) {
                const Pairs sp = row_pairs(r);
                for (uint32_t i = WAVE + lane; i < nbs[k]; i += WAVE) {
                    const uint32_t x[1] = {sp.key(sp.ns + i)};
                    uint2 f[1];
                    lds_map_find(umap, umask, x, f);
                    if (f[0].x == x[0]) atomicOr(&R[r * words + (f[0].y >> 5)], 1u << (f[0].y & 31));
                }
            }
        }
    }
    __syncthreads();
    // (b) stable order by detour count: the last wave; keyword flags of all pairs: flag(c, s) = (R[s] & ~R[c]) != 0, lane s for one c at a time
    if (wave == NWAVES - 1) {
        uint32_t key[KL], rank[KL];
#pragma unroll
        for (int q = 0; q < KL; q++) {
            const uint32_t i = q * WAVE + lane;
            key[q] = i < m ? (det[i] << 16) | i : ~0u;
            rank[q] = 0;
        }
#pragma unroll
        for (int q = 0; q < KL; q++) {
            for (uint32_t i = 0; i < WAVE && q * WAVE + i < m; i++) {
                const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)key[q], (int)i);
#pragma unroll
                for (int p = 0; p < KL; p++) rank[p] += x < key[p];
            }
        }
#pragma unroll
        for (int q = 0; q < KL; q++)
            if (q * WAVE + (uint32_t)lane < m) order[rank[q]] = q * WAVE + lane;
    }
    for (uint32_t c = wave; c < m; c += NWAVES) {
#pragma unroll
        for (int q = 0; q < KL; q++) {
            const uint32_t s = q * WAVE + lane;
            uint32_t any = 0;
            for (uint32_t w = 0; w < words; w++) any |= (s < m ? R[s * words + w] : 0u) & ~R[c * words + w];
            const uint64_t f = __ballot(any != 0);
            if (lane == 0) F[c * KL + q] = f;
        }
    }
    __syncthreads();
    // (c)+(d) sequential selection as in prune_gram_kernel: position 64 q + lane of the order in register q
    if (wave == 0) {
        uint32_t ord[KL], id_o[KL], det_o[KL];
        uint64_t up[KL][KL], dn[KL][KL], fl[KL][KL], live[KL] = {}, taken[KL] = {}, flagged[KL] = {};
        bool plain = true;
#pragma unroll
        for (int q = 0; q < KL; q++) {
            const uint32_t t = q * WAVE + lane;
            ord[q] = t < m ? order[t] : 0u;
            id_o[q] = t < m ? nb_id[ord[q]] : EMPTY;
            det_o[q] = t < m ? det[ord[q]] : 0u;
#pragma unroll
            for (int w = 0; w < KL; w++) {
                up[q][w] = t < m ? above[ord[q] * KL + w] : 0ull;
                dn[q][w] = t < m ? below[ord[q] * KL + w] : 0ull;
                fl[q][w] = t < m ? F[ord[q] * KL + w] : 0ull;
                plain = plain && (up[q][w] | dn[q][w]) == 0;
            }
        }
        plain = __ballot(!plain) == 0; // no product exceeds a norm: all are taken and stay
#pragma unroll
        for (int q = 0; q < KL; q++) {
            for (uint32_t i = 0; i < WAVE && q * WAVE + i < m; i++) {
                const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)ord[q], (int)i);
                bool reject = false, allflag = q * WAVE + i > 0;
#pragma unroll
                for (int w = 0; w < KL; w++) {
                    allflag = allflag && (live[w] & ~readlane64(fl[q][w], i)) == 0;
                    if (!plain) {
                        reject = reject || (readlane64(up[q][w], i) & live[w]) != 0;
                    }
                }
                if (!plain) {
#pragma unroll
                    for (int w = 0; w < KL; w++) live[w] &= ~readlane64(dn[q][w], i);
                }
                if (!reject) {
#pragma unroll
                    for (int w = 0; w < KL; w++) live[w] |= (c >> 6) == (uint32_t)w ? 1ull << (c & 63) : 0ull;
                    taken[q] |= 1ull << i;
                    if (allflag) flagged[q] |= 1ull << i;
                }
            }
        }
        // (e) emit: live members in selection order fill the row, flagged ones beyond d become keyword candidates
        bool alive[KL];
        uint64_t lb[KL];
        uint32_t n_live = 0, n_kw = 0;
#pragma unroll
        for (int q = 0; q < KL; q++) {
            uint64_t lw = live[0];
#pragma unroll
            for (int w = 1; w < KL; w++) lw = (ord[q] >> 6) == (uint32_t)w ? live[w] : lw;
            alive[q] = ((taken[q] >> lane) & 1) && ((lw >> (ord[q] & 63)) & 1);
            lb[q] = __ballot(alive[q]);
            const uint32_t pos = n_live + __popcll(lb[q] & lane_lt);
            if (alive[q] && pos < d) { o_fwd[pos] = id_o[q]; o_det[pos] = det_o[q]; }
            const bool kwc = alive[q] && pos >= d && ((flagged[q] >> lane) & 1);
            const uint64_t kb = __ballot(kwc);
            const uint32_t kpos = n_kw + __popcll(kb & lane_lt);
            if (kwc && kpos < APOE_KW_CAND) o_kw[1 + kpos] = id_o[q];
            n_live += __popcll(lb[q]);
            n_kw += __popcll(kb);
        }
        uint32_t cnt = min(n_live, d);
        const uint32_t nkw = min(n_kw, (uint32_t)APOE_KW_CAND);
        if (cnt < d) { // fewer survivors than the row has slots: the remaining neighbours in order, each id once
            bool add[KL];
#pragma unroll
            for (int q = 0; q < KL; q++) add[q] = q * WAVE + (uint32_t)lane < m;
#pragma unroll
            for (int p = 0; p < KL; p++) {
                for (uint64_t rest = lb[p]; rest; rest &= rest - 1) {
                    const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)id_o[p], __builtin_ctzll(rest));
#pragma unroll
                    for (int q = 0; q < KL; q++) add[q] = add[q] && x != id_o[q];
                }
                for (uint32_t i = 0; i < WAVE && p * WAVE + i < m; i++) {
                    const uint32_t x = (uint32_t)__builtin_amdgcn_readlane((int)id_o[p], (int)i);
#pragma unroll
                    for (int q = 0; q < KL; q++) add[q] = add[q] && !(q * WAVE + (uint32_t)lane > p * WAVE + i && x == id_o[q]);
                }
            }
#pragma unroll
            for (int q = 0; q < KL; q++) {
                const uint64_t ab = __ballot(add[q]);
                const uint32_t at = cnt + __popcll(ab & lane_lt);
                if (add[q] && at < d) { o_fwd[at] = id_o[q]; o_det[at] = det_o[q]; }
                cnt = min(d, cnt + (uint32_t)__popcll(ab));
            }
        }
        if (lane == 0) { ctl[PC_CNT] = cnt; o_kw[0] = nkw; }
        for (uint32_t i = cnt + lane; i < d; i += WAVE) { o_fwd[i] = u; o_det[i] = EMPTY; }
        for (uint32_t i = nkw + lane; i < APOE_KW_CAND; i += WAVE) o_kw[1 + i] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < d; i += NT) {
        fwd[(size_t)u * d + i] = o_fwd[i];
        det_out[(size_t)u * d + i] = o_det[i];
    }
    for (uint32_t i = tid; i < 1 + APOE_KW_CAND; i += NT) kw_out[(size_t)u * (1 + APOE_KW_CAND) + i] = o_kw[i];
    if (tid == 0) cnt_out[u] = ctl[PC_CNT];
}

// ---- the prune on a Gram matrix that the tile kernel of join.hip has left in memory (lists of up to 128 entries) ----

constexpr uint32_t PS_MAX = 128;            // longest list
constexpr int PS_THREADS = 256;

struct SelectLds {
    uint32_t F, rdesc, idmap, umap, R, nb_id, nb_dist, nrm, det, order, o_fwd, o_det, o_kw, ctl, total;
    __host__ __device__ SelectLds(uint32_t umap_slots, uint32_t map_slots, uint32_t words) {
        uint32_t o = 0;
        F = o; o += PS_MAX * (PS_MAX / 32) * 4; // keyword-flag matrix: bit s of row c = "s holds a term of u that c lacks"
        o = (o + 7) & ~7u;
        rdesc = o; o += PS_MAX * 8;             // descriptors of the rows
        idmap = o; o += map_slots * 8;
        umap = o; o += umap_slots * 8;
        R = o; o += PS_MAX * words * 4;
        nb_id = o; o += PS_MAX * 4;
        nb_dist = o; o += PS_MAX * 4;
        nrm = o; o += PS_MAX * 4;
        det = o; o += PS_MAX * 4;
        order = o; o += PS_MAX * 4;
        o_fwd = o; o += PS_MAX * 4;
        o_det = o; o += PS_MAX * 4;
        o_kw = o; o += (1 + APOE_KW_CAND) * 4;
        ctl = o; o += 16 * 4;
        total = o;
    }
};

// allan_poe (index.cu:539-714) for node u = nodes[node0 + blockIdx.x], as prune_kernel, with every inner product <c, s> read from the
// node's Gram matrix gram[blockIdx.x][i][j] (i <= j: positions in the list of valid entries) instead of being evaluated:
// detour counts and the (detour, rank) order as there; the keyword flag of a pair from bit masks R[i] = the BM25 terms of u
// that row i holds (flag(c, s) = R[s] has a bit that R[c] lacks); the sequential selection by wave 0 alone, two selected
// members per lane (slots `lane` and `lane + 64` of the selection order), every member's product with the NEXT candidate
// requested from the matrix in memory while the current candidate is decided. The workgroup keeps no copy of the matrix:
// several nodes share a CU, and the others cover the selection's waits.
__global__ __launch_bounds__(PS_THREADS) void prune_select_kernel(CorpusView C, const float* __restrict__ norms, uint32_t K, const uint32_t* __restrict__ ids,
                                                                  const float* __restrict__ dist, uint32_t d, const uint32_t* __restrict__ nodes, uint32_t node0, const float* __restrict__ gram,
                                                                  uint32_t* fwd, uint32_t* det_out, uint32_t* cnt_out, uint32_t* kw_out, uint32_t umap_slots,
                                                                  uint32_t map_slots, uint32_t words) {
    extern __shared__ __align__(16) char smem[];
    const SelectLds L(umap_slots, map_slots, words);
    uint32_t* F = reinterpret_cast<uint32_t*>(smem + L.F);
    uint64_t* rdesc = reinterpret_cast<uint64_t*>(smem + L.rdesc);
    uint2* idmap = reinterpret_cast<uint2*>(smem + L.idmap);
    uint2* umap = reinterpret_cast<uint2*>(smem + L.umap);
    uint32_t* R = reinterpret_cast<uint32_t*>(smem + L.R);
    uint32_t* nb_id = reinterpret_cast<uint32_t*>(smem + L.nb_id);
    float* nb_dist = reinterpret_cast<float*>(smem + L.nb_dist);
    float* nrm = reinterpret_cast<float*>(smem + L.nrm);
    uint32_t* det = reinterpret_cast<uint32_t*>(smem + L.det);
    uint32_t* order = reinterpret_cast<uint32_t*>(smem + L.order);
    uint32_t* o_fwd = reinterpret_cast<uint32_t*>(smem + L.o_fwd);
    uint32_t* o_det = reinterpret_cast<uint32_t*>(smem + L.o_det);
    uint32_t* o_kw = reinterpret_cast<uint32_t*>(smem + L.o_kw);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(smem + L.ctl);

    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id();
    constexpr uint32_t NWV = PS_THREADS / WAVE;
    const uint32_t u = nodes[node0 + blockIdx.x], umask = umap_slots - 1, mmask = map_slots - 1;
    const size_t base = (size_t)u * K;
    const uint64_t lane_lt = (1ull << lane) - 1;
    const float* gu = gram + (size_t)blockIdx.x * PS_MAX * PS_MAX;

    for (uint32_t i = tid; i < map_slots; i += PS_THREADS) idmap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < umap_slots; i += PS_THREADS) umap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < PS_MAX * words; i += PS_THREADS) R[i] = 0;
    for (uint32_t i = tid; i < PS_MAX; i += PS_THREADS) det[i] = 0;
    if (tid < 16) ctl[tid] = 0;
    __syncthreads();
    // valid list entries, in list order (the rows and columns of the Gram matrix)
    if (wave == 0) {
        uint32_t m = 0;
        for (uint32_t b0 = 0; b0 < K; b0 += WAVE) {
            const uint32_t v = ids[base + b0 + lane] & ~FLAG;
            const float dv = dist[base + b0 + lane];
            const bool ok = dv < INF_DIS && v < C.n && v != u;
            const uint64_t b = __ballot(ok);
            if (ok) {
                const uint32_t pos = m + __popcll(b & lane_lt);
                nb_id[pos] = v;
                nb_dist[pos] = dv;
                nrm[pos] = norms[v];
                rdesc[pos] = C.desc[v];
            }
            m += __popcll(b);
        }
        if (lane == 0) ctl[PC_M] = m;
    }
    {   // u's BM25 terms -> their index in u's row
        const uint64_t du = C.desc[u];
        const Pairs sp = record_pairs(C, du);
        const uint32_t ns = desc_nnz_s(du), nb = desc_nnz_b(du);
        for (uint32_t j = tid; j < nb; j += PS_THREADS) {
            const uint32_t key = sp.key(ns + j);
            uint32_t h = term_hash(key, umask);
            while (true) {
                const uint32_t old = atomicCAS(&umap[h].x, EMPTY, key);
                if (old == EMPTY) { umap[h].y = j; break; }
                if (old == key) break;
                h = (h + 1) & umask;
            }
        }
    }
    __syncthreads();
    const uint32_t m = ctl[PC_M];
    // (a) detour counts
    for (uint32_t i = tid; i < m; i += PS_THREADS) {
        const uint32_t key = nb_id[i];
        uint32_t h = term_hash(key, mmask);
        while (true) {
            const uint32_t old = atomicCAS(&idmap[h].x, EMPTY, key);
            if (old == EMPTY) { idmap[h].y = i; break; }
            if (old == key) break;
            h = (h + 1) & mmask;
        }
    }
    // R[r] = bits of u's BM25 terms that row r holds too: one wave per row, lanes over its BM25 pairs; the first 128 BM25 terms
    // of four rows are requested before the first of them is looked up
    auto mark = [&](uint32_t r, uint32_t key) {
        uint32_t h = term_hash(key, umask);
        while (true) {
            const uint2 e = umap[h];
            if (e.x == key) { atomicOr(&R[r * words + (e.y >> 5)], 1u << (e.y & 31)); break; }
            if (e.x == EMPTY) break;
            h = (h + 1) & umask;
        }
    };
    for (uint32_t r0 = wave; r0 < m; r0 += 4 * NWV) {
        uint32_t key[4][2], nbs[4];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t r = r0 + b * NWV;
            nbs[b] = 0;
            key[b][0] = key[b][1] = EMPTY;
            if (r < m) {
                const uint64_t dr = rdesc[r];
                const Pairs sp = record_pairs(C, dr);
                const uint32_t ns = desc_nnz_s(dr);
                nbs[b] = desc_nnz_b(dr);
                if ((uint32_t)lane < nbs[b]) key[b][0] = sp.key(ns + lane);
                if ((uint32_t)lane + WAVE < nbs[b]) key[b][1] = sp.key(ns + lane + WAVE);
            }
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const uint32_t r = r0 + b * NWV;
            if ((uint32_t)lane < nbs[b]) mark(r, key[b][0]);
            if ((uint32_t)lane + WAVE < nbs[b]) mark(r, key[b][1]);
            if (nbs[b] > 2 * WAVE) { // a longer row: the rest as it comes
                const uint64_t dr = rdesc[r];
                const Pairs sp = record_pairs(C, dr);
                const uint32_t ns = desc_nnz_s(dr);
                for (uint32_t j = 2 * WAVE + lane; j < nbs[b]; j += WAVE) mark(r, sp.key(ns + j));
            }
        }
    }
    __syncthreads();
    // sixteen list entries of this thread are requested before the first of them is looked up
    for (uint32_t t0 = 0; t0 < m * K; t0 += 16 * PS_THREADS) {
        uint32_t xs[16];
        float dxs[16];
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const uint32_t t = t0 + tid + k * PS_THREADS;
            xs[k] = EMPTY;
            dxs[k] = 0.f;
            if (t < m * K) {
                const size_t at = (size_t)nb_id[t / K] * K + t % K;
                xs[k] = ids[at] & ~FLAG;
                dxs[k] = dist[at];
            }
        }
#pragma unroll
        for (int k = 0; k < 16; k++) {
            const uint32_t r = (t0 + tid + k * PS_THREADS) / K, x = xs[k];
            if (x == EMPTY) continue;
            uint32_t h = term_hash(x, mmask);
            while (true) {
                const uint2 e = idmap[h];
                if (e.x == x) {
                    if (e.y > r && dxs[k] < nb_dist[e.y]) atomicAdd(&det[e.y], 1u);
                    break;
                }
                if (e.x == EMPTY) break;
                h = (h + 1) & mmask;
            }
        }
    }
    __syncthreads();
    // (b) stable order by detour count
    for (uint32_t i = tid; i < m; i += PS_THREADS) {
        const uint32_t key = (det[i] << 16) | i;
        uint32_t r = 0;
        for (uint32_t j = 0; j < m; j++) r += ((det[j] << 16) | j) < key;
        order[r] = i;
    }
    // keyword flags of all pairs at once (index.cu:637,651-654): flag(c, s) = (R[s] & ~R[c]) != 0. A thread takes one row c and
    // half of the columns: its own mask stays in registers (the first four words), the lanes of a wave read the same R[s]
    {
        static_assert(PS_THREADS == 2 * PS_MAX && PS_MAX == 128, "one row and two flag words per thread");
        const uint32_t c = tid % PS_MAX, half = tid / PS_MAX;
        uint32_t rc[4];
#pragma unroll
        for (int w = 0; w < 4; w++) rc[w] = (uint32_t)w < words && c < m ? R[c * words + w] : 0u;
#pragma unroll
        for (int q2 = 0; q2 < 2; q2++) {
            const uint32_t q = half * 2 + q2;
            uint32_t word = 0;
            for (uint32_t b = 0; b < 32 && q * 32 + b < m; b++) {
                const uint32_t sidx = q * 32 + b;
                uint32_t any = 0;
#pragma unroll
                for (int w = 0; w < 4; w++)
                    if ((uint32_t)w < words) any |= R[sidx * words + w] & ~rc[w];
                for (uint32_t w = 4; w < words; w++) any |= R[sidx * words + w] & ~(c < m ? R[c * words + w] : 0u);
                word |= (any != 0 ? 1u : 0u) << b;
            }
            F[c * (PS_MAX / 32) + q] = c < m ? word : 0u;
        }
    }
    __syncthreads();
    // (c)+(d) sequential selection, wave 0: member k of the selection order lives in slot k / 64 of lane k % 64; what a step
    // needs of its candidate (Gram index, norm, flag row) is read one step ahead
    if (wave == 0) {
        uint32_t gi[2] = {0, 0}, kw[2] = {0, 0}; // Gram index (position in the list) and keyword flag of the member
        bool live[2] = {false, false};
        float mn[2] = {0.f, 0.f};
        uint32_t n_sel = 0;
        if (m > 0) {
            const uint32_t c0 = order[0];
            if (lane == 0) { gi[0] = c0; live[0] = true; mn[0] = nrm[c0]; }
            n_sel = 1;
        }
        uint32_t c_next = m > 1 ? order[1] : 0u;
        float norm_next = nrm[c_next];
        uint4 f_next = *reinterpret_cast<const uint4*>(&F[c_next * (PS_MAX / 32)]);
        auto product = [&](uint32_t a, uint32_t b) { return gu[(size_t)min(a, b) * PS_MAX + max(a, b)]; };
        float p_next[2] = {0.f, 0.f}; // <member, next candidate>
        if (m > 1 && lane == 0) p_next[0] = product(gi[0], c_next);
        for (uint32_t t = 1; t < m; t++) {
            const uint32_t c = c_next;
            const float norm_c = norm_next;
            const uint4 fc = f_next;
            const float p_cur[2] = {p_next[0], p_next[1]};
            if (t + 1 < m) {
                c_next = order[t + 1];
                norm_next = nrm[c_next];
                f_next = *reinterpret_cast<const uint4*>(&F[c_next * (PS_MAX / 32)]);
#pragma unroll
                for (int s = 0; s < 2; s++) { // also for the slot that c takes if it is accepted
                    const uint32_t slot = (uint32_t)lane + 64u * s;
                    if (slot < n_sel && live[s]) p_next[s] = product(gi[s], c_next);
                    else if (slot == n_sel) p_next[s] = product(c, c_next);
                }
            }
            bool rej = false, noflag = false;
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const bool act = (uint32_t)lane + 64u * s < n_sel && live[s];
                if (act) {
                    const float p = p_cur[s];
                    const uint32_t q = gi[s] >> 5, fw = q == 0 ? fc.x : q == 1 ? fc.y : q == 2 ? fc.z : fc.w;
                    rej |= norm_c < p;
                    if (mn[s] < p) live[s] = false;
                    noflag |= !((fw >> (gi[s] & 31)) & 1u);
                }
            }
            const bool reject = __ballot(rej) != 0;
            const bool allflag = __ballot(noflag) == 0;
            if (!reject) {
#pragma unroll
                for (int s = 0; s < 2; s++) {
                    if ((uint32_t)lane + 64u * s == n_sel) { gi[s] = c; live[s] = true; mn[s] = norm_c; kw[s] = allflag ? 1u : 0u; }
                }
                n_sel++;
            }
        }
        // (e) emit: live members in selection order fill the row, flagged ones beyond d become keyword candidates
        uint32_t seen_live = 0, seen_kw = 0;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const bool lv = (uint32_t)lane + 64u * s < n_sel && live[s];
            const uint64_t lb = __ballot(lv);
            const uint32_t pos = seen_live + __popcll(lb & lane_lt);
            if (lv && pos < d) { o_fwd[pos] = nb_id[gi[s]]; o_det[pos] = det[gi[s]]; }
            const bool kwc = lv && pos >= d && kw[s];
            const uint64_t kb = __ballot(kwc);
            const uint32_t kpos = seen_kw + __popcll(kb & lane_lt);
            if (kwc && kpos < APOE_KW_CAND) o_kw[1 + kpos] = nb_id[gi[s]];
            seen_live += __popcll(lb);
            seen_kw += __popcll(kb);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (lane == 0) {
            uint32_t cnt = min(seen_live, d);
            const uint32_t nkw = min(seen_kw, (uint32_t)APOE_KW_CAND);
            // fewer survivors than the row has slots: the remaining neighbours in order, each id once, then the node itself
            for (uint32_t t = 0; t < m && cnt < d; t++) {
                const uint32_t cidx = order[t], cid = nb_id[cidx];
                bool present = false;
                for (uint32_t j = 0; j < cnt; j++) present |= o_fwd[j] == cid;
                if (!present) { o_fwd[cnt] = cid; o_det[cnt] = det[cidx]; cnt++; }
            }
            ctl[PC_CNT] = cnt;
            for (; cnt < d; cnt++) { o_fwd[cnt] = u; o_det[cnt] = EMPTY; }
            o_kw[0] = nkw;
            for (uint32_t j = nkw; j < APOE_KW_CAND; j++) o_kw[1 + j] = 0;
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < d; i += PS_THREADS) {
        fwd[(size_t)u * d + i] = o_fwd[i];
        det_out[(size_t)u * d + i] = o_det[i];
    }
    for (uint32_t i = tid; i < 1 + APOE_KW_CAND; i += PS_THREADS) kw_out[(size_t)u * (1 + APOE_KW_CAND) + i] = o_kw[i];
    if (tid == 0) cnt_out[u] = ctl[PC_CNT];
}

// ---- gather-once form of the prune (K = 64) ----

constexpr int PRUNE_DENSE_NB = 2; // 8-float blocks of the rows a wave requests ahead of the ones it multiplies
constexpr int GRAM_THREADS = 512; // 8 waves share one node's tables: more lookups in flight per byte of LDS

struct GramPruneLds {
    uint32_t G, tabs, ovf_cnt, rowptr, rownnz, umap, R, F, above, below, row, idmap, nb_id, nb_dist, nrm, det, order, o_fwd, o_det, o_kw, ctl, total;
    // union_slots != 0: the table region holds one union table (apoe_gram.h) instead of tgroup pivot tables;
    // rank_slots != 0: it holds a rank table (apoe_ranktab.h) of rank_bits index bits instead
    __host__ __device__ __forceinline__ GramPruneLds(uint32_t term_slots, uint32_t tgroup, uint32_t umap_slots, uint32_t map_slots, uint32_t words,
                                     uint32_t union_slots, uint32_t rank_bits = 0, uint32_t rank_slots = 0, bool narrow = true) {
        uint32_t o = 0;
        G = o; o += GRAM_ROWS * GRAM_STRIDE * 4;
        o = (o + 15) & ~15u;
        tabs = o; o += rank_slots ? RankTabLds(rank_bits, rank_slots, narrow).total
                           : union_slots ? GramUnionLds(union_slots).total : tgroup * (term_slots + GRAM_OVF) * 8;
        o = (o + 15) & ~15u;
        ovf_cnt = o; o += 24 * 4; // also the scratch of the rank table's running counts
        rowptr = o; o += GRAM_ROWS * 8;
        rownnz = o; o += GRAM_ROWS * 4;
        umap = o; o += umap_slots * 8;
        idmap = o; // for the detour counts; then, in the same bytes, what the tests of the pairs need:
        row = o;                       // dense norm, scale and error of the sketch, norm of the sparse part
        above = row + GRAM_ROWS * 16;  // bit s of row c: <c, s> exceeds c's norm ...
        below = above + GRAM_ROWS * 8; // ... and s's norm
        o += map_slots * 8 > GRAM_ROWS * 32 ? map_slots * 8 : GRAM_ROWS * 32;
        R = o; o += GRAM_ROWS * words * 4;
        F = o; o += GRAM_ROWS * 8; // keyword-flag matrix: bit s of row c = "s holds a term of u that c lacks"
        nb_id = o; o += GRAM_ROWS * 4;
        nb_dist = o; o += GRAM_ROWS * 4;
        nrm = o; o += GRAM_ROWS * 4;
        det = o; o += GRAM_ROWS * 4;
        order = o; o += GRAM_ROWS * 4;
        o_fwd = o; o += GRAM_ROWS * 4;
        o_det = o; o += GRAM_ROWS * 4;
        o_kw = o; o += (1 + APOE_KW_CAND) * 4;
        ctl = o; o += 16 * 4;
        total = o;
    }
};

// Sparse part of the Gram matrix with the rows in registers (K = 64, eight waves): wave w owns rows w, w + 8, ...
// (own[k] = row w + 8k, shape nnz | ns << 16, 0 where the row does not exist), loaded once. The pivots are taken
// eight at a time, one per wave (group g = rows 8g .. 8g + 7: every wave scatters ITS row own[g] into the rank
// table, apoe_ranktab.h), and every wave then probes the table with its own rows of index >= 8g, two per batch:
// no global memory access in the whole phase but for rows longer than the register window. G[p][b] += <p, b>
// for p < b. A group whose distinct terms exceed the table is done in passes of 4, 2 or 1 pivots.
constexpr int GR_OWN = GRAM_ROWS / 8;
template <bool NARROW>
__device__ __forceinline__ void gram_sparse_rank(const CorpusView& C, uint32_t m, float* G, const RankTab& T, uint32_t* scan,
                                                 const unsigned long long* rowptr, const uint32_t* rownnz, const RtRow<NARROW> (&own)[GR_OWN],
                                                 const uint32_t (&own_shape)[GR_OWN], uint32_t* fail, int tid, int nthreads) {
    const int wave = (int)uniform(tid / WAVE), lane = tid & (WAVE - 1);
    auto row_pairs = [&](uint32_t i) { Pairs p = gram_row(C, rowptr, rownnz, i); p.narrow = NARROW ? 1u : 0u; return p; };
    const uint32_t ng = m >= 2 ? (m - 2) / 8 + 1 : 0; // the last row is never a pivot
    uint32_t shape_lanes = 0; // lane k holds own_shape[k]: a wave-uniform pick by index without an indexed array
#pragma unroll
    for (int k = 0; k < GR_OWN; k++) shape_lanes = lane == k ? own_shape[k] : shape_lanes;
    for (uint32_t g = 0; g < ng; g++) {
        // this wave's pivot of the group: own[g], picked with wave-uniform selects so that own[] stays in registers
        RtRow<NARROW> pr = own[0];
#pragma unroll
        for (int k = 1; k < GR_OWN; k++) rt_row_select(pr, own[k], g == (uint32_t)k);
        const uint32_t pshape = (uint32_t)__builtin_amdgcn_readlane((int)shape_lanes, (int)g);
        const uint32_t prow = 8 * g + wave;
        const Pairs ptail = row_pairs(min(prow, m - 1));
        uint32_t lo = 0, cnt = 8;
        while (lo < 8) {
            const bool mine = (uint32_t)wave >= lo && (uint32_t)wave < lo + cnt && prow < m;
            const uint32_t built = ranktab_build_rows<NARROW>(T, pr, pshape, mine, wave - (int)lo, ptail, scan, tid, nthreads);
            if (built == EMPTY) {
                if (cnt == 1) { // one row alone does not fit: the caller falls back
                    if (tid == 0) *fail = 1;
                    lo += 1;
                } else {
                    cnt >>= 1;
                }
                continue;
            }
            const uint32_t n_ovf = NARROW ? 0u : uniform(min(scan[16], (uint32_t)RT_OVF));
#pragma unroll
            for (int k = 0; k < GR_OWN; k++) {
                if ((uint32_t)k >= g && own_shape[k] != 0) { // wave-uniform: rows of earlier groups have met these pivots as pivots themselves
                    float acc[1][RT_T];
                    RtRow<NARROW> rows[1];
                    uint32_t shape[1];
                    rows[0] = own[k];
                    rows[0].touch();
                    shape[0] = own_shape[k];
                    asm volatile("" : "+s"(shape[0]));
#pragma unroll
                    for (int t = 0; t < RT_T; t++) acc[0][t] = 0.f;
                    ranktab_probe_rows<NARROW, 1>(T, rows, shape, [&](int) { return row_pairs(wave + 8 * k); }, n_ovf, acc, lane);
                    uint32_t t;
                    const float z = wave_sum_1x8(acc[0], lane, &t);
                    const uint32_t b = wave + 8 * k, p = 8 * g + lo + t;
                    if ((lane & 15) < 4 && (lane & 32) == 0 && t < cnt && p < b) G[p * GRAM_STRIDE + b] += z;
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            lo += cnt;
            __syncthreads(); // the table is rebuilt next
        }
    }
}

// Sparse part of the Gram matrix from one numbering of the terms that at least two of the rows hold (narrow corpora; a term of one row
// only multiplies nothing). A bitmap over the term space counts a term's first and second appearance,
// the rank of its second-appearance bit is its slot; every wave writes the slots of its rows' pairs in place of their terms, drops the
// pairs without one (a third of them, for 64 rows of 180 Zipf terms) and deals the rest out to the lanes, 64 to a chunk. A group of
// eight pivots is then written straight into a table of eight values a slot (one word per pair, no clearing: a wave takes its pivot's words
// out again and puts the next in) and a row reads eight values per pair: no bitmap, no key, no hit test, empty lanes read a slot of zeros.
// Per node of 64 rows of 180 terms (1 290 shared ones) against the group-by-group rank table: 106 000 cycles
// instead of 151 000 (two nodes a CU), of them 31 000 for the numbering; what is left is bound by the 16-byte table reads (100 000 i.i.d.
// docs: prune 22.1 -> 16.4 ms).
// `region` / `bytes`: LDS for bitmap and table, one after the other. Returns false (for all threads alike, nothing written to G) when
// the slots do not fit the table or a row keeps more than 256 pairs. All threads call it; it ends with a barrier.
constexpr int GS_CHUNKS = 4;
struct SharedRow {
    float v[GS_CHUNKS];
    uint32_t s2[GS_CHUNKS / 2]; // slots of two pairs a word
    __device__ __forceinline__ uint32_t slot(int c) const { return (c & 1) ? s2[c >> 1] >> 16 : s2[c >> 1] & 0xFFFFu; }
};
__device__ __forceinline__ void gram_shared_groups(uint32_t m, float* G, float4* table, uint32_t plane, const SharedRow (&own)[GR_OWN], uint32_t chunks, int wave,
                                                   int lane) {
    // group g = rows 8 g .. 8 g + 7, row r in own[r / 8] of wave r % 8: wave w's pivot of group g is its own[g]; `chunks`: lane k holds the
    // chunks of own[k]
    float* words = reinterpret_cast<float*>(table) + ((wave >> 2) * plane * 4 + (wave & 3)); // this wave's word of slot 0
    const uint32_t ng = m >= 2 ? (m - 2) / 8 + 1 : 0; // the last row is never a pivot
    SharedRow pr = own[0];
    for (uint32_t g = 0; g < ng; g++) {
#pragma unroll
        for (int k = 1; k < GR_OWN; k++) { // wave-uniform selects, so that own[] stays in registers
            const bool take = g == (uint32_t)k;
#pragma unroll
            for (int c = 0; c < GS_CHUNKS; c++) pr.v[c] = take ? own[k].v[c] : pr.v[c];
#pragma unroll
            for (int c = 0; c < GS_CHUNKS / 2; c++) pr.s2[c] = take ? own[k].s2[c] : pr.s2[c];
        }
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) words[pr.slot(c) * 4] = pr.v[c]; // an empty lane's value is zero: the slot of zeros stays one
        __syncthreads();
#pragma unroll
        for (int k = 0; k < GR_OWN; k++) {
            const uint32_t nc = (uint32_t)__builtin_amdgcn_readlane((int)chunks, k), b = wave + 8 * k;
            if (b > 8 * g && nc != 0) { // wave-uniform
                float acc[8];
#pragma unroll
                for (int t = 0; t < 8; t++) acc[t] = 0.f;
                auto add = [&](float v, const float4& lo, const float4& hi) {
                    acc[0] = fmaf(v, lo.x, acc[0]);
                    acc[1] = fmaf(v, lo.y, acc[1]);
                    acc[2] = fmaf(v, lo.z, acc[2]);
                    acc[3] = fmaf(v, lo.w, acc[3]);
                    acc[4] = fmaf(v, hi.x, acc[4]);
                    acc[5] = fmaf(v, hi.y, acc[5]);
                    acc[6] = fmaf(v, hi.z, acc[6]);
                    acc[7] = fmaf(v, hi.w, acc[7]);
                };
                SharedRow r = own[k];
                asm volatile("" : "+v"(r.s2[0]), "+v"(r.s2[1])); // addresses are worked out here, not kept for all rows and groups
                // the reads of three chunks together, whether the row has them or not (an average row keeps 122 to 135 pairs), a fourth where it has
                float4 lo[GS_CHUNKS - 1], hi[GS_CHUNKS - 1];
#pragma unroll
                for (int c = 0; c < GS_CHUNKS - 1; c++) {
                    lo[c] = table[r.slot(c)];
                    hi[c] = table[plane + r.slot(c)];
                }
                asm volatile("" : "+v"(lo[0].x), "+v"(lo[1].x), "+v"(lo[2].x), "+v"(hi[0].x), "+v"(hi[1].x), "+v"(hi[2].x));
#pragma unroll
                for (int c = 0; c < GS_CHUNKS - 1; c++) add(r.v[c], lo[c], hi[c]);
                if (nc == GS_CHUNKS) add(r.v[GS_CHUNKS - 1], table[r.slot(GS_CHUNKS - 1)], table[plane + r.slot(GS_CHUNKS - 1)]);
                uint32_t t;
                const float z = wave_sum_1x8(acc, lane, &t);
                const uint32_t p = 8 * g + t;
                if ((lane & 15) < 4 && (lane & 32) == 0 && p < b) G[p * GRAM_STRIDE + b] = z;
            }
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) words[pr.slot(c) * 4] = 0.f;
    }
    __syncthreads();
}
template <typename TailFn> // tail(k): the Pairs of own row k, for those beyond the register window
__device__ __forceinline__ bool gram_sparse_shared(uint32_t m, float* G, char* region, uint32_t bytes, uint32_t index_bits, uint32_t span, uint32_t* scan,
                                                   const RtRow<true> (&rows)[GR_OWN], const uint32_t (&shapes)[GR_OWN], TailFn tail, int tid, int wave, int lane) {
    constexpr int NT = 8 * WAVE;
    constexpr uint32_t WINDOW = RT_CHUNKS * WAVE, KEPT = GS_CHUNKS * WAVE;
    RankTab T; // the bitmap: x = terms seen at least twice, y = terms seen, then the count of the x bits before
    T.word = reinterpret_cast<uint2*>(region);
    T.index_bits = index_bits;
    T.span = span;
    const uint32_t W = index_bits / 32, counts = W * 8;
    uint2* out = reinterpret_cast<uint2*>(region + counts) + wave * GS_CHUNKS * WAVE; // a row's pairs on their way to other lanes
    if (counts + 8 * GS_CHUNKS * WAVE * 8 > bytes) return false;
    for (uint32_t w = tid; w < W; w += NT) T.word[w] = make_uint2(0u, 0u);
    uint32_t* overfull = scan + 17;
    if (tid == 0) *overfull = 0;
    __syncthreads();
    auto seen = [&](uint32_t idx) {
        const uint32_t bit = 1u << (idx & 31);
        if (atomicOr(&T.word[idx >> 5].y, bit) & bit) atomicOr(&T.word[idx >> 5].x, bit);
    };
    auto index_of = [&](int k, int c) { return ranktab_index<true>(T, rows[k].key(c), rt_pair(c, lane) >= (shapes[k] >> 16)); };
#pragma unroll
    for (int k = 0; k < GR_OWN; k++) {
        const uint32_t nnz = shapes[k] & 0xFFFFu;
        uint32_t idx[GS_CHUNKS], old[GS_CHUNKS];
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) {
            idx[c] = index_of(k, c);
            old[c] = 0;
            if (rt_pair(c, lane) < nnz) old[c] = atomicOr(&T.word[idx[c] >> 5].y, 1u << (idx[c] & 31));
        }
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) {
            const uint32_t bit = 1u << (idx[c] & 31);
            if (old[c] & bit) atomicOr(&T.word[idx[c] >> 5].x, bit);
        }
        if (nnz > WINDOW) {
            const Pairs sp = tail(k);
            for (uint32_t j = WINDOW + lane; j < nnz; j += WAVE) seen(ranktab_index<true>(T, sp.raw(j).x, j >= sp.ns));
        }
    }
    __syncthreads();
    // counts: thread i owns the words [i * per, (i + 1) * per), two words (16 bytes) at a time
    const uint32_t per = ((W + NT - 1) / NT + 1) & ~1u;
    uint4* word2 = reinterpret_cast<uint4*>(T.word);
    uint32_t some = 0;
    for (uint32_t k = 0; k < per; k += 2) {
        const uint32_t w = tid * per + k;
        if (w < W) {
            const uint4 two = word2[w >> 1];
            some += __popc(two.x) + __popc(two.z);
        }
    }
    const uint32_t incl = wave_scan_add_dpp(some);
    if (lane == WAVE - 1) scan[wave] = incl;
    __syncthreads();
    uint32_t before = incl - some, total = 0;
    for (int w = 0; w < 8; w++) {
        const uint32_t x = scan[w];
        if (w < wave) before += x;
        total += x;
    }
    const uint32_t plane = total + 1; // the last slot stays zero
    if (plane * 32 > bytes || plane > 0xFFFFu) {
        __syncthreads();
        return false;
    }
    for (uint32_t k = 0; k < per; k += 2) {
        const uint32_t w = tid * per + k;
        if (w < W) {
            uint4 two = word2[w >> 1];
            two.y = before;
            before += __popc(two.x);
            two.w = before;
            before += __popc(two.z);
            word2[w >> 1] = two;
        }
    }
    __syncthreads();
    SharedRow own[GR_OWN];
    uint32_t chunks = 0;
#pragma unroll
    for (int k = 0; k < GR_OWN; k++) {
        const uint32_t nnz = shapes[k] & 0xFFFFu;
        uint32_t slot[GS_CHUNKS], mine = 0;
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) {
            slot[c] = EMPTY;
            if (rt_pair(c, lane) < nnz) {
                const uint32_t idx = index_of(k, c);
                slot[c] = ranktab_slot(T.word[idx >> 5], idx);
            }
            mine += slot[c] != EMPTY;
        }
        const uint32_t upto = wave_scan_add_dpp(mine);
        uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)upto, WAVE - 1);
        uint32_t at = upto - mine;
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++)
            if (slot[c] != EMPTY) out[at++] = make_uint2(slot[c], rows[k].v[c]);
        if (nnz > WINDOW) {
            const Pairs sp = tail(k);
            for (uint32_t j0 = WINDOW; j0 < nnz; j0 += WAVE) {
                const uint32_t j = j0 + lane;
                uint32_t sl = EMPTY;
                uint2 kv = make_uint2(0u, 0u);
                if (j < nnz) {
                    kv = sp.raw(j);
                    const uint32_t idx = ranktab_index<true>(T, kv.x, j >= sp.ns);
                    sl = ranktab_slot(T.word[idx >> 5], idx);
                }
                const uint64_t keep = __ballot(sl != EMPTY);
                const uint32_t to = all + __popcll(keep & ((1ull << lane) - 1));
                if (sl != EMPTY && to < KEPT) out[to] = make_uint2(sl, kv.y);
                all += __popcll(keep);
            }
            if (all > KEPT) *overfull = 1;
        }
        wave_fence_lds();
#pragma unroll
        for (int c = 0; c < GS_CHUNKS; c++) {
            uint2 x = make_uint2(total, 0u);
            if ((uint32_t)(c * WAVE + lane) < all) x = out[c * WAVE + lane];
            own[k].v[c] = __uint_as_float(x.y);
            if (c & 1) own[k].s2[c >> 1] |= x.x << 16;
            else own[k].s2[c >> 1] = x.x;
        }
        wave_fence_lds();
        const uint32_t nc = (all + WAVE - 1) / WAVE;
        chunks = lane == k ? nc : chunks;
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads(); // the bitmap is done with
    if (uniform(*overfull)) {
        __syncthreads();
        return false;
    }
    float4* table = reinterpret_cast<float4*>(region);
    for (uint32_t i = tid; i < 2 * plane; i += NT) table[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    __syncthreads();
    gram_shared_groups(m, G, table, plane, own, chunks, wave, lane);
    return true;
}

// Code products of up to 64 sketches (apoe_device.h), added as integers to the words above the diagonal of G, which hold zeros: wave w takes
// the codes 128 w .. 128 w + 127 of every row, so every sketch is read once; two v_mfma_i32_16x16x64_i8 per 16 x 16 block. Integer sums are
// exact: they do not depend on the order of the atomics. Lane (j, g), j = lane % 16, g = lane / 16, supplies codes 64 b + 16 g .. of
// block b for row j of a block and holds row 4 g + e, column j of a product.
__device__ __forceinline__ void gram_sketch_upper(const uint4* sketch, const uint32_t* ids, uint32_t m, int* Gi, int wave, int lane) {
    constexpr int NB = GRAM_ROWS / 16, KB = SKETCH_BYTES / 8 / 64;
    const int j = lane & 15, g = lane >> 4;
    intx4 x[NB][KB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint4* p = sketch + (size_t)ids[min((uint32_t)(16 * b + j), m - 1)] * (SKETCH_BYTES / 16) + wave * (SKETCH_BYTES / 8 / 16) + g;
#pragma unroll
        for (int k = 0; k < KB; k++) x[b][k] = __builtin_bit_cast(intx4, p[4 * k]);
    }
#pragma unroll
    for (int bi = 0; bi < NB; bi++) {
#pragma unroll
        for (int bj = bi; bj < NB; bj++) {
            if (16 * bj >= (int)m) continue; // wave-uniform
            intx4 acc = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < KB; k++) acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[bi][k], x[bj][k], acc, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = 16 * bi + 4 * g + e, c = 16 * bj + j;
                if (r < c && c < (int)m) atomicAdd(&Gi[r * GRAM_STRIDE + c], acc[e]);
            }
        }
    }
}

// Same result as prune_kernel, different traffic. The selection asks of two neighbours c and s of the node only whether <c, s> exceeds
// either one's norm, and mostly bounds tell: the dense part from the 8-bit sketches (64 KB a node instead of 256), the sparse part
// first as the product of the two sparse norms and, where that leaves a pair open, as the exact sparse Gram matrix of the node's rows (rank
// table, apoe_ranktab.h). A node with a pair that is open even then, and a corpus without sketches, takes the dense Gram matrix on the fp32
// matrix cores. The answers are two 64-bit masks per row, every row's overlap with the centre node's BM25 terms is a bit
// mask too, and the sequential RNG-IP selection with its keyword flags is a few scalar instructions per neighbour:
//   rejected(c) = above[c] & live;   live &= ~below[c];   flag(c, s) = (R[s] & ~R[c]) != 0   with R[x] = bm25(x) ∩ bm25(u).
// (100 000 docs, every node: cycles of wave 0 on one CU's two nodes, with the Gram matrix / as it is: dense part and its sums 68 000 / 6 000,
// keyword masks and flags 35 000 / 25 000, selection 28 000 / 2 500.)
template <int NT, bool NARROW>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 4))) void prune_gram_kernel(CorpusView C, float dense_mul, const float* __restrict__ norms,
                                                                const uint32_t* __restrict__ ids, const float* __restrict__ dist,
                                                                uint32_t d, uint32_t* fwd, uint32_t* det_out, uint32_t* cnt_out,
                                                                uint32_t* kw_out, uint32_t term_slots, uint32_t tgroup,
                                                                uint32_t umap_slots, uint32_t map_slots, uint32_t words,
                                                                uint32_t union_slots, uint32_t rank_bits, uint32_t rank_slots,
                                                                uint32_t rank_span, const SketchMeta* __restrict__ sketch_meta,
                                                                const uint4* __restrict__ sketch, const uint32_t* __restrict__ nodes, unsigned long long* gfail) {
    constexpr uint32_t K = GRAM_ROWS;
    constexpr int NWAVES = NT / WAVE;
    static_assert(NWAVES == 8, "dimensions and rows are dealt out to eight waves");
    C.narrow = NARROW ? 1u : 0u; // the pair format as a compile-time constant: no branch at the loads
    extern __shared__ __align__(16) char smem[];
    const GramPruneLds L(term_slots, tgroup, umap_slots, map_slots, words, union_slots, rank_bits, rank_slots, NARROW);
    float* G = reinterpret_cast<float*>(smem + L.G); // [i][j], i < j: sparse part of <i, j>; [j][i]: its dense part
    uint2* tabs = reinterpret_cast<uint2*>(smem + L.tabs);
    uint32_t* ovf_cnt = reinterpret_cast<uint32_t*>(smem + L.ovf_cnt);
    unsigned long long* rowptr = reinterpret_cast<unsigned long long*>(smem + L.rowptr);
    uint32_t* rownnz = reinterpret_cast<uint32_t*>(smem + L.rownnz);
    uint2* umap = reinterpret_cast<uint2*>(smem + L.umap);
    uint2* idmap = reinterpret_cast<uint2*>(smem + L.idmap);
    uint32_t* R = reinterpret_cast<uint32_t*>(smem + L.R);
    uint64_t* F = reinterpret_cast<uint64_t*>(smem + L.F);
    uint64_t* above = reinterpret_cast<uint64_t*>(smem + L.above);
    uint64_t* below = reinterpret_cast<uint64_t*>(smem + L.below);
    float4* row = reinterpret_cast<float4*>(smem + L.row); // dense norm, scale and error of the sketch, bound of the norm of the sparse part
    uint32_t* nb_id = reinterpret_cast<uint32_t*>(smem + L.nb_id);
    float* nb_dist = reinterpret_cast<float*>(smem + L.nb_dist);
    float* nrm = reinterpret_cast<float*>(smem + L.nrm);
    uint32_t* det = reinterpret_cast<uint32_t*>(smem + L.det);
    uint32_t* order = reinterpret_cast<uint32_t*>(smem + L.order);
    uint32_t* o_fwd = reinterpret_cast<uint32_t*>(smem + L.o_fwd);
    uint32_t* o_det = reinterpret_cast<uint32_t*>(smem + L.o_det);
    uint32_t* o_kw = reinterpret_cast<uint32_t*>(smem + L.o_kw);
    uint32_t* ctl = reinterpret_cast<uint32_t*>(smem + L.ctl);

    const int tid = threadIdx.x, wave = (int)uniform(tid / WAVE), lane = lane_id();
    const uint32_t u = nodes[blockIdx.x], umask = umap_slots - 1, mmask = map_slots - 1;
    const size_t base = (size_t)u * K;
    const uint64_t lane_lt = (1ull << lane) - 1;

    for (uint32_t i = tid; i < map_slots; i += NT) idmap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < umap_slots; i += NT) umap[i] = make_uint2(EMPTY, 0u);
    for (uint32_t i = tid; i < K * words; i += NT) R[i] = 0;
    for (uint32_t i = tid; i < K; i += NT) det[i] = 0;
    for (uint32_t i = tid; i < K * GRAM_STRIDE; i += NT) G[i] = 0.f;
    if (tid < 16) ctl[tid] = 0;
    __syncthreads();

    if (wave == 0) {
        const uint32_t v = ids[base + lane] & ~FLAG;
        const float dv = dist[base + lane];
        const bool ok = dv < INF_DIS && v < C.n && v != u;
        const uint64_t b = __ballot(ok);
        if (ok) {
            const uint32_t pos = __popcll(b & lane_lt);
            const uint64_t desc = C.desc[v];
            nb_id[pos] = v;
            nb_dist[pos] = dv;
            nrm[pos] = norms[v];
            rowptr[pos] = desc_off(desc) * 16 + DENSE_BYTES;
            rownnz[pos] = (desc_nnz_s(desc) + desc_nnz_b(desc)) | (desc_nnz_s(desc) << 16);
            lds_map_insert(idmap, mmask, v, pos);
        }
        if (lane == 0) ctl[PC_M] = __popcll(b);
    } else { // u's BM25 terms -> index
        const uint64_t du = C.desc[u];
        const Pairs sp = record_pairs(C, du);
        const uint32_t ns = desc_nnz_s(du), nb = desc_nnz_b(du);
        for (uint32_t j = tid - WAVE; j < nb; j += NT - WAVE) lds_map_insert(umap, umask, sp.key(ns + j), j);
    }
    __syncthreads();
    const uint32_t m = uniform(ctl[PC_M]);
    if (sketch && m) gram_sketch_upper(sketch, nb_id, m, reinterpret_cast<int*>(G), wave, lane);

    {   // (a) detour counts: all list entries of this thread are requested before the first one is looked up
        constexpr uint32_t PER = K * K / NT;
        uint32_t xs[PER];
        float dxs[PER];
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            const uint32_t t = tid + k * NT, r = t / K, j = t % K;
            xs[k] = EMPTY;
            dxs[k] = 0.f;
            if (t < m * K) {
                const size_t at = (size_t)nb_id[r] * K + j;
                xs[k] = ids[at] & ~FLAG;
                dxs[k] = dist[at];
            }
        }
        uint2 e[PER];
        lds_map_find(idmap, mmask, xs, e);
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            const uint32_t r = (tid + k * NT) / K;
            if (xs[k] != EMPTY && e[k].x == xs[k] && e[k].y > r && dxs[k] < nb_dist[e[k].y]) atomicAdd(&det[e[k].y], 1u);
        }
    }
    {   // R[r] = bits of u's BM25 terms that row r holds too: one wave per row, the first 64 BM25 terms of all its rows requested at once
        uint32_t key[GR_OWN], nbs[GR_OWN];
        auto row_pairs = [&](uint32_t r) {
            Pairs sp = gram_row(C, rowptr, rownnz, r);
            sp.narrow = NARROW ? 1u : 0u;
            return sp;
        };
#pragma unroll
        for (int k = 0; k < GR_OWN; k++) {
            const uint32_t r = wave + NWAVES * k;
            nbs[k] = 0;
            key[k] = EMPTY;
            if (r < m) { // wave-uniform
                const Pairs sp = row_pairs(r);
                nbs[k] = uniform(sp.nnz - sp.ns);
                if ((uint32_t)lane < nbs[k]) key[k] = sp.raw(sp.ns + lane).x; // the path bit follows where the key is used
            }
        }
        uint2 e[GR_OWN];
#pragma unroll
        for (int k = 0; k < GR_OWN; k++) key[k] |= BM25_BIT;
        lds_map_find(umap, umask, key, e);
#pragma unroll
        for (int k = 0; k < GR_OWN; k++) {
            const uint32_t r = wave + NWAVES * k;
            if (key[k] != EMPTY && e[k].x == key[k]) atomicOr(&R[r * words + (e[k].y >> 5)], 1u << (e[k].y & 31));
            if (nbs[k] > WAVE) {
                const Pairs sp = row_pairs(r);
                for (uint32_t j = WAVE + lane; j < nbs[k]; j += WAVE) {
                    const uint32_t x[1] = {sp.key(sp.ns + j)};
                    uint2 f[1];
                    lds_map_find(umap, umask, x, f);
                    if (f[0].x == x[0]) atomicOr(&R[r * words + (f[0].y >> 5)], 1u << (f[0].y & 31));
                }
            }
        }
    }
    __syncthreads();
    // the last wave, which has the fewest rows, reads what the tests need of a row: the map's bytes are free now
    if (wave == NWAVES - 1 && (uint32_t)lane < m) {
        const uint32_t v = nb_id[lane];
        const float nv = nrm[lane], dn = C.dnorm[v];
        SketchMeta sm = {0.f, 0.f};
        if (sketch) sm = sketch_meta[v];
        // what the hybrid norm leaves to the sparse part, with room for the rounding of both norms
        row[lane] = make_float4(dn, sm.scale, sm.err, sqrtf(fmaxf(nv - dense_mul * dn * dn, 0.f) + 1e-5f * (nv + dense_mul * dn * dn)));
    }
    // (b) stable order by detour count
    if (wave == 0) {
        const uint32_t key = (uint32_t)lane < m ? (det[lane] << 16) | (uint32_t)lane : ~0u;
        uint32_t r = 0;
        for (uint32_t j = 0; j < m; j++) r += (uint32_t)__builtin_amdgcn_readlane((int)key, (int)j) < key;
        if ((uint32_t)lane < m) order[r] = lane;
    }
    // keyword flags of all pairs (index.cu:637,651-654): flag(c, s) = (R[s] & ~R[c]) != 0, lane s of a wave for one c at a time
    {
        uint32_t rs[4];
#pragma unroll
        for (int w = 0; w < 4; w++) rs[w] = (uint32_t)w < words && (uint32_t)lane < m ? R[lane * words + w] : 0u;
        for (uint32_t c = wave; c < m; c += NWAVES) {
            uint32_t any = 0;
#pragma unroll
            for (int w = 0; w < 4; w++)
                if ((uint32_t)w < words) any |= rs[w] & ~(uint32_t)__builtin_amdgcn_readlane((int)rs[w], (int)c);
            for (uint32_t w = 4; w < words; w++) any |= ((uint32_t)lane < m ? R[lane * words + w] : 0u) & ~R[c * words + w];
            const uint64_t f = __ballot(any != 0);
            if (lane == 0) F[c] = f;
        }
    }
    // the dense Gram matrix on the matrix cores, below the diagonal: every wave takes an eighth of the dimensions and computes the
    // three tiles for it from one read of the rows; the partial tiles are added in a fixed order (barriers between them): the
    // result does not depend on timing
    auto dense_all = [&]() {
        constexpr int BLOCKS = DIM / 8;
        floatx16 dacc00, dacc01, dacc11;
        gram_dense_upper<PRUNE_DENSE_NB>(C, nb_id, m, lane, wave * (BLOCKS / NWAVES), (wave + 1) * (BLOCKS / NWAVES), dacc00, dacc01, dacc11);
        for (int ph = 0; ph < NWAVES; ph++) {
            if (wave == ph && m > 0) {
                gram_dense_store(G, 0, lane, dacc00, dense_mul, ph != 0);
                if (m > 32) {
                    gram_dense_store(G, 1, lane, dacc01, dense_mul, ph != 0);
                    gram_dense_store(G, 3, lane, dacc11, dense_mul, ph != 0);
                }
            }
            __syncthreads();
        }
    };
    auto code_product = [&](uint32_t i, uint32_t j) { // i < j
        return dense_mul * ((float)reinterpret_cast<const int*>(G)[i * GRAM_STRIDE + j] * (row[i].y * row[j].y));
    };
    // above[c], below[c] from what is known; returns whether a pair of the node stays open. bounded: the dense parts are within the sketches'
    // error, and until the sparse parts are `summed` they stand above the diagonal as integers; until then the sparse parts are known to lie
    // within the product of the sparse norms. any_open: an LDS word of this call, cleared
    auto decide = [&](bool bounded, bool summed, uint32_t& any_open) -> bool {
        bool open = false;
        const float4 rs = (uint32_t)lane < m ? row[lane] : make_float4(0.f, 0.f, 0.f, 0.f);
        const float ns = (uint32_t)lane < m ? nrm[lane] : 0.f;
        for (uint32_t c = wave; c < m; c += NWAVES) {
            const uint32_t lo = min(c, (uint32_t)lane), hi = max(c, (uint32_t)lane);
            const bool pair = (uint32_t)lane < m && (uint32_t)lane != c;
            const float4 rc = row[c];
            const float nc = nrm[c];
            float p = 0.f;
            if (pair) {
                if (bounded && !summed) p = code_product(lo, hi);
                else p = G[lo * GRAM_STRIDE + hi] + G[hi * GRAM_STRIDE + lo];
            }
            float e = 0.f; // p is exact but for e
            if (bounded) e = dense_mul * (rs.x * rc.z + rs.z * (rc.x + rc.z));
            if (!summed) e += rs.w * rc.w;
            if (bounded || !summed) e += 1e-5f * (dense_mul * rs.x * rc.x + rs.w * rc.w + 1.0f);
            const bool up = pair && nc < p, dn = pair && ns < p;
            if (bounded || !summed) open |= pair && !(fabsf(p - nc) > e && fabsf(p - ns) > e); // not a number: open
            const uint64_t a = __ballot(up), b = __ballot(dn);
            if (lane == 0) { above[c] = a; below[c] = b; }
        }
        if (open) any_open = 1;
        __syncthreads();
        return uniform(any_open) != 0;
    };
    const bool bounded = sketch != nullptr;
    if (bounded) __syncthreads(); // the order and the flags are behind one barrier with the code products
    else dense_all();
    if (decide(bounded, false, ctl[PC_OPEN])) {
        if (bounded) { // code products above the diagonal -> dense parts below it
            for (uint32_t t = tid; t < m * K; t += NT) {
                const uint32_t i = t / K, j = t % K;
                if (i < j && j < m) {
                    G[j * GRAM_STRIDE + i] = code_product(i, j);
                    G[i * GRAM_STRIDE + j] = 0.f;
                }
            }
            __syncthreads();
        }
        if (rank_slots != 0) { // the rank table, with this wave's rows w, w + 8, ... in registers
            auto own_rows = [&](RtRow<NARROW> (&own)[GR_OWN], uint32_t (&own_shape)[GR_OWN]) {
#pragma unroll
                for (int k = 0; k < GR_OWN; k++) {
                    const uint32_t b = wave + 8 * k;
                    own_shape[k] = 0;
                    if (b < m) {
                        own_shape[k] = uniform(rownnz[b]);
                        Pairs sp = gram_row(C, rowptr, rownnz, b);
                        sp.narrow = NARROW ? 1u : 0u;
                        rt_row_load(own[k], sp, lane);
                    }
                }
            };
            bool summed = false;
            if constexpr (NARROW) {
                RtRow<NARROW> own[GR_OWN];
                uint32_t own_shape[GR_OWN];
                own_rows(own, own_shape);
                summed = gram_sparse_shared(m, G, reinterpret_cast<char*>(tabs), RankTabLds(rank_bits, rank_slots, true).total, rank_bits, rank_span, ovf_cnt, own, own_shape,
                                            [&](int k) {
                                                Pairs sp = gram_row(C, rowptr, rownnz, wave + 8 * k);
                                                sp.narrow = 1u;
                                                return sp;
                                            }, tid, wave, lane);
            }
            if (!summed) {
                RtRow<NARROW> own[GR_OWN];
                uint32_t own_shape[GR_OWN];
                own_rows(own, own_shape);
                const RankTab T = ranktab_at(reinterpret_cast<char*>(tabs), rank_bits, rank_slots, rank_span, NARROW);
                gram_sparse_rank<NARROW>(C, m, G, T, ovf_cnt, rowptr, rownnz, own, own_shape, &ctl[PC_FAIL], tid, NT);
            }
        } else if (union_slots) gram_sparse_union(C, nb_id, m, G, reinterpret_cast<char*>(tabs), union_slots, ovf_cnt, rowptr, rownnz, &ctl[PC_FAIL], tid, NT);
        else if (tgroup == 8) gram_sparse_64<8>(C, nb_id, m, G, tabs, term_slots, ovf_cnt, rowptr, rownnz, &ctl[PC_FAIL], tid, NT);
        else gram_sparse_64<4>(C, nb_id, m, G, tabs, term_slots, ovf_cnt, rowptr, rownnz, &ctl[PC_FAIL], tid, NT);
        if (decide(bounded, true, ctl[PC_STILL_OPEN])) {
            dense_all();
            decide(false, true, ctl[PC_STILL_OPEN]);
        }
    }
    // (c)+(d) sequential selection, wave 0: lane t holds the masks of the candidate at position t of the order; `live` = the selected
    // members that are not tombstoned, `taken` = the positions that were selected
    if (wave == 0 && m > 0) {
        const uint32_t ord = (uint32_t)lane < m ? order[lane] : order[0];
        const uint64_t up = above[ord], dn = below[ord], fl = F[ord];
        uint64_t live = 1ull << (uint32_t)__builtin_amdgcn_readlane((int)ord, 0), taken = 1, flagged = 0;
        if (__ballot((uint32_t)lane < m && (up | dn) != 0) == 0) { // no product exceeds a norm: all are taken, a flag needs what stands before only
            uint64_t before = (uint32_t)lane < m ? 1ull << ord : 0ull;
            for (int o = 1; o < WAVE; o <<= 1) {
                const uint64_t x = ((uint64_t)(uint32_t)__shfl_up((uint32_t)(before >> 32), o, WAVE) << 32) | (uint32_t)__shfl_up((uint32_t)before, o, WAVE);
                if (lane >= o) before |= x;
            }
            live = taken = m == 64 ? ~0ull : (1ull << m) - 1;
            flagged = __ballot(lane > 0 && (uint32_t)lane < m && (before & ~(1ull << ord) & ~fl) == 0);
        } else for (uint32_t t = 1; t < m; t++) {
            const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)ord, (int)t);
            const bool reject = (readlane64(up, t) & live) != 0, allflag = (live & ~readlane64(fl, t)) == 0;
            live &= ~readlane64(dn, t);
            if (!reject) {
                live |= 1ull << c;
                taken |= 1ull << t;
                if (allflag) flagged |= 1ull << t;
            }
        }
        // (e) emit: live members in selection order fill the row, flagged ones beyond d become keyword candidates
        const uint32_t id_o = nb_id[ord], det_o = det[ord];
        const bool alive = ((taken >> lane) & 1) && ((live >> ord) & 1);
        const uint64_t lb = __ballot(alive);
        const uint32_t pos = __popcll(lb & lane_lt);
        if (alive && pos < d) { o_fwd[pos] = id_o; o_det[pos] = det_o; }
        uint32_t cnt = min((uint32_t)__popcll(lb), d);
        const bool kwc = alive && pos >= d && ((flagged >> lane) & 1);
        const uint64_t kb = __ballot(kwc);
        const uint32_t kpos = __popcll(kb & lane_lt);
        if (kwc && kpos < APOE_KW_CAND) o_kw[1 + kpos] = id_o;
        const uint32_t nkw = min((uint32_t)__popcll(kb), (uint32_t)APOE_KW_CAND);
        if (cnt < d) { // fewer survivors than the row has slots: the remaining neighbours in order, each id once
            bool add = (uint32_t)lane < m;
            for (uint64_t rest = lb; rest; rest &= rest - 1) add = add && (uint32_t)__builtin_amdgcn_readlane((int)id_o, __builtin_ctzll(rest)) != id_o;
            for (uint32_t t = 0; t + 1 < m; t++) add = add && !((uint32_t)lane > t && (uint32_t)__builtin_amdgcn_readlane((int)id_o, (int)t) == id_o);
            const uint64_t ab = __ballot(add);
            const uint32_t at = cnt + __popcll(ab & lane_lt);
            if (add && at < d) { o_fwd[at] = id_o; o_det[at] = det_o; }
            cnt = min(d, cnt + (uint32_t)__popcll(ab));
        }
        if (lane == 0) { ctl[PC_CNT] = cnt; o_kw[0] = nkw; }
        for (uint32_t j = cnt + lane; j < d; j += WAVE) { o_fwd[j] = u; o_det[j] = EMPTY; }
        for (uint32_t j = nkw + lane; j < APOE_KW_CAND; j += WAVE) o_kw[1 + j] = 0;
    }
    if (m == 0 && tid == 0) {
        for (uint32_t j = 0; j < d; j++) { o_fwd[j] = u; o_det[j] = EMPTY; }
        for (uint32_t j = 0; j <= APOE_KW_CAND; j++) o_kw[j] = 0;
        ctl[PC_CNT] = 0;
    }
    __syncthreads();
    for (uint32_t i = tid; i < d; i += NT) {
        fwd[(size_t)u * d + i] = o_fwd[i];
        det_out[(size_t)u * d + i] = o_det[i];
    }
    for (uint32_t i = tid; i < 1 + APOE_KW_CAND; i += NT) kw_out[(size_t)u * (1 + APOE_KW_CAND) + i] = o_kw[i];
    if (tid == 0) {
        cnt_out[u] = ctl[PC_CNT];
        if (ctl[PC_FAIL]) atomicOr(gfail, 1ull);
        // an overflow list was too short: the host redoes the prune with prune_kernel
    }
}

// ---- final rows (index.cu:717-807) ----

__global__ __launch_bounds__(256) void indegree_kernel(uint32_t n, uint32_t d, const uint32_t* __restrict__ fwd, const uint32_t* __restrict__ cnt,
                                                       uint32_t* indeg) {
    const uint64_t total = (uint64_t)n * d;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t u = (uint32_t)(t / d), j = (uint32_t)(t % d);
        if (j >= cnt[u]) continue;
        const uint32_t v = fwd[t];
        if (v < n && v != u) atomicAdd(&indeg[v], 1u);
    }
}

__global__ __launch_bounds__(256) void fill_in_edges_kernel(uint32_t n, uint32_t d, const uint32_t* __restrict__ fwd,
                                                            const uint32_t* __restrict__ det, const uint32_t* __restrict__ cnt,
                                                            const uint32_t* __restrict__ in_off, uint32_t* cursor, uint64_t* in_edges) {
    const uint64_t total = (uint64_t)n * d;
    for (uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; t < total; t += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t u = (uint32_t)(t / d), j = (uint32_t)(t % d);
        if (j >= cnt[u]) continue;
        const uint32_t v = fwd[t];
        if (v < n && v != u) in_edges[in_off[v] + atomicAdd(&cursor[v], 1u)] = ((uint64_t)det[t] << 32) | u;
    }
}

__device__ __forceinline__ uint64_t wave_min64(uint64_t v) {
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        const uint64_t other = shfl_xor64(v, o);
        v = other < v ? other : v;
    }
    return v;
}

// One wave per node v. Row = first half of v's forward list, then up to d/2 reverse
// neighbours in (detour, id) order that are not in the first half, topped up from the
// second half of the forward list and finally with v itself; then the keyword slots.
__global__ __launch_bounds__(256) void final_rows_kernel(uint32_t n, uint32_t d, const uint32_t* __restrict__ fwd, const uint32_t* __restrict__ kw,
                                                         const uint32_t* __restrict__ in_off, const uint64_t* __restrict__ in_edges,
                                                         uint32_t* rows) {
    __shared__ uint32_t s_row[4][WAVE + APOE_KW_SLOTS];
    const int wave = threadIdx.x / WAVE, lane = lane_id();
    const uint32_t v = blockIdx.x * 4 + wave;
    if (v >= n) return;
    uint32_t* row = s_row[wave];
    const uint32_t W = d + APOE_KW_SLOTS, h = d / 2;
    const uint32_t* fw = fwd + (size_t)v * d;
    if ((uint32_t)lane < h) row[lane] = fw[lane];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t fill = h;
    const uint32_t e0 = in_off[v], e1 = in_off[v + 1];
    {
        // the h smallest (detour, source) keys among the in-edges whose source is not in the first half, in one pass:
        // lanes 0 .. h-1 hold the best keys so far in ascending order; a chunk of 64 in-edges is tested against the
        // largest of them first (after a few chunks almost no key passes: a node with 10^5 in-edges costs one load and
        // one compare per 64 of them), the keys that pass are inserted one at a time
        uint64_t best = ~0ull; // lane i: the i-th smallest key so far (lanes >= h unused)
        for (uint32_t eb = e0; eb < e1; eb += WAVE) {
            const uint32_t e = eb + lane;
            uint64_t k = e < e1 ? in_edges[e] : ~0ull;
            const uint64_t worst = readlane64(best, h - 1);
            bool cand = k < worst;
            if (__ballot(cand) == 0) continue;
            if (cand) {
                const uint32_t uu = (uint32_t)k;
                bool present = false;
                for (uint32_t j = 0; j < h; j++) present |= row[j] == uu;
                cand = !present;
            }
            for (uint64_t rest = __ballot(cand); rest; rest &= rest - 1) {
                const uint64_t x = readlane64(k, (uint32_t)__builtin_ctzll(rest));
                const uint32_t pos = __popcll(__ballot(best < x)); // best is ascending: the lanes below pos keep their keys
                if (pos >= h) continue;
                const uint64_t up = __shfl_up(best, 1, WAVE);
                best = (uint32_t)lane == pos ? x : (uint32_t)lane > pos ? up : best;
            }
        }
        const uint32_t got = min((uint32_t)__popcll(__ballot(best != ~0ull && (uint32_t)lane < h)), h);
        if ((uint32_t)lane < got) row[h + lane] = (uint32_t)best;
        fill = h + got;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (uint32_t j = h; j < d && fill < d; j++) {
        const uint32_t c = fw[j];
        bool present = false;
        for (uint32_t t = lane; t < fill; t += WAVE) present |= row[t] == c;
        if (!__any(present)) {
            if (lane == 0) row[fill] = c;
            fill++;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    for (uint32_t j = fill + lane; j < d; j += WAVE) row[j] = v;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // keyword edges
    const uint32_t* kv = kw + (size_t)v * (1 + APOE_KW_CAND);
    const uint32_t nk = min(kv[0], (uint32_t)APOE_KW_CAND);
    if (lane < APOE_KW_SLOTS) row[d + lane] = 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint32_t c = 0;
    for (uint32_t j = 0; j < nk && c < APOE_KW_SLOTS - 1; j++) {
        const uint32_t x = kv[1 + j];
        bool present = false;
        for (uint32_t t = h + lane; t < d; t += WAVE) present |= row[t] == x;
        if (!__any(present)) {
            if (lane == 0) row[d + 1 + c] = x;
            c++;
        }
    }
    if (lane == 0) row[d] = c;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (uint32_t j = lane; j < W; j += WAVE) rows[(size_t)v * W + j] = row[j];
}

static uint32_t doc_term_slots(const apoe_corpus* c) { return next_pow2(std::max(64u, 2 * (c->max_nnz_s + c->max_nnz_b))); }

// Where no bounds can be asked (a corpus without sketches): every node is open, but for those that the table-probing kernel takes. One wave per node.
__global__ __launch_bounds__(256) void prune_triage_kernel(uint32_t n, uint32_t K, const uint32_t* __restrict__ ids, const float* __restrict__ dist,
                                                           const float* __restrict__ norms, uint32_t* open) {
    const uint32_t u = blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE, lane = lane_id();
    if (u >= n) return;
    bool far = false;
    for (uint32_t i = lane; i < K; i += WAVE) {
        const uint32_t v = ids[(size_t)u * K + i] & ~FLAG;
        if (dist[(size_t)u * K + i] < INF_DIS && v < n && v != u) far |= !(norms[v] < __builtin_inff());
    }
    const bool table = __ballot(far) != 0;
    if (lane == 0) open[u] = table ? NODE_TABLE : NODE_OPEN;
}

// The nodes of either flag, in no order: those of NODE_OPEN from the front of the list, those of NODE_TABLE from its end (`table` = 0: they
// count as open). One atomic per wave and flag (one per node on a single counter is 19 ns each, one after the other).
__global__ __launch_bounds__(256) void open_nodes_kernel(uint32_t n, uint32_t table, const uint32_t* __restrict__ flag, uint32_t* count, uint32_t* nodes) {
    const uint32_t u = blockIdx.x * blockDim.x + threadIdx.x, f = u < n ? flag[u] : (uint32_t)NODE_SETTLED;
    const bool to_table = table && f == NODE_TABLE;
    for (int side = 0; side < 2; side++) {
        const uint64_t b = __ballot(side ? to_table : f != NODE_SETTLED && !to_table);
        if (b == 0) continue;
        uint32_t at = 0;
        if (lane_id() == 0) at = atomicAdd(count + side, (uint32_t)__popcll(b));
        at = uniform(at) + __popcll(b & ((1ull << lane_id()) - 1));
        if ((b >> lane_id()) & 1) nodes[side ? n - 1 - at : at] = u;
    }
}

// Prunes the nodes that bounds settle (prune_bound_kernel) and lists the others, in no order.
struct OpenNodes {
    uint32_t open = 0, table = 0; // how many are left to the gathered forms and to the table-probing kernel
    const uint32_t *open_nodes = nullptr, *table_nodes = nullptr;
};
static int launch_prune_bounds(apoe_knn* g, uint32_t degree, uint32_t umap_slots, uint32_t map_slots, uint32_t words, bool table_form, OpenNodes* left) {
    apoe_ctx* ctx = g->ctx;
    const uint32_t n = g->n;
    const uint32_t lds = g->K == 64 ? BoundLds<64>(umap_slots, map_slots, words).total : BoundLds<128>(umap_slots, map_slots, words).total;
    if (!g->open.p) APOE_TRY(g->open.alloc(2 * (size_t)n + 2)); // flags, numbers, nodes
    APOE_HIP(hipMemsetAsync(g->open.p, 0, ((size_t)n + 2) * sizeof(uint32_t), ctx->stream));
    if (g->corpus->sketch.p && lds <= ctx->lds_per_block) {
        auto kernel = g->K == 64 ? (g->corpus->narrow ? &prune_bound_kernel<64, true> : &prune_bound_kernel<64, false>)
                                 : (g->corpus->narrow ? &prune_bound_kernel<128, true> : &prune_bound_kernel<128, false>);
        APOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        kernel<<<n, g->K * 4, lds, ctx->stream>>>(g->corpus->view(), g->dense_scale * g->dense_scale, g->norms.p, g->ids.p, g->dist.p, degree, g->fwd.p, g->det.p,
                                                  g->cnt.p, g->kw.p, umap_slots, map_slots, words, g->corpus->sketch_meta.p,
                                                  reinterpret_cast<const uint4*>(g->corpus->sketch.p), g->open.p);
    } else {
        prune_triage_kernel<<<(n + 3) / 4, 256, 0, ctx->stream>>>(n, g->K, g->ids.p, g->dist.p, g->norms.p, g->open.p);
    }
    APOE_HIP(hipGetLastError());
    uint32_t *count = g->open.p + n, *list = count + 2, h[2] = {0, 0};
    open_nodes_kernel<<<(n + 255) / 256, 256, 0, ctx->stream>>>(n, table_form, g->open.p, count, list);
    APOE_HIP(hipGetLastError());
    APOE_HIP(hipMemcpyAsync(h, count, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
    APOE_HIP(hipStreamSynchronize(ctx->stream));
    left->open = h[0];
    left->table = h[1];
    left->open_nodes = list;
    left->table_nodes = list + (n - h[1]);
    return APOE_OK;
}

int launch_prune(apoe_knn* g, uint32_t degree) {
    apoe_ctx* ctx = g->ctx;
    const uint32_t term_slots = doc_term_slots(g->corpus);
    const uint32_t uset_slots = next_pow2(std::max(64u, 2 * g->corpus->max_nnz_b));
    const uint32_t map_slots = next_pow2(4 * g->K);
    // gather-once form: K = 64 and the BM25 overlap masks fit in LDS
    const uint32_t words = (g->corpus->max_nnz_b + 31) / 32 + (g->corpus->max_nnz_b == 0);
    const uint32_t gram_slots = next_pow2(std::max(64u, 2 * (g->corpus->max_nnz_s + g->corpus->max_nnz_b)));
    // 8 live pivot tables if two workgroups then still share a CU's LDS, else 4
    const uint32_t lds_budget = (uint32_t)std::min<size_t>(ctx->lds_per_block, 80 * 1024);
    uint32_t tgroup = GramPruneLds(gram_slots, 8, uset_slots, map_slots, words, 0).total <= lds_budget ? 8 : 4;
    // one union table for GU_T pivots when it fits: 2.5 slots per term of an average group, and room for the longest row alone
    const double mean_nnz = g->n ? (double)g->corpus->total_pairs / g->n : 0.0;
    uint32_t union_slots = std::max(next_pow2((uint32_t)std::ceil(2.5 * GU_T * mean_nnz)), std::max(512u, gram_slots));
    if (GramPruneLds(gram_slots, tgroup, uset_slots, map_slots, words, union_slots).total > lds_budget) union_slots = 0;
    // rank table for eight pivots when its bitmap leaves room for the values of at least the longest row (and then as many
    // slots as the budget allows, up to eight rows' worth): the sparse part then runs with the rows held in registers
    const bool narrow = g->corpus->narrow;
    const uint32_t rank_span = next_pow2(std::max(g->corpus->max_term + 1, 1024u));
    const uint32_t rank_bits = narrow ? 2 * rank_span : 65536u;
    uint32_t rank_slots = 0;
    {
        const uint32_t longest = g->corpus->max_nnz_s + g->corpus->max_nnz_b;
        const uint32_t fixed = GramPruneLds(gram_slots, tgroup, uset_slots, map_slots, words, 0, rank_bits, 64, narrow).total -
                               RankTabLds(rank_bits, 64, narrow).total + RankTabLds(rank_bits, 0, narrow).total;
        const uint32_t per_slot = RT_T * 4 + (narrow ? 0 : 4);
        if (fixed + 64 < lds_budget) {
            uint32_t fit = ((lds_budget - fixed - 64) / per_slot) & ~63u;
            fit = std::min(fit, (RT_T * longest + 63) & ~63u);
            if (fit >= std::max(longest, 64u)) rank_slots = fit;
        }
    }
    const GramPruneLds GL(gram_slots, tgroup, uset_slots, map_slots, words, union_slots, rank_bits, rank_slots, narrow);
    const bool gathered = !g->force_sequential_prune && (g->K == GRAM_ROWS ? GL.total <= lds_budget : g->K <= PS_MAX && gram_tiles_fit(g));
    const PruneLds L(term_slots, uset_slots, map_slots, g->K);
    const bool table_fits = L.total <= 64 * 1024;
    auto table_form = [&](uint32_t count, const uint32_t* nodes) -> int { // the table-probing kernel; null: all nodes
        APOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&prune_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)L.total));
        prune_kernel<<<count, PR_THREADS, L.total, ctx->stream>>>(g->corpus->view(), g->dense_scale * g->dense_scale, g->norms.p, g->K, g->ids.p, g->dist.p, degree,
                                                                  nodes, g->fwd.p, g->det.p, g->cnt.p, g->kw.p, term_slots, uset_slots, map_slots);
        APOE_HIP(hipGetLastError());
        return APOE_OK;
    };
    // nodes that bounds settle are done here; the others are left in two lists
    OpenNodes left;
    if (gathered) {
        APOE_TRY(launch_prune_bounds(g, degree, uset_slots, map_slots, words, table_fits, &left));
        if (left.table) APOE_TRY(table_form(left.table, left.table_nodes));
        if (left.open == 0) return APOE_OK;
    }
    if (g->K == GRAM_ROWS && gathered) {
        APOE_HIP(hipMemsetAsync(g->counter.p + 1, 0, sizeof(unsigned long long), ctx->stream));
        auto kernel = g->corpus->narrow ? &prune_gram_kernel<GRAM_THREADS, true> : &prune_gram_kernel<GRAM_THREADS, false>;
        APOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)GL.total));
        kernel<<<left.open, GRAM_THREADS, GL.total, ctx->stream>>>(g->corpus->view(), g->dense_scale * g->dense_scale, g->norms.p, g->ids.p, g->dist.p, degree,
                                                                g->fwd.p, g->det.p, g->cnt.p, g->kw.p, gram_slots, tgroup, uset_slots, map_slots, words,
                                                                union_slots, rank_bits, rank_slots, rank_span, g->corpus->sketch_meta.p,
                                                                reinterpret_cast<const uint4*>(g->corpus->sketch.p), left.open_nodes, g->counter.p + 1);
        APOE_HIP(hipGetLastError());
        unsigned long long failed = 0;
        APOE_HIP(hipMemcpyAsync(&failed, g->counter.p + 1, sizeof(failed), hipMemcpyDeviceToHost, ctx->stream));
        APOE_HIP(hipStreamSynchronize(ctx->stream));
        if (!failed) return APOE_OK;
        // a row's terms clustered on the same table slots: redo with the table-probing kernel below
    }
    // lists longer than 64 entries: Gram matrices by the tile kernel of the local join, a batch of nodes at a time, and the
    // selection on them; a row too long for a tile's table sends the whole prune to the table-probing kernel below
    if (g->K > GRAM_ROWS && gathered) {
        const SelectLds SL(uset_slots, map_slots, words);
        if (SL.total <= ctx->lds_per_block) {
            const uint32_t batch = std::min<uint32_t>(left.open, 32768u);
            DevBuf<float> gram;
            APOE_TRY(gram.alloc((size_t)batch * PS_MAX * PS_MAX));
            APOE_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&prune_select_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)SL.total));
            unsigned long long unfit = 0;
            bool pair = false;
            APOE_TRY(gram_tiles_pair(g, left.open_nodes, left.open, &pair));
            for (uint32_t node0 = 0; node0 < left.open && !unfit; node0 += batch) {
                const uint32_t cnt = std::min(batch, left.open - node0);
                APOE_TRY(launch_gram_tiles(g, left.open_nodes, node0, cnt, pair, gram.p, &unfit));
                if (unfit) break;
                prune_select_kernel<<<cnt, PS_THREADS, SL.total, ctx->stream>>>(g->corpus->view(), g->norms.p, g->K, g->ids.p, g->dist.p, degree, left.open_nodes, node0, gram.p,
                                                                              g->fwd.p, g->det.p, g->cnt.p, g->kw.p, uset_slots, map_slots, words);
                APOE_HIP(hipGetLastError());
            }
            APOE_HIP(hipStreamSynchronize(ctx->stream)); // the batch buffer is freed on return
            if (!unfit) return APOE_OK;
        }
    }
    APOE_REQUIRE(table_fits, "prune needs %u bytes of LDS (rows with up to %u sparse terms)", L.total, g->corpus->max_nnz_s + g->corpus->max_nnz_b);
    return table_form(g->n, nullptr);
}

int launch_final_graph(apoe_knn* g, uint32_t* rows_dev) {
    apoe_ctx* ctx = g->ctx;
    const uint32_t n = g->n, d = g->degree;
    DevBuf<uint32_t> indeg, in_off, cursor;
    DevBuf<uint64_t> in_edges;
    DevBuf<char> temp;
    APOE_TRY(indeg.alloc((size_t)n + 1));
    APOE_TRY(in_off.alloc((size_t)n + 1));
    APOE_TRY(cursor.alloc(n));
    APOE_TRY(in_edges.alloc((size_t)n * d));
    APOE_HIP(hipMemsetAsync(indeg.p, 0, ((size_t)n + 1) * sizeof(uint32_t), ctx->stream));
    APOE_HIP(hipMemsetAsync(cursor.p, 0, (size_t)n * sizeof(uint32_t), ctx->stream));
    const uint32_t grid = (uint32_t)std::min<uint64_t>(((uint64_t)n * d + 255) / 256, 1u << 20);
    indegree_kernel<<<grid, 256, 0, ctx->stream>>>(n, d, g->fwd.p, g->cnt.p, indeg.p);
    APOE_HIP(hipGetLastError());
    size_t temp_bytes = 0;
    APOE_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, temp_bytes, indeg.p, in_off.p, (int)(n + 1), ctx->stream));
    APOE_TRY(temp.alloc(temp_bytes));
    APOE_HIP(hipcub::DeviceScan::ExclusiveSum(temp.p, temp_bytes, indeg.p, in_off.p, (int)(n + 1), ctx->stream));
    fill_in_edges_kernel<<<grid, 256, 0, ctx->stream>>>(n, d, g->fwd.p, g->det.p, g->cnt.p, in_off.p, cursor.p, in_edges.p);
    APOE_HIP(hipGetLastError());
    final_rows_kernel<<<(n + 3) / 4, 256, 0, ctx->stream>>>(n, d, g->fwd.p, g->kw.p, in_off.p, in_edges.p, rows_dev);
    APOE_HIP(hipGetLastError());
    APOE_HIP(hipStreamSynchronize(ctx->stream)); // temporaries are released on return
    return APOE_OK;
}

} // namespace apoe

using namespace apoe;

extern "C" {

int apoe_knn_set_prune_form(apoe_knn* g, int form) {
    APOE_REQUIRE(g, "null argument");
    APOE_REQUIRE(form == 0 || form == 1, "prune form must be 0 (gather-once forms where they apply) or 1 (the table-probing kernel), got %d", form);
    g->force_sequential_prune = form == 1;
    return APOE_OK;
}

int apoe_prune(apoe_knn* g, uint32_t degree) {
    APOE_REQUIRE(g, "null argument");
    APOE_REQUIRE(degree >= 2 && degree <= 64 && degree % 2 == 0 && degree <= g->K, "degree must be even, in [2, 64] and <= K, got %u", degree);
    APOE_REQUIRE_STATE(g->ready, "the lists are empty: call apoe_nnd_init or apoe_knn_upload first");
    APOE_HIP(hipSetDevice(g->ctx->device));
    g->degree = degree;
    APOE_TRY(g->fwd.alloc((size_t)g->n * degree));
    APOE_TRY(g->det.alloc((size_t)g->n * degree));
    APOE_TRY(g->cnt.alloc(g->n));
    APOE_TRY(g->kw.alloc((size_t)g->n * (1 + APOE_KW_CAND)));
    float ms = 0.f;
    APOE_TRY(timed(g->ctx, &ms, [&]() { return launch_prune(g, degree); }));
    g->elapsed_ms += ms;
    g->pruned = true;
    return APOE_OK;
}

int apoe_prune_download(apoe_knn* g, uint32_t* fwd, uint32_t* det, uint32_t* cnt, uint32_t* kw) {
    APOE_REQUIRE(g, "null argument");
    if (!g->pruned) {
        set_error("apoe_prune has not run on this handle");
        return APOE_ERR_STATE;
    }
    APOE_HIP(hipSetDevice(g->ctx->device));
    if (fwd) APOE_TRY(copy_out(g->ctx, fwd, g->fwd.p, g->fwd.bytes()));
    if (det) APOE_TRY(copy_out(g->ctx, det, g->det.p, g->det.bytes()));
    if (cnt) APOE_TRY(copy_out(g->ctx, cnt, g->cnt.p, (size_t)g->n * sizeof(uint32_t)));
    if (kw) APOE_TRY(copy_out(g->ctx, kw, g->kw.p, g->kw.bytes()));
    return APOE_OK;
}

int apoe_finalize_graph(apoe_knn* g, apoe_graph** out) {
    APOE_REQUIRE(g && out, "null argument");
    *out = nullptr;
    if (!g->pruned) {
        set_error("apoe_prune has not run on this handle");
        return APOE_ERR_STATE;
    }
    APOE_HIP(hipSetDevice(g->ctx->device));
    std::unique_ptr<apoe_graph> gr(new apoe_graph());
    gr->ctx = g->ctx;
    gr->n = g->n;
    gr->width = g->degree + APOE_KW_SLOTS;
    gr->n_entry = g->degree;
    APOE_TRY(gr->rows.alloc((size_t)gr->n * gr->width));
    APOE_TRY(gr->entry.alloc(gr->n_entry));
    float ms = 0.f;
    APOE_TRY(timed(g->ctx, &ms, [&]() { return launch_final_graph(g, gr->rows.p); }));
    g->elapsed_ms += ms;
    // entry points: the `degree` documents of smallest hybrid norm, ties by id (index.cu:916-925)
    std::vector<float> nrm(g->n);
    APOE_TRY(copy_out(g->ctx, nrm.data(), g->norms.p, (size_t)g->n * sizeof(float)));
    std::vector<std::pair<float, uint32_t>> dp(g->n);
    for (uint32_t i = 0; i < g->n; i++) dp[i] = {nrm[i], i};
    const uint32_t k = std::min(gr->n_entry, g->n);
    std::partial_sort(dp.begin(), dp.begin() + k, dp.end());
    std::vector<uint32_t> ep(gr->n_entry);
    for (uint32_t i = 0; i < gr->n_entry; i++) ep[i] = dp[i % k].second;
    APOE_TRY(copy_in(g->ctx, gr->entry.p, ep.data(), ep.size() * sizeof(uint32_t)));
    *out = gr.release();
    return APOE_OK;
}

} // extern "C"
