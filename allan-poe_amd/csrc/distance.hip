// Corpus packing, fused hybrid distance (batch and pair forms) and hybrid norms.
#include "apoe_internal.h"

namespace apoe {

// Largest value of an index array (decides whether the corpus can use narrow pairs).
__global__ __launch_bounds__(256) void max_u32_kernel(const uint32_t* __restrict__ a, size_t n, uint32_t* out) {
    uint32_t m = 0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) m = max(m, a[i]);
#pragma unroll
    for (int o = WAVE / 2; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor(m, o, WAVE));
    if (lane_id() == 0 && m) atomicMax(out, m);
}

int launch_max_u32(apoe_ctx* ctx, const uint32_t* a_dev, size_t n, uint32_t* out_dev) { // *out_dev must hold 0 (or a running maximum)
    if (n == 0) return APOE_OK;
    const uint32_t grid = (uint32_t)std::min<size_t>((n + 255) / 256, 4096);
    max_u32_kernel<<<grid, 256, 0, ctx->stream>>>(a_dev, n, out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// One workgroup per document: dense row, then SPLADE pairs, then BM25 pairs, written as one
// contiguous record in the wide (path bit in the term key) or the narrow pair format.
__global__ __launch_bounds__(256) void pack_kernel(uint32_t n, const float* __restrict__ dense, const uint32_t* __restrict__ s_off,
                                                   const uint32_t* __restrict__ s_idx, const float* __restrict__ s_val,
                                                   const uint32_t* __restrict__ b_off, const uint32_t* __restrict__ b_idx,
                                                   const float* __restrict__ b_val, const uint64_t* __restrict__ desc, char* recs, float* dnorm,
                                                   SketchMeta* sketch_meta, uint32_t* sketch, uint32_t narrow, uint32_t coded) {
    __shared__ float part[4], top[4], rest[4], most[2][4];
    for (uint32_t doc = blockIdx.x; doc < n; doc += gridDim.x) {
        const uint64_t d = desc[doc];
        char* rec = recs + desc_off(d) * 16;
        const float4* src = reinterpret_cast<const float4*>(dense + (size_t)doc * DIM);
        float4* dst = reinterpret_cast<float4*>(rec);
        static_assert(DIM / 4 == 256, "a thread per float4 of the dense row");
        const uint32_t s0 = s_off[doc], ns = desc_nnz_s(d), b0 = b_off[doc], nb = desc_nnz_b(d), nnz = ns + nb;
        const float4 x = src[threadIdx.x];
        // a pair per thread, requested with the dense row (narrow records; rows of more than 256 pairs read the rest below)
        auto value = [&](uint32_t j) { return j < ns ? s_val[s0 + j] : b_val[b0 + (j - ns)]; };
        auto term = [&](uint32_t j) { return j < ns ? s_idx[s0 + j] : b_idx[b0 + (j - ns)]; };
        float v = 0.f;
        uint32_t id = 0;
        if (narrow && threadIdx.x < nnz) {
            v = value(threadIdx.x);
            id = term(threadIdx.x);
        }
        dst[threadIdx.x] = x;
        const float sq = wave_sum_dpp(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w);
        const float high = -wave_min_dpp(-max_abs4(x));
        float largest[2] = {0.f, 0.f}; // magnitude per path; a value that is no number counts as infinite
        if (coded) {
            auto raise = [&](uint32_t j, float y) { float& to = largest[j < ns ? 0 : 1]; to = y == y ? fmaxf(to, fabsf(y)) : __builtin_inff(); };
            if (threadIdx.x < nnz) raise(threadIdx.x, v);
            for (uint32_t j = threadIdx.x + 256; j < nnz; j += 256) raise(j, value(j));
            largest[0] = -wave_min_dpp(-largest[0]);
            largest[1] = -wave_min_dpp(-largest[1]);
        }
        __syncthreads();
        if (lane_id() == 0) {
            part[threadIdx.x / WAVE] = sq;
            top[threadIdx.x / WAVE] = high;
            most[0][threadIdx.x / WAVE] = largest[0];
            most[1][threadIdx.x / WAVE] = largest[1];
        }
        __syncthreads();
        const float norm = sqrtf(part[0] + part[1] + part[2] + part[3]);
        const float peak = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
        const float per = sketch_per(peak), scale = per > 0.f ? peak / 127.f : 0.f;
        if (sketch) sketch[(size_t)doc * (SKETCH_BYTES / 4) + threadIdx.x] = sketch_pack(x, per);
        const float left = wave_sum_dpp(sketch_residual(x, per, scale));
        if (lane_id() == 0) rest[threadIdx.x / WAVE] = left;
        __syncthreads();
        if (threadIdx.x == 0) {
            dnorm[doc] = norm;
            // rounded up; a row with an entry that is no number or overflows half precision has no sketch (the same bound serves the half-precision rows)
            const float err = norm < __builtin_inff() && peak < 65504.f ? 1.0001f * sqrtf(rest[0] + rest[1] + rest[2] + rest[3]) : __builtin_inff();
            if (sketch) sketch_meta[doc] = SketchMeta{scale, err};
        }
        if (narrow) {
            float* vals = reinterpret_cast<float*>(rec + DENSE_BYTES);
            uint16_t* keys = reinterpret_cast<uint16_t*>(rec + DENSE_BYTES + narrow_keys_offset(nnz));
            signed char* codes = reinterpret_cast<signed char*>(rec + DENSE_BYTES + codes_offset(nnz));
            float per[2], step[2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
                const float m = fmaxf(fmaxf(most[p][0], most[p][1]), fmaxf(most[p][2], most[p][3]));
                const bool usable = m > 1e-30f; // below, half a step of 2e-30 covers the value
                per[p] = usable ? 127.f / m : 0.f;
                step[p] = usable ? m / 127.f : m > 0.f ? 2e-30f : 0.f;
            }
            auto put = [&](uint32_t j, float y, uint32_t key) {
                vals[j] = y;
                keys[j] = (uint16_t)key;
                if (coded) codes[j] = (signed char)sketch_code(y, j < ns ? per[0] : per[1]);
            };
            if (threadIdx.x < nnz) put(threadIdx.x, v, id);
            for (uint32_t j = threadIdx.x + 256; j < nnz; j += 256) put(j, value(j), term(j));
            // fill the alignment gaps so that a record never holds stale bytes
            for (uint32_t j = nnz + threadIdx.x; j < narrow_keys_offset(nnz) / 4; j += 256) vals[j] = 0.f;
            const uint32_t end = (uint32_t)(record_units(nnz, true, coded) * 16 - DENSE_BYTES);
            if (!coded) {
                for (uint32_t j = nnz + threadIdx.x; j < (end - narrow_keys_offset(nnz)) / 2; j += 256) keys[j] = 0xFFFFu;
            } else {
                const uint32_t scales = code_scales_offset(nnz);
                if (threadIdx.x < 2) reinterpret_cast<float*>(rec + DENSE_BYTES + scales)[threadIdx.x] = threadIdx.x ? step[1] : step[0];
                if (threadIdx.x < scales - codes_offset(nnz) - nnz) codes[nnz + threadIdx.x] = 0;
                for (uint32_t j = scales + 8 + 4 * threadIdx.x; j < end; j += 4 * 256) *reinterpret_cast<uint32_t*>(rec + DENSE_BYTES + j) = ~0u;
            }
        } else {
            uint2* sp = reinterpret_cast<uint2*>(rec + DENSE_BYTES);
            for (uint32_t j = threadIdx.x; j < ns; j += blockDim.x) sp[j] = make_uint2(s_idx[s0 + j], __float_as_uint(s_val[s0 + j]));
            for (uint32_t j = threadIdx.x; j < nb; j += blockDim.x)
                sp[ns + j] = make_uint2(b_idx[b0 + j] | BM25_BIT, __float_as_uint(b_val[b0 + j]));
            const uint32_t pair_slots = (uint32_t)(record_units(nnz, false, false) * 16 - DENSE_BYTES) / 8;
            for (uint32_t j = nnz + threadIdx.x; j < pair_slots; j += blockDim.x) sp[j] = make_uint2(EMPTY, 0u);
        }
    }
}

// Squared norms of the three parts of every sampled row (row i * n / sample), summed per wave: a wave takes rows w, w + ROW_SCALE_PARTS, ...
__global__ __launch_bounds__(256) void row_scale_kernel(uint32_t n, uint32_t sample, const float* __restrict__ dense, const uint32_t* __restrict__ s_off,
                                                        const float* __restrict__ s_val, const uint32_t* __restrict__ b_off, const float* __restrict__ b_val, float* out) {
    const uint32_t w = blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE, lane = lane_id();
    float sq[3] = {0.f, 0.f, 0.f};
    for (uint32_t i = w; i < sample; i += ROW_SCALE_PARTS) {
        const uint32_t doc = (uint32_t)((uint64_t)i * n / sample);
        const float4* row = reinterpret_cast<const float4*>(dense + (size_t)doc * DIM);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const float4 x = row[lane + WAVE * k];
            sq[0] += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
        }
        for (uint32_t j = s_off[doc] + lane; j < s_off[doc + 1]; j += WAVE) sq[1] = fmaf(s_val[j], s_val[j], sq[1]);
        for (uint32_t j = b_off[doc] + lane; j < b_off[doc + 1]; j += WAVE) sq[2] = fmaf(b_val[j], b_val[j], sq[2]);
    }
    for (int p = 0; p < 3; p++) {
        const float x = wave_sum_dpp(sq[p]);
        if (lane == 0) out[w * 3 + p] = x;
    }
}
int launch_row_scale(apoe_ctx* ctx, uint32_t n, uint32_t sample, const float* dense, const uint32_t* s_off, const float* s_val, const uint32_t* b_off, const float* b_val,
                     float* out_dev) {
    row_scale_kernel<<<ROW_SCALE_PARTS / (256 / WAVE), 256, 0, ctx->stream>>>(n, sample, dense, s_off, s_val, b_off, b_val, out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

int launch_pack(apoe_ctx* ctx, uint32_t n, const float* dense, const uint32_t* s_off, const uint32_t* s_idx, const float* s_val,
                const uint32_t* b_off, const uint32_t* b_idx, const float* b_val, const uint64_t* desc, char* recs, float* dnorm,
                SketchMeta* sketch_meta, uint32_t* sketch, bool narrow, bool coded) {
    uint32_t grid = n < 65536u * 16u ? n : 65536u * 16u;
    if (grid == 0) return APOE_OK;
    pack_kernel<<<grid, 256, 0, ctx->stream>>>(n, dense, s_off, s_idx, s_val, b_off, b_idx, b_val, desc, recs, dnorm, sketch_meta, sketch, narrow ? 1u : 0u, coded ? 1u : 0u);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// One workgroup (4 waves) per query and candidate chunk. The query's dense part is
// held in registers by every wave, its sparse terms sit in the LDS table; each wave
// takes every 4th candidate.
__global__ __launch_bounds__(256) void distance_batch_kernel(CorpusView C, SetView Q, float w_d, float w_s, float w_b, uint32_t paths,
                                                             const uint32_t* __restrict__ ids, uint32_t M, uint32_t chunk,
                                                             uint32_t slots, float* __restrict__ out) {
    extern __shared__ uint2 tab[];
    const uint32_t q = blockIdx.x, mask = slots - 1;
    const int tid = threadIdx.x, wave = tid / WAVE, lane = lane_id();
    term_table_clear(tab, slots, tid, blockDim.x);
    PivotDense pv;
    pivot_dense_load(pv, Q.dense + (size_t)q * DIM, w_d);
    __syncthreads();
    pivot_terms_from_query(tab, mask, Q, q, w_s, w_b, paths & PATH_SPARSE, paths & PATH_BM25, tid, blockDim.x);
    __syncthreads();
    const uint32_t m0 = blockIdx.y * chunk, m1 = min(M, m0 + chunk);
    for (uint32_t m = m0 + wave; m < m1; m += blockDim.x / WAVE) {
        const uint32_t id = ids[(size_t)q * M + m];
        float dist = INF_DIS;
        if (id < C.n) {
            EvalOut e = eval_wave(C, id, pv, tab, mask, paths, 1.0f);
            dist = 1.0f - e.ip;
        }
        if (lane == 0) out[(size_t)q * M + m] = dist;
    }
}

static uint32_t path_mask(const float* w3) {
    uint32_t p = 0;
    if (!(w3[0] < 1e-5f)) p |= PATH_DENSE;
    if (!(w3[1] < 1e-5f)) p |= PATH_SPARSE;
    if (!(w3[2] < 1e-5f)) p |= PATH_BM25;
    return p;
}

int launch_distance_batch(apoe_ctx* ctx, const apoe_corpus* c, const apoe_queries* q, const float* w3, const uint32_t* ids_dev,
                          uint32_t M, float* out_dev) {
    if (q->n == 0 || M == 0) return APOE_OK;
    const uint32_t slots = next_pow2(std::max(64u, 2 * q->max_nnz));
    const size_t lds = (size_t)slots * sizeof(uint2);
    APOE_REQUIRE(lds <= 64 * 1024, "query rows with %u sparse terms exceed the LDS term table", q->max_nnz);
    const uint32_t chunk = 1024;
    dim3 grid(q->n, (M + chunk - 1) / chunk);
    distance_batch_kernel<<<grid, 256, lds, ctx->stream>>>(c->view(), q->view(), w3[0], w3[1], w3[2], path_mask(w3), ids_dev, M, chunk,
                                                           slots, out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// One wave per pair: document a is the pivot, document b the candidate.
__global__ __launch_bounds__(64) void distance_pairs_kernel(CorpusView C, float dense_mul, const uint32_t* __restrict__ a,
                                                            const uint32_t* __restrict__ b, uint32_t n_pairs, uint32_t slots,
                                                            float* __restrict__ out) {
    extern __shared__ uint2 tab[];
    const uint32_t mask = slots - 1;
    const int lane = lane_id();
    for (uint32_t t = blockIdx.x; t < n_pairs; t += gridDim.x) {
        const uint32_t ia = a[t], ib = b[t];
        float dist = INF_DIS;
        if (ia < C.n && ib < C.n) {
            term_table_clear(tab, slots, lane, WAVE);
            __syncthreads();
            const uint64_t d = C.desc[ia];
            const char* rec = C.recs + desc_off(d) * 16;
            PivotDense pv;
            pivot_dense_load(pv, reinterpret_cast<const float*>(rec), 1.0f);
            pivot_terms_from_record(tab, mask, record_pairs(C, d), lane, WAVE);
            __syncthreads();
            EvalOut e = eval_wave(C, ib, pv, tab, mask, PATH_DENSE | PATH_SPARSE | PATH_BM25, dense_mul);
            dist = 1.0f - e.ip;
            __syncthreads();
        }
        if (lane == 0) out[t] = dist;
    }
}

int launch_distance_pairs(apoe_ctx* ctx, const apoe_corpus* c, float dense_scale, const uint32_t* a_dev, const uint32_t* b_dev,
                          uint32_t n_pairs, float* out_dev) {
    if (n_pairs == 0) return APOE_OK;
    const uint32_t slots = next_pow2(std::max(64u, 2 * (c->max_nnz_s + c->max_nnz_b)));
    const size_t lds = (size_t)slots * sizeof(uint2);
    APOE_REQUIRE(lds <= 64 * 1024, "document rows with %u sparse terms exceed the LDS term table", c->max_nnz_s + c->max_nnz_b);
    uint32_t grid = std::min<uint32_t>(n_pairs, 1u << 20);
    distance_pairs_kernel<<<grid, 64, lds, ctx->stream>>>(c->view(), dense_scale * dense_scale, a_dev, b_dev, n_pairs, slots, out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// One wave per document: the dense row rounded to half precision (round to nearest even), 2 KB per row.
__global__ __launch_bounds__(256) void half_rows_kernel(CorpusView C, uint16_t* __restrict__ out) {
    const int lane = lane_id();
    const uint32_t waves = gridDim.x * (blockDim.x / WAVE);
    for (uint32_t doc = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE; doc < C.n; doc += waves) {
        const float4* r = reinterpret_cast<const float4*>(C.recs + desc_off(C.desc[doc]) * 16);
        uint2* o = reinterpret_cast<uint2*>(out + (size_t)doc * DIM);
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const float4 x = r[lane + WAVE * i];
            const uint32_t a = __builtin_bit_cast(uint16_t, (_Float16)x.x), b = __builtin_bit_cast(uint16_t, (_Float16)x.y);
            const uint32_t c = __builtin_bit_cast(uint16_t, (_Float16)x.z), d = __builtin_bit_cast(uint16_t, (_Float16)x.w);
            o[lane + WAVE * i] = make_uint2(a | (b << 16), c | (d << 16));
        }
    }
}

int launch_half_rows(apoe_ctx* ctx, const apoe_corpus* c, uint16_t* out_dev) {
    if (c->n == 0) return APOE_OK;
    uint32_t grid = std::min<uint32_t>((c->n + 3) / 4, 1u << 16);
    half_rows_kernel<<<grid, 256, 0, ctx->stream>>>(c->view(), out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

// One wave per document: dense_mul*|dense|^2 + sum of squared pair values.
__global__ __launch_bounds__(256) void norms_kernel(CorpusView C, float dense_mul, float* __restrict__ out) {
    const int lane = lane_id();
    const uint32_t waves = gridDim.x * (blockDim.x / WAVE);
    for (uint32_t doc = blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE; doc < C.n; doc += waves) {
        const uint64_t d = C.desc[doc];
        const char* rec = C.recs + desc_off(d) * 16;
        const float4* r = reinterpret_cast<const float4*>(rec);
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            float4 x = r[lane + WAVE * i];
            acc += x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w;
        }
        acc *= dense_mul;
        const Pairs sp = record_pairs(C, d);
        for (uint32_t j = lane; j < sp.nnz; j += WAVE) {
            float v = __uint_as_float(sp[j].y);
            acc = fmaf(v, v, acc);
        }
        acc = wave_sum(acc);
        if (lane == 0) out[doc] = acc;
    }
}

int launch_norms(apoe_ctx* ctx, const apoe_corpus* c, float dense_scale, float* out_dev) {
    if (c->n == 0) return APOE_OK;
    uint32_t grid = std::min<uint32_t>((c->n + 3) / 4, 1u << 16);
    norms_kernel<<<grid, 256, 0, ctx->stream>>>(c->view(), dense_scale * dense_scale, out_dev);
    APOE_HIP(hipGetLastError());
    return APOE_OK;
}

} // namespace apoe
