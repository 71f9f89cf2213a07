// Scores of a few query tokens against V2 keys in one launch (upstream turboquant/compressors.py:124-158):
//   score[row][q][t] = norm_t * (Pi q) . centroids[codes_t]  +  residual_norm_t * (c S q) . signs_t ,  c = sqrt(pi/2) / 128
// from the raw queries: they are rotated and projected inside (two 128 x 128 float32 products a block), so that a decode step is one launch
// instead of a conversion, two library products and tq_qjl_scores.  More query tokens than MAX_Q take that way still: the products
// are then worth a launch of their own.
#include "tq_lut.h"

namespace {

struct QueryScoreArgs {
    const uint8_t *idx_bytes;
    const uint16_t *vec_norms;
    const uint8_t *sign_bytes;
    const uint16_t *residual_norm;
    const uint8_t *table;
    const float *both;       // [2, 128, 128]: Pi^T, c S^T
    const uint8_t *queries;  // [rows, n_q, 128]
    float *scores;           // [rows, n_q, tokens]
    uint32_t tokens, n_q, chunk;
    int dtype;
};

constexpr int QD = TQ_HEAD_DIM;
constexpr int QW = LUT_THREADS / TQ_WAVE;
constexpr int MAX_Q = 8;

// Block (part of the tokens, row) of eight waves, one per compute unit: its waves share the tables of codes (byte -> centroids) and signs (byte ->
// eight times +-1), spread over the banks.  A wave takes runs of 64 tokens, loaded one run ahead; a lane holds 32 coordinates of one of 16
// tokens and a column of the 16x16x32 products is a query: two fp16 terms of the rotated one against the codes, one of the projected
// one against the signs (that term is a correction of the size of the quantisation residual).  Bound by its start, products of the
// queries and tables; us a call, conversion, two products and tq_qjl_scores before / this: 8 rows x 32768 tokens, 2-bit codes (14 MB, 3 us), 1
// query 26.7 / 9.2; 128 x 45 26.4 / 6.1; 256 x 1500, 3-bit codes 44.0 / 12.4; 1 x 500000, 3-bit codes, 8 queries 38.5 / 17.7.
// MAX_Q: the parts of the products of 8 queries take 64 of the 160 KiB of LDS, the tables another 64.
template <int IPB>
__global__ __launch_bounds__(LUT_THREADS) void tq_qjl_query_scores_kernel(QueryScoreArgs a) {
    constexpr int KB = QD / 4 / IPB, NW = KB / 4;        // bytes and words of codes of a lane (32 coordinates)
    constexpr int PARTS = 8, ROWS = QD / PARTS;          // the contraction over a query's coordinates in parts of 16
    __shared__ __attribute__((aligned(1024))) uint8_t lds_lut[65536];
    __shared__ __attribute__((aligned(16))) float lds_part[PARTS][2][MAX_Q][QD];
    __shared__ __attribute__((aligned(16))) float lds_q[2][MAX_Q][QD + 4];
    __shared__ __attribute__((aligned(16))) float lds_in[MAX_Q][QD];
    __shared__ __attribute__((aligned(16))) float lds_norm[QW][2][64];

    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tq_uniform32(tid >> 6);
    const uint32_t row = blockIdx.y, n16 = lane & 15u, q4 = lane >> 4;
    const uint32_t t_begin = blockIdx.x * a.chunk, t_end = min(a.tokens, t_begin + a.chunk);
    const size_t slot0 = (size_t)row * a.tokens;

    // ---- loads in the order of their use: queries, the matrices, the table, the first run
    const uint32_t nq = a.n_q, qn = nq * QD;
    uint32_t qv[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t e = min(tid + k * LUT_THREADS, qn - 1u);
        const TQ_GLOBAL uint8_t *q = (const TQ_GLOBAL uint8_t *)a.queries;
        const size_t at = (size_t)row * qn + e;
        qv[k] = a.dtype == TQ_F32 ? ((const TQ_GLOBAL uint32_t *)q)[at] : (uint32_t)((const TQ_GLOBAL uint16_t *)q)[at];
    }
    const uint32_t mat = (tid >> 5) & 1u, c4 = (tid & 31u) * 4u, kp = tid >> 6;       // four columns of a matrix, part of the contraction
    tq_u4 m4[ROWS];
#pragma unroll
    for (int k = 0; k < ROWS; ++k) m4[k] = tq_gload16(reinterpret_cast<const uint8_t *>(a.both + ((size_t)mat * QD + kp * ROWS + k) * QD + c4));
    Lut<IPB> table;
    table.load(a.table + TQ_OFF_LUT(QD), tid);
    uint32_t raw[4][NW], sraw[4];
    uint16_t nrm, rnrm;
    auto issue = [&](uint32_t t0) __attribute__((always_inline)) {       // past the end the last token is read again
        const uint32_t last = t_end - 1u - t0;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const size_t slot = slot0 + t0 + min(16u * b + n16, last);
            const uint8_t *src = a.idx_bytes + slot * (4 * KB) + q4 * KB;
            if constexpr (KB % 16 == 0) {
#pragma unroll
                for (int p = 0; p < KB / 16; ++p) {
                    const tq_u4 v = tq_gload16(src + 16 * p);
#pragma unroll
                    for (int i = 0; i < 4; ++i) raw[b][4 * p + i] = v[i];
                }
            } else if constexpr (KB == 8) {
                const tq_u2 v = tq_gload8(src);
                raw[b][0] = v[0]; raw[b][1] = v[1];
            } else {
                raw[b][0] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)src);
            }
            sraw[b] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)a.sign_bytes + slot * 16u + q4 * 4u);
        }
        nrm = tq_gload2(a.vec_norms + slot0 + t0 + min(lane, last));
        rnrm = tq_gload2(a.residual_norm + slot0 + t0 + min(lane, last));
    };
    uint32_t t0 = t_begin + wave * 64u;
    __builtin_amdgcn_sched_barrier(0);
    issue(t0 < t_end ? t0 : t_begin);
    __builtin_amdgcn_sched_barrier(0);

    // ---- queries to LDS as float32, tables
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t e = tid + k * LUT_THREADS;
        const float x = a.dtype == TQ_F32 ? __uint_as_float(qv[k]) : a.dtype == TQ_BF16 ? __uint_as_float(qv[k] << 16) : (float)__builtin_bit_cast(_Float16, (uint16_t)qv[k]);
        if (e < qn) lds_in[e / QD][e % QD] = x;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {        // signs: bit 7 - i of a byte belongs to coordinate i
        const uint32_t piece = k * LUT_THREADS + tid, byte = piece >> 3;
        tq_u4 e;
#pragma unroll
        for (int d = 0; d < 4; ++d)
            e[d] = 0x3c003c00u | (((byte >> (7 - 2 * d)) & 1u) ? 0u : 0x8000u) | (((byte >> (6 - 2 * d)) & 1u) ? 0u : 0x80000000u);
        *reinterpret_cast<tq_u4 *>(lds_lut + byte * 256u + 128u + (piece & 7u) * 16u) = e;
    }
    __syncthreads();
    for (uint32_t g = 0; g < nq; ++g) {
        float x[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < ROWS; k += 4) {
            const float4 q = *reinterpret_cast<const float4 *>(&lds_in[g][kp * ROWS + k]);
            const float qk[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) x[c] = fmaf(qk[i], __uint_as_float(m4[k + i][c]), x[c]);
        }
        *reinterpret_cast<float4 *>(&lds_part[kp][mat][g][c4]) = make_float4(x[0], x[1], x[2], x[3]);
    }
    table.store(lds_lut, tid);
    __syncthreads();
    for (uint32_t p = tid; p < 2u * qn; p += LUT_THREADS) {
        const uint32_t m = p / qn, e = p - m * qn;
        float v = 0.f;
#pragma unroll
        for (int k = 0; k < PARTS; ++k) v += lds_part[k][m][e / QD][e % QD];
        lds_q[m][e / QD][e % QD] = v;
    }
    __syncthreads();

    // ---- B operands: fp16 terms of q * 2^(10 - e), e = binary exponent of the query's largest magnitude
    tq_u4 qb[3][4];
    float scale[2];
    const bool live = n16 < nq;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
        float x[32], big = 0.f;
#pragma unroll
        for (int i = 0; i < 32; i += 4) {
            const float4 f = *reinterpret_cast<const float4 *>(&lds_q[m][live ? n16 : 0u][32u * q4 + i]);
            x[i] = f.x; x[i + 1] = f.y; x[i + 2] = f.z; x[i + 3] = f.w;
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) big = fmaxf(big, fabsf(x[i]));
        big = reduce_rows(big, OpMax());
        int e = 0;
        if (big > 0.f && big < __builtin_inff()) (void)frexpf(big, &e);
        e = e < -100 ? -100 : e;             // rows that small give zero scores either way; keeps 2^(10-e) finite
        const float up = ldexpf(1.f, TQ_F16_PI_SHIFT - e);
        scale[m] = ldexpf(1.f, e - TQ_F16_PI_SHIFT);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            tq_half8 hi, lo;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float y = x[8 * s + i] * up;
                hi[i] = (_Float16)y;
                lo[i] = (_Float16)(y - (float)hi[i]);
            }
            qb[2 * m][s] = __builtin_bit_cast(tq_u4, hi);
            if (m == 0) qb[1][s] = __builtin_bit_cast(tq_u4, lo);
        }
    }

    const uint32_t slot_k = RepLut<IPB>::lane_offset(lane), slot_s = 128u + RepLut<8>::lane_offset(lane);
    TQ_GLOBAL float *out = (TQ_GLOBAL float *)a.scores + ((size_t)row * nq + (live ? n16 : 0u)) * a.tokens;
    for (; t0 < t_end; t0 += 64u * QW) {
        lds_norm[wave][0][lane] = (float)__builtin_bit_cast(_Float16, nrm);
        lds_norm[wave][1][lane] = (float)__builtin_bit_cast(_Float16, rnrm);
        tq_f4v sc[4], ss[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            sc[b] = ss[b] = tq_f4v{0.f, 0.f, 0.f, 0.f};
            const uint32_t signs[1] = {sraw[b]};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const tq_u4 kd = decode_keys<IPB, NW>(raw[b], s, lds_lut, slot_k);
                sc[b] = mfma16_f16(kd, qb[0][s], sc[b]);
                sc[b] = mfma16_f16(kd, qb[1][s], sc[b]);
                ss[b] = mfma16_f16(decode_keys<8, 1>(signs, s, lds_lut, slot_s), qb[2][s], ss[b]);
            }
        }
        const uint32_t t_next = t0 + 64u * QW;
        issue(t_next < t_end ? t_next : t_begin);
        asm volatile("" ::: "memory");       // (the LDS serves a wave in order)
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const uint32_t tl = 16u * b + 4u * q4;
            const float4 n4 = *reinterpret_cast<const float4 *>(&lds_norm[wave][0][tl]), r4 = *reinterpret_cast<const float4 *>(&lds_norm[wave][1][tl]);
            const float nn[4] = {n4.x, n4.y, n4.z, n4.w}, rr[4] = {r4.x, r4.y, r4.z, r4.w};
            tq_u4 v;
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = __float_as_uint(fmaf(ss[b][r] * scale[1], rr[r], sc[b][r] * scale[0] * nn[r]));
            if (live) {
                if (t0 + tl + 4u <= t_end) {
                    typedef uint32_t u4_any __attribute__((ext_vector_type(4), aligned(4)));
                    *reinterpret_cast<TQ_GLOBAL u4_any *>(out + t0 + tl) = v;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (t0 + tl + r < t_end) out[t0 + tl + r] = __uint_as_float(v[r]);
                }
            }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace

extern "C" int tq_qjl_query_scores(const uint8_t *idx_bytes, const uint16_t *vec_norms, const uint8_t *sign_bytes, const uint16_t *residual_norm,
                                   long long rows, long long tokens, const void *table_dev, const float *both_dev, int head_dim, int mse_bits,
                                   const void *queries, int dtype, long long n_queries, float *scores, void *stream) {
    if (head_dim != QD) return TQ_ERR_HEAD_DIM;
    if (mse_bits < 1 || mse_bits > 8) return TQ_ERR_BITS;
    if (dtype != TQ_F32 && dtype != TQ_F16 && dtype != TQ_BF16) return TQ_ERR_DTYPE;
    if (rows < 0 || rows > 65535 || tokens < 0 || n_queries < 0 || n_queries > MAX_Q) return TQ_ERR_SIZE;
    if (rows == 0 || tokens == 0 || n_queries == 0) return TQ_OK;
    if (tokens > 0x7fffffffll / rows) return TQ_ERR_SIZE;
    if (!idx_bytes || !vec_norms || !sign_bytes || !residual_norm || !table_dev || !both_dev || !queries || !scores) return TQ_ERR_NULL;
    if (((uintptr_t)idx_bytes & 15u) || ((uintptr_t)vec_norms & 1u) || ((uintptr_t)sign_bytes & 3u) || ((uintptr_t)residual_norm & 1u) || ((uintptr_t)table_dev & 15u) ||
        ((uintptr_t)both_dev & 15u) || ((uintptr_t)queries & (dtype == TQ_F32 ? 3u : 1u)) || ((uintptr_t)scores & 3u))
        return TQ_ERR_ALIGN;
    int cus = 0;
    const int rc = tq_device_cus(cus);
    if (rc) return rc;
    QueryScoreArgs a;
    a.idx_bytes = idx_bytes;
    a.vec_norms = vec_norms;
    a.sign_bytes = sign_bytes;
    a.residual_norm = residual_norm;
    a.table = static_cast<const uint8_t *>(table_dev);
    a.both = both_dev;
    a.queries = static_cast<const uint8_t *>(queries);
    a.scores = scores;
    a.tokens = (uint32_t)tokens;
    a.n_q = (uint32_t)n_queries;
    a.dtype = dtype;
    // one block per compute unit, and none with less than a run for each of its waves
    long long parts = (cus + rows - 1) / rows;
    const long long most = (tokens + 64 * QW - 1) / (64 * QW);
    if (parts > most) parts = most;
    a.chunk = (uint32_t)(((tokens + parts - 1) / parts + 63) / 64 * 64);
    const dim3 grid((unsigned)((tokens + a.chunk - 1) / a.chunk), (unsigned)rows, 1), block(LUT_THREADS);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    switch (8 / mse_bits) {
        case 8: hipLaunchKernelGGL(tq_qjl_query_scores_kernel<8>, grid, block, 0, s, a); break;
        case 4: hipLaunchKernelGGL(tq_qjl_query_scores_kernel<4>, grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL(tq_qjl_query_scores_kernel<2>, grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL(tq_qjl_query_scores_kernel<1>, grid, block, 0, s, a); break;
    }
    return (int)hipGetLastError();
}
