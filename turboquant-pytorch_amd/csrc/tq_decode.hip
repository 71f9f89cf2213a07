// One decode step of a streaming cache layer in two launches, for head dimensions 64, 96, 128 and 256 and 16-bit elements:
//   tq_decode_append   the token that leaves the window is compressed into the next packed slot and the new token takes its
//                      window slot, keys and values, every row, in one launch;
//   tq_decode_attend   softmax(scale q K^T) V over the packed history and the uncompressed window, one launch: the queries are
//                      rotated, the window is attended to and the splits are merged inside the kernel that reads the codes.
// Few rows: a step is a chain of latencies (tables, query rotation, one or two runs per wave, merge), so launches are what
// counts; many rows: the main loop, which is bound by the vector and LDS work of the table lookups (counted on this kernel at
// 512 rows x 16384 tokens: vector instructions take 60 % of the issue slots, the LDS is busy 44 % of the time).
// Per layer and whole step, six launches / these two (MI355X): 8 rows x 32768 tokens, K4/V2, 4 heads a row 48.9 -> 30.1 us;
// 512 rows x 16384 tokens 226 -> 212 us, of which attention 200-204; head dimension 64, 32 rows x 6000 tokens, K6/V4 (before:
// de-quantised to float32 and multiplied by library products) 190 -> 25 us.  Attention alone at 256, 32 rows x 6000 tokens, before /
// this: K4/V2 307 -> 43 us, K8/V8 344 -> 58 us.
// What they compute is what tq_compress and the prepare / partials / merge trio of tq_attend.hip compute (upstream
// turboquant/generation_test_v2.py:96-135, score definition validate_v3.py:87); at 128 those remain for float32 caches, queries of
// another type than the cache's and more than 65535 rows.  A value whose norm is infinite in float16 makes its row's results NaN, as there.
#include <type_traits>

#include "tq_device.h"

namespace {

typedef float tq_f4v __attribute__((ext_vector_type(4)));

struct DecodeArgs {
    const uint8_t *queries;          // [rows, group, D] 16-bit elements, contiguous
    const uint8_t *k_idx, *v_idx;
    const uint16_t *k_norms, *v_norms;
    const uint8_t *table_k, *table_v;
    const float *pi_v;               // [D, D] rotation of the value codec
    const uint8_t *k_win, *v_win;    // row r, token t at element r * win_stride + t * D
    float *partial;                  // [rows, splits, group, D + 2]: reference score, sum of exp, D sums in the rotated value space
    float *win_part;                 // [rows, window tiles, group, D + 2]: the same over 32 window tokens, sums in the plain space
    uint32_t *arrived;               // [rows] blocks of the row that are done; zero before and after every launch (splits > 1)
    uint8_t *out;                    // [rows, group, D]
    long long win_stride;
    float scale;
    uint32_t tokens, packed_row_stride, group, chunk, n_win, bf16;
};

constexpr int DW = 8;                // waves per block: one block per compute unit (two waves per SIMD), its waves share the tables
constexpr int DTHREADS = DW * TQ_WAVE;
constexpr int MAX_GROUP = 16;
constexpr int WIN_TILE = 32;
constexpr int MAX_WINDOW = 512;
constexpr int MAX_SPLITS = 256;     // (the merge keeps a weight per record and head in 32 KiB of LDS)
static_assert(MAX_GROUP * (MAX_SPLITS + MAX_WINDOW / WIN_TILE) * 4 <= 32768, "weights of the records");

__device__ __forceinline__ tq_f4v mfma16_f16(tq_u4 a, tq_u4 b, tq_f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(tq_half8, a), __builtin_bit_cast(tq_half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ tq_f4v mfma16_bf16(tq_u4 a, tq_u4 b, tq_f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tq_bf8, a), __builtin_bit_cast(tq_bf8, b), c, 0, 0, 0);
}

// Exact split of eight fp16 values into two bf16 terms each: a truncation keeps eight of the eleven bits, the rest fits the second.
__device__ __forceinline__ void split_f16x8(tq_u4 v, tq_u4 &hi, tq_u4 &lo) {
    const tq_half8 h = __builtin_bit_cast(tq_half8, v);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint32_t x0 = __float_as_uint((float)h[2 * d]), x1 = __float_as_uint((float)h[2 * d + 1]);
        const uint32_t r0 = __float_as_uint(__uint_as_float(x0) - __uint_as_float(x0 & 0xffff0000u));
        const uint32_t r1 = __float_as_uint(__uint_as_float(x1) - __uint_as_float(x1 & 0xffff0000u));
        hi[d] = __builtin_amdgcn_perm(x1, x0, 0x07060302u);
        lo[d] = __builtin_amdgcn_perm(r1, r0, 0x07060302u);
    }
}

// Records of a row with several splits travel between blocks past the caches that are not shared (stores and loads of device
// scope), so that nothing has to be written back or invalidated around the arrival counter: with fences there a step of
// 8 rows x 32768 tokens took 32.0 us and now 30.0, one of 32 rows x 6000 tokens, 64 wide, 27.3 and now 24.7.  A row with one split keeps
// its records in its own block: they stay cached (512 rows x 16384 tokens: 2 % longer otherwise).
// No release and acquire of the language stand behind this order, all accesses are relaxed: it rests on the hardware, where a
// store of device scope counts in vmcnt until every compute unit sees it, and on both sides going through put_record and
// get_record.  Plain accesses to a record of a row with several splits would be a race.
__device__ __forceinline__ void put_record(bool across, TQ_GLOBAL float *p, float v) {
    if (across) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
template <bool ACROSS>
__device__ __forceinline__ float get_record(const TQ_GLOBAL float *p) {
    if constexpr (ACROSS) return __hip_atomic_load(const_cast<TQ_GLOBAL float *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else return *p;
}

// The byte -> centroids table spread over the banks (RepLut): consecutive threads write consecutive 16-byte pieces, so the
// writes are free of conflicts; the eight threads of a table row read the same entry.
template <int IPB>
__device__ __forceinline__ void stage_lut(uint8_t *lds, const uint8_t *src, uint32_t tid) {
    constexpr int ES = 2 * IPB;
    constexpr int TRIPS = 256 * 8 / DTHREADS;
    tq_u4 v[TRIPS];
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) {
        const TQ_GLOBAL uint8_t *g = (const TQ_GLOBAL uint8_t *)src + ((k * DTHREADS + tid) >> 3) * ES;
        if constexpr (ES == 2) {
            const uint32_t x = *reinterpret_cast<const TQ_GLOBAL uint16_t *>(g);
            v[k] = tq_u4{x, x, x, x};
        } else if constexpr (ES == 4) {
            const uint32_t x = *reinterpret_cast<const TQ_GLOBAL uint32_t *>(g);
            v[k] = tq_u4{x, x, x, x};
        } else if constexpr (ES == 8) {
            const tq_u2 x = *reinterpret_cast<const TQ_GLOBAL tq_u2 *>(g);
            v[k] = tq_u4{x[0], x[1], x[0], x[1]};
        } else {
            v[k] = *reinterpret_cast<const TQ_GLOBAL tq_u4 *>(g);
        }
    }
#pragma unroll
    for (int k = 0; k < TRIPS; ++k) *reinterpret_cast<tq_u4 *>(lds + (k * DTHREADS + tid) * 16u) = v[k];
}

// Coordinates of a lane on the value side, D / 16 of them: contiguous for multiples of 64; four of the first 64 and two of
// the last 32 for 96, so that a group of them never starts inside a packed byte that another lane shares more than once.
template <int D>
__device__ __forceinline__ uint32_t value_coord(uint32_t n16, int c) {
    if constexpr (D % 64 == 0) return n16 * (D / 16) + (uint32_t)c;
    else return c < 4 ? 4u * n16 + (uint32_t)c : (uint32_t)(D - 32) + 2u * n16 + (uint32_t)(c - 4);
}

// N consecutive coordinates (8, 4 or 2) of a staged value vector -> fp16 pairs; `codes` points at the vector's packed bytes,
// first = index of the first coordinate.
template <int IPB, int N>
__device__ __forceinline__ void decode_values(const uint8_t *codes, uint32_t first, const uint8_t *lut, uint32_t (&out)[N / 2]) {
    if constexpr (IPB == 8) {
        static_assert(N == 8, "whole bytes");
        const tq_u4 v = *reinterpret_cast<const tq_u4 *>(lut + ((uint32_t)codes[first / 8u] << 7));
        out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; out[3] = v[3];
    } else if constexpr (IPB == 4) {
        if constexpr (N == 8) {
            const uint32_t two = *reinterpret_cast<const uint16_t *>(codes + first / 4u);
            const tq_u2 a = *reinterpret_cast<const tq_u2 *>(lut + ((two & 0xffu) << 7));
            const tq_u2 b = *reinterpret_cast<const tq_u2 *>(lut + ((two >> 8) << 7));
            out[0] = a[0]; out[1] = a[1]; out[2] = b[0]; out[3] = b[1];
        } else if constexpr (N == 4) {
            const tq_u2 a = *reinterpret_cast<const tq_u2 *>(lut + ((uint32_t)codes[first / 4u] << 7));
            out[0] = a[0]; out[1] = a[1];
        } else {        // half a byte
            out[0] = *reinterpret_cast<const uint32_t *>(lut + ((uint32_t)codes[first / 4u] << 7) + 2u * (first & 3u));
        }
    } else if constexpr (IPB == 2) {
        uint32_t raw;
        if constexpr (N == 8) raw = *reinterpret_cast<const uint32_t *>(codes + first / 2u);
        else if constexpr (N == 4) raw = *reinterpret_cast<const uint16_t *>(codes + first / 2u);
        else raw = codes[first / 2u];
#pragma unroll
        for (int i = 0; i < N / 2; ++i) out[i] = *reinterpret_cast<const uint32_t *>(lut + (((raw >> (8 * i)) & 0xffu) << 7));
    } else {
        uint32_t raw[2] = {0u, 0u};
        if constexpr (N == 8) { const tq_u2 v = *reinterpret_cast<const tq_u2 *>(codes + first); raw[0] = v[0]; raw[1] = v[1]; }
        else if constexpr (N == 4) raw[0] = *reinterpret_cast<const uint32_t *>(codes + first);
        else raw[0] = *reinterpret_cast<const uint16_t *>(codes + first);
#pragma unroll
        for (int i = 0; i < N / 2; ++i) {
            const uint32_t b = raw[i / 2] >> (16 * (i & 1));
            const uint32_t lo = *reinterpret_cast<const uint16_t *>(lut + ((b & 0xffu) << 7));
            const uint32_t hi = *reinterpret_cast<const uint16_t *>(lut + (((b >> 8) & 0xffu) << 7));
            out[i] = lo | (hi << 16);
        }
    }
}

// Block (split, row), eight waves.  The main loop is the one of tq_attend_kernel (tq_attend.hip): a wave takes runs of 32 or 64
// tokens of the split, loaded one run ahead; scores transposed (A = decoded keys, B = rotated queries, heads padded to 16
// columns), softmax in base 2 against a lazily moved per-head reference, probabilities times value norms as the A operand
// of the value product, whose B operand is built in the lanes from the staged codes.  Around it, in the same launch:
//   * waves 0 .. D/32 - 1 rotate the row's queries on the matrix cores (operands of the key codec's table; Pi as three bf16 terms that
//     add up to its float32 value, or for fp16 queries as two fp16 terms, 22 bits), while the other waves attend to the window, 32 tokens each: raw 16-bit keys and queries multiply exactly,
//     probabilities enter the value product as three bf16 terms that add up to their float32 value, fp16 values as two that add up to
//     theirs (two fp16 terms of a probability lie on a grid of 2^-38 of the largest one: at 2^-30 of it eight bits were left);
//   * the waves' sums meet in LDS; with several splits per row the block that arrives last at the row's counter merges the
//     records of all splits and of the window, rotates the value sums back and stores the result.
// At 128 queries (against 8-bit keys: two terms) and weights enter the packed products as one fp16 term, as in tq_attend_kernel:
// their 2^-12 roundings stay under what the fp16 centroids cost.  The other head dimensions are as exact as float32 arithmetic:
//   * queries enter as two fp16 terms, Pi of fp16 caches as well (22 bits each).  Logits that come about by cancellation, where the
//     roundings show, are off by 0.5 to 0.8 of what the same products in float32 are off by (rotation and score, 64 to 256 wide).
//   * weights enter as three fp16 terms of p * 2^P_SHIFT * (value norm / 2^ev_ref) <= 2^15: 24 bits or more down to 2^-10 of the
//     reference weight times the largest value norm's binade, a grid of 2^-34 of that below (the smaller SLACK_LOG2, the finer).
//     Two terms on a grid of 2^-30 lost up to 2^-8 of weights around 2^-22 of the reference, a short history behind one token
//     that takes nearly everything.  The third one costs 4 to 5 % where rows are many (96 wide, 512 rows x 8000 tokens: 102 -> 107 us).
template <int D, int IPBK, int IPBV>
__global__ __launch_bounds__(DTHREADS, DW / 4) void tq_decode_kernel(DecodeArgs a) {
    constexpr int QT = D != 128 || IPBK == 1 ? 2 : 1;    // fp16 terms of a rotated query
    constexpr int QREG = D == 256 && (IPBK == 1 || IPBV == 1) ? 1 : QT;      // terms held in registers, the others in LDS (see below)
    constexpr int PT = D != 128 ? 3 : 1;                 // fp16 terms of a weight
    constexpr int SETS = D == 256 ? 1 : 2;               // register sets of the loads that run one run ahead
    constexpr int PART = D + 2;
    constexpr int STEPS = D / 16, TILES = D / 32;        // query rotation: 32x32x16 matrix instructions
    constexpr int SK = D / 32;                           // score product: steps of 32 coordinates, 8 per lane
    constexpr int NC = D / 16;                           // value coordinates per lane
    constexpr int KB = D / 4 / IPBK;                     // key bytes per lane and token (D / 4 coordinates)
    constexpr int NWK = (KB + 3) / 4;
    constexpr int GBV = D / IPBV;                        // value bytes per vector
    constexpr int RUN = (D == 256 || (D > 64 && (IPBK == 1 || IPBV == 1))) ? 32 : 64;     // tokens per wave and trip
    constexpr int SUB = RUN / 32;
    constexpr int VPB = GBV % 16 ? 8 : 16;               // value codes are staged in pieces of this size
    constexpr int VBYTES = RUN * GBV, VPIECES = VBYTES / VPB, NVP = (VPIECES + 63) / 64;
    constexpr int SLACK_LOG2 = PT == 1 ? 8 : 4;          // (several terms: the smaller it is, the finer the grid of small weights)
    constexpr int P_SHIFT = 14 - SLACK_LOG2;             // p * 2^P_SHIFT * (value norm / 2^ev_ref < 2) <= 2^15 fits fp16
    constexpr int HR = D == 256 ? 8 : MAX_GROUP;         // heads per round of the merge through LDS
    constexpr int AREA = VBYTES > HR * PART * 4 ? VBYTES : HR * PART * 4;    // per wave: staged value codes, later its sums
    constexpr int QROW = D + 4;                          // rotated queries in LDS, floats per head
    constexpr int ROTP = DTHREADS / (D / 4) >= 16 ? 16 : DTHREADS / (D / 4);     // parts of the contraction when rotating back
    constexpr int ROTK = D / ROTP;                       // rows of Pi_v per part
    static_assert(DW * AREA >= MAX_GROUP * QROW * 4 && DW * AREA >= 2 * MAX_GROUP * D * 4 && ROTP * 4 * D * 4 <= 32768, "LDS areas too small");

    __shared__ __attribute__((aligned(16))) uint8_t lds_lut_k[32768];
    __shared__ __attribute__((aligned(16))) uint8_t lds_lut_v[32768];
    __shared__ __attribute__((aligned(16))) uint8_t lds_area[DW][AREA];
    __shared__ __attribute__((aligned(16))) float lds_kn[DW][RUN];
    __shared__ __attribute__((aligned(16))) std::conditional_t<PT == 1, uint16_t, float> lds_vn[DW][RUN];     // value norms / 2^ev_ref (uint16_t: as fp16)
    __shared__ __attribute__((aligned(16))) tq_u4 lds_q[QT > QREG ? (QT - QREG) * SK : 1][TQ_WAVE];
    __shared__ __attribute__((aligned(16))) float lds_corr[DW][16];
    __shared__ float lds_den[MAX_GROUP];
    __shared__ uint32_t lds_last;
    __shared__ uint32_t lds_trips[DW];                   // runs a wave has begun

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = tq_uniform32(tid >> 6);
    const uint32_t row = blockIdx.y, split = blockIdx.x, splits = gridDim.x;
    const uint32_t n16 = lane & 15u, q4 = lane >> 4;
    const TqTableHeader *hk_hd = reinterpret_cast<const TqTableHeader *>(a.table_k);
    const TqTableHeader *hv_hd = reinterpret_cast<const TqTableHeader *>(a.table_v);
    const uint32_t G = a.group;
    const bool live = n16 < G;

    const uint32_t t_begin = min(a.tokens, split * a.chunk);
    const uint32_t t_end = min(a.tokens, t_begin + a.chunk);
    const size_t slot0 = (size_t)row * a.packed_row_stride;
    uint8_t *vcodes = lds_area[wave];

    // Loads of a run, issued one run ahead into the other of two register sets.  At 256, where registers are short, there is
    // one set: values and norms are loaded again as soon as the run has been staged, keys when its scores are done.
    uint32_t kraw_buf[SETS][SUB][2][NWK];
    tq_u4 vpiece_buf[SETS][NVP];
    uint16_t kn_buf[SETS], vn_buf[SETS];
    auto issue_keys = [&](auto bsel, auto full_tag, uint32_t t0) __attribute__((always_inline)) {
        constexpr int B = decltype(bsel)::value;
        constexpr bool FULL = decltype(full_tag)::value;     // the run has all its tokens: no address is clamped
        auto &kraw_next = kraw_buf[B];
        const uint32_t n_tok = FULL ? (uint32_t)RUN : min((uint32_t)RUN, t_end - t0);
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const uint32_t tl = 32u * u + 16u * b + n16;
                const uint8_t *src = a.k_idx + (slot0 + t0 + ((FULL || tl < n_tok) ? tl : 0u)) * (4 * KB) + q4 * KB;
                if constexpr (KB % 16 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 16; ++p) {
                        const tq_u4 v = tq_gload16(src + 16 * p);
#pragma unroll
                        for (int i = 0; i < 4; ++i) kraw_next[u][b][4 * p + i] = v[i];
                    }
                } else if constexpr (KB % 8 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 8; ++p) {
                        const tq_u2 v = tq_gload8(src + 8 * p);
                        kraw_next[u][b][2 * p] = v[0]; kraw_next[u][b][2 * p + 1] = v[1];
                    }
                } else if constexpr (KB % 4 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 4; ++p)
                        kraw_next[u][b][p] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)src + 4 * p);
                } else {
                    static_assert(KB % 2 == 0, "key bytes of a lane");
                    uint32_t h[KB / 2];
#pragma unroll
                    for (int p = 0; p < KB / 2; ++p) h[p] = tq_gload2(reinterpret_cast<const uint16_t *>(src) + p);
#pragma unroll
                    for (int p = 0; p < NWK; ++p) kraw_next[u][b][p] = h[2 * p] | (2 * p + 1 < KB / 2 ? h[2 * p + 1 < KB / 2 ? 2 * p + 1 : 0] << 16 : 0u);
                }
            }
    };
    auto issue_values = [&](auto bsel, auto full_tag, uint32_t t0) __attribute__((always_inline)) {
        constexpr int B = decltype(bsel)::value;
        constexpr bool FULL = decltype(full_tag)::value;
        auto &vpiece_next = vpiece_buf[B];
        const uint32_t n_tok = FULL ? (uint32_t)RUN : min((uint32_t)RUN, t_end - t0);
        const uint8_t *vsrc = a.v_idx + (slot0 + t0) * GBV;
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
            const uint32_t piece = p * 64u + lane;
            const bool ok = piece < VPIECES && (FULL || piece * VPB < n_tok * GBV);
            if constexpr (VPB == 16) vpiece_next[p] = tq_gload16(vsrc + (ok ? piece : 0u) * 16u);
            else { const tq_u2 v = tq_gload8(vsrc + (ok ? piece : 0u) * 8u); vpiece_next[p][0] = v[0]; vpiece_next[p][1] = v[1]; }
        }
        kn_buf[B] = lane < n_tok ? tq_gload2(a.k_norms + slot0 + t0 + lane) : (uint16_t)0;
        vn_buf[B] = lane < n_tok ? tq_gload2(a.v_norms + slot0 + t0 + lane) : (uint16_t)0;   // tokens past the end weigh nothing
    };
    const uint32_t t_first = t_begin + RUN * wave;
    if (t_first < t_end) {
        issue_keys(std::integral_constant<int, 0>{}, std::false_type{}, t_first);
        issue_values(std::integral_constant<int, 0>{}, std::false_type{}, t_first);
    }

    if (tid < (uint32_t)DW) lds_trips[tid] = 0u;
    stage_lut<IPBK>(lds_lut_k, a.table_k + hk_hd->off_lut, tid);
    stage_lut<IPBV>(lds_lut_v, a.table_v + hv_hd->off_lut, tid);

    // ---- rotated queries: q_rot[g][j] = scale * sum_i Pi[j][i] q[g][i], wave w the coordinates 32 w .. 32 w + 31
    float *qrot = reinterpret_cast<float *>(&lds_area[0][0]);
    if (wave < (uint32_t)TILES) {
        const uint32_t n = lane & 31u, hk = lane >> 5;
        const uint8_t *qsrc = a.queries + (((size_t)row * G + (n < G ? n : 0u)) * D + 8u * hk) * 2u;
        const uint8_t *asrc = a.table_k + (a.bf16 ? hk_hd->off_a_bf16 : hk_hd->off_a_f16) + ((size_t)wave * STEPS * 64u + lane) * 16u;
        tq_f16v acc = tq_zero16();
        auto rotate = [&](auto bf_tag) __attribute__((always_inline)) {
            constexpr bool BF = decltype(bf_tag)::value;
            constexpr int TERMS = BF ? 3 : 2, CH = 4;        // steps whose operands are in flight together
#pragma unroll 1
            for (int s0 = 0; s0 < STEPS; s0 += 2 * CH) {
                tq_u4 q[2 * CH], p[TERMS][2 * CH];
#pragma unroll
                for (int s = 0; s < 2 * CH; ++s) {
                    if (s0 + s < STEPS) {
                        q[s] = tq_gload16(qsrc + (s0 + s) * 32);
#pragma unroll
                        for (int t = 0; t < TERMS; ++t) p[t][s] = tq_gload16(asrc + (size_t)t * TQ_OPERAND_BYTES_FOR(D) + (size_t)(s0 + s) * 1024u);
                    }
                }
#pragma unroll
                for (int s = 0; s < 2 * CH; ++s) {
                    if (s0 + s < STEPS) {
#pragma unroll
                        for (int t = 0; t < TERMS; ++t) acc = BF ? mfma_bf16(p[t][s], q[s], acc) : mfma_f16(p[t][s], q[s], acc);
                    }
                }
            }
        };
        if (a.bf16) rotate(std::true_type{}); else rotate(std::false_type{});
        const float f = a.bf16 ? a.scale : a.scale * (1.0f / (float)(1 << TQ_F16_PI_SHIFT));
        if (n < (uint32_t)MAX_GROUP) {
#pragma unroll
            for (int r = 0; r < 16; r += 4)
                *reinterpret_cast<float4 *>(qrot + n * QROW + 32u * wave + 16u * hk + r) = make_float4(acc[r] * f, acc[r + 1] * f, acc[r + 2] * f, acc[r + 3] * f);
        }
    }

    // ---- the window: tile w of 32 tokens goes to the block of split w % splits, there to the waves from the last one down
    const uint32_t win_tiles = (a.n_win + WIN_TILE - 1u) / WIN_TILE;
    auto window_tile = [&](auto bf_tag, uint32_t wt) __attribute__((always_inline)) {
        constexpr bool BF = decltype(bf_tag)::value;
        auto mm = [](tq_u4 x, tq_u4 y, tq_f4v c) { return BF ? mfma16_bf16(x, y, c) : mfma16_f16(x, y, c); };
        const uint32_t t0 = wt * WIN_TILE, left = min((uint32_t)WIN_TILE, a.n_win - t0);
        const uint8_t *kw = a.k_win + ((size_t)row * a.win_stride + (size_t)t0 * D) * 2u;
        const uint8_t *vw = a.v_win + ((size_t)row * a.win_stride + (size_t)t0 * D) * 2u;
        const uint8_t *qs = a.queries + (((size_t)row * G + (live ? n16 : 0u)) * D + 8u * q4) * 2u;
        tq_f4v sc[2] = {tq_f4v{0.f, 0.f, 0.f, 0.f}, tq_f4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < SK; ++s) {
            const tq_u4 q = tq_gload16(qs + 64 * s);
#pragma unroll
            for (int b = 0; b < 2; ++b)      // past the end the last token is read again and not used
                sc[b] = mm(tq_gload16(kw + (size_t)min(16u * b + n16, left - 1u) * (2 * D) + 64 * s + 16u * q4), q, sc[b]);
        }
        float t[8], m = -3.0e38f, l = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            t[j] = sc[j / 4][j % 4] * a.scale;       // token 16 (j / 4) + 4 q4 + j % 4 of the tile, head n16
            if (16u * (j / 4) + 4u * q4 + (j % 4) >= left) t[j] = -3.0e38f;
            m = fmaxf(m, t[j]);
        }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = 16u * (j / 4) + 4u * q4 + (j % 4) < left ? __expf(t[j] - m) : 0.f;
            l += p[j];
        }
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        tq_u4 pa[3];
        split_f32x8(p, pa[0], pa[1], pa[2]);
        TQ_GLOBAL float *rec = (TQ_GLOBAL float *)a.win_part + ((size_t)row * win_tiles + wt) * G * PART;
        if (q4 == 0u && live) { put_record(splits > 1u, rec + n16 * PART, m); put_record(splits > 1u, rec + n16 * PART + 1u, l); }
        // columns in chunks of 8 (or 4, 2): the same element of token pairs side by side, one operand per coordinate
        auto columns = [&](auto n_tag, int c0) __attribute__((always_inline)) {
            constexpr int N = decltype(n_tag)::value;
            uint32_t v[8][N / 2];
            const uint32_t first = value_coord<D>(n16, c0);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const uint8_t *src = vw + (size_t)min(16u * (j / 4) + 4u * q4 + (j % 4), left - 1u) * (2 * D) + 2u * first;
                if constexpr (N == 8) { const tq_u4 x = tq_gload16(src); v[j][0] = x[0]; v[j][1] = x[1]; v[j][2] = x[2]; v[j][3] = x[3]; }
                else if constexpr (N == 4) { const tq_u2 x = tq_gload8(src); v[j][0] = x[0]; v[j][1] = x[1]; }
                else v[j][0] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)src);
            }
            float odd = 0.f;         // NaN once a sum is not finite
            auto column = [&](uint32_t c, tq_u4 bt, tq_f4v acc) __attribute__((always_inline)) {
                tq_u4 hi = bt, lo;
                if constexpr (!BF) split_f16x8(bt, hi, lo);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    acc = mfma16_bf16(pa[k], hi, acc);
                    if constexpr (!BF) acc = mfma16_bf16(pa[k], lo, acc);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    odd = fmaf(acc[r], 0.f, odd);
                    if (4u * q4 + r < G) put_record(splits > 1u, rec + (4u * q4 + r) * PART + 2u + first + c, acc[r]);
                }
            };
#pragma unroll
            for (int c = 0; c < N; ++c) {
                tq_u4 bt;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    bt[d] = __builtin_amdgcn_perm(v[2 * d + 1][c / 2], v[2 * d][c / 2], (c & 1) ? 0x07060302u : 0x05040100u);
                column((uint32_t)c, bt, tq_f4v{0.f, 0.f, 0.f, 0.f});
            }
            if (__any(odd != odd)) {
                // An infinite (or NaN) value met a lower term of its probability that is zero, or the zero weight of a token read
                // again.  Once more: such values as bf16 against the leading terms, tokens past the end left out.
#pragma unroll 1
                for (uint32_t c = 0; c < (uint32_t)N; ++c) {
                    tq_u4 bt, wild;
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        uint32_t pair = 0u;
#pragma unroll
                        for (int k = 0; k < 2; ++k) {
                            const uint32_t t = 16u * (d / 2) + 4u * q4 + 2u * (d % 2) + k;
                            if (t < left) pair |= (uint32_t)tq_gload2(reinterpret_cast<const uint16_t *>(vw + (size_t)t * (2 * D)) + first + c) << (16 * k);
                        }
                        constexpr uint32_t EXPO = BF ? 0x7f807f80u : 0x7c007c00u, ONE = BF ? 0x00800080u : 0x04000400u;
                        const uint32_t mask = ((((pair & EXPO) + ONE) >> 15) & 0x00010001u) * 0xffffu;     // exponent all ones
                        wild[d] = pair & mask;
                        if constexpr (!BF)
                            wild[d] = (wild[d] & 0x80008000u) | (mask & 0x7f807f80u) | ((((wild[d] & 0x03ff03ffu) + 0x03ff03ffu) >> 4) & 0x00400040u);
                        bt[d] = pair & ~mask;
                    }
                    column(c, bt, mfma16_bf16(pa[0], wild, tq_f4v{0.f, 0.f, 0.f, 0.f}));
                }
            }
        };
        if constexpr (D == 64) columns(std::integral_constant<int, 4>{}, 0);
        else if constexpr (D == 96) { columns(std::integral_constant<int, 4>{}, 0); columns(std::integral_constant<int, 2>{}, 4); }
        else {
#pragma unroll 1
            for (int c0 = 0; c0 < NC; c0 += 8) columns(std::integral_constant<int, 8>{}, c0);
        }
    };
    for (uint32_t k = DW - 1u - wave; split + k * splits < win_tiles; k += DW) {
        if (a.bf16) window_tile(std::true_type{}, split + k * splits);
        else window_tile(std::false_type{}, split + k * splits);
    }
    __syncthreads();

    // ---- B operand of the score product: fp16 of q * 2^(10 - e), e = binary exponent of the head's largest magnitude.  At 256 with
    // 8-bit codes on either side registers run out (28 spilled with 8-bit keys and values): the low term, the same in every wave, lies
    // in LDS and serves both blocks of a step (128 rows x 8000 tokens, K8/V8: 211 -> 156 us).
    tq_u4 qb[QREG][SK];
    float c1;                // score in base-2 units = t * c1, t = accumulator * key norm
    float rowscale;          // natural score = t * rowscale
    {
        const float *q = qrot + n16 * QROW + (D / 4) * q4;
        float x[D / 4];
#pragma unroll
        for (int i = 0; i < D / 4; i += 4) {
            const float4 f = *reinterpret_cast<const float4 *>(q + i);
            x[i] = f.x; x[i + 1] = f.y; x[i + 2] = f.z; x[i + 3] = f.w;
        }
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < D / 4; ++i) big = fmaxf(big, fabsf(x[i]));
        big = fmaxf(big, __shfl_xor(big, 16));
        big = fmaxf(big, __shfl_xor(big, 32));
        int e = 0;
        if (big > 0.f && big < __builtin_inff()) (void)frexpf(big, &e);
        e = e < -100 ? -100 : e;
        const float up = ldexpf(1.f, TQ_F16_PI_SHIFT - e);
        rowscale = live ? ldexpf(1.f, e - TQ_F16_PI_SHIFT) : 0.f;
        c1 = rowscale * 1.44269504088896341f;
#pragma unroll
        for (int s = 0; s < SK; ++s) {
            tq_half8 term[QT];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float y = live ? x[8 * s + i] * up : 0.f;
#pragma unroll
                for (int k = 0; k < QT; ++k) {
                    term[k][i] = (_Float16)y;
                    y -= (float)term[k][i];
                }
            }
#pragma unroll
            for (int k = 0; k < QREG; ++k) qb[k][s] = __builtin_bit_cast(tq_u4, term[k]);
#pragma unroll
            for (int k = QREG; k < QT; ++k)         // the same in every wave
                if (wave == 0u) lds_q[(k - QREG) * SK + s][lane] = __builtin_bit_cast(tq_u4, term[k]);
        }
    }
    __syncthreads();         // (the queries' LDS is the waves' staging area from here on)

    const uint8_t *lut_k = lds_lut_k + RepLut<IPBK>::lane_offset(lane);
    const uint8_t *lut_v = lds_lut_v + RepLut<IPBV>::lane_offset(lane);
    tq_f4v acc[NC];          // weighted value sums: register r = query head 4 q4 + r, column c = coordinate value_coord(n16, c)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = tq_f4v{0.f, 0.f, 0.f, 0.f};
    // Softmax reference of this lane's head, in units of t (the four lanes of a head agree): it moves only when a score
    // exceeds it by more than SLACK_LOG2 binary orders, so the common tile needs no exchange between lanes.
    float m_ref = -1e30f;
    float l_run = 0.f;       // running sum of p * 2^P_SHIFT over this lane's tokens
    const float slack = live ? (float)SLACK_LOG2 / c1 : 3.0e38f;
    int ev_ref = -100;       // largest binary exponent of a value norm this wave has seen; the sums are in units of 2^ev_ref

    // one run of staged tokens; FULL: all of them exist.  The score products of all its tiles come first, so that a later
    // tile's matrix work runs under an earlier one's softmax.
    auto run = [&](auto bsel, auto full_tag, uint32_t n_tok, uint32_t t_next) __attribute__((always_inline)) {
        constexpr int B = decltype(bsel)::value;
        constexpr bool FULL = decltype(full_tag)::value;
        const auto &kraw = kraw_buf[B];
        tq_f4v sc[SUB][2];   // register r of block b = token 32 u + 16 b + 4 q4 + r
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            sc[u][0] = sc[u][1] = tq_f4v{0.f, 0.f, 0.f, 0.f};
            if (!FULL && 32u * u >= n_tok) continue;       // uniform
            auto step = [&](int b, int s, const tq_u4 (&q)[QT]) __attribute__((always_inline)) {
                const tq_u4 kd = decode_rep<IPBK, NWK>(kraw[u][b], s, lut_k);
#pragma unroll
                for (int k = 0; k < QT; ++k) sc[u][b] = mfma16_f16(kd, q[k], sc[u][b]);
            };
            auto terms = [&](int s, tq_u4 (&q)[QT]) __attribute__((always_inline)) {
#pragma unroll
                for (int k = 0; k < QT; ++k) q[k] = k < QREG ? qb[k < QREG ? k : 0][s] : lds_q[(k - QREG) * SK + s][lane];
            };
            tq_u4 q[QT];
            if constexpr (QREG == QT) {
#pragma unroll
                for (int b = 0; b < 2; ++b)
#pragma unroll
                    for (int s = 0; s < SK; ++s) { terms(s, q); step(b, s, q); }
            } else {         // a term from LDS serves both blocks
#pragma unroll
                for (int s = 0; s < SK; ++s) {
                    terms(s, q);
                    step(0, s, q);
                    step(1, s, q);
                    if (s % 2 == 1) __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if constexpr (SETS == 1 && FULL) {
            if (t_next + RUN <= t_end) issue_keys(bsel, std::true_type{}, t_next);
            else if (t_next < t_end) issue_keys(bsel, std::false_type{}, t_next);
        }
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            if (!FULL && 32u * u >= n_tok) break;  // uniform
            float t[8];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const float4 k4 = *reinterpret_cast<const float4 *>(&lds_kn[wave][32u * u + 16u * b + 4u * q4]);
                t[4 * b + 0] = sc[u][b][0] * k4.x; t[4 * b + 1] = sc[u][b][1] * k4.y;
                t[4 * b + 2] = sc[u][b][2] * k4.z; t[4 * b + 3] = sc[u][b][3] * k4.w;
            }
            if constexpr (!FULL) {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (32u * u + 16u * (j / 4) + 4u * q4 + (j % 4) >= n_tok) t[j] = -1e30f;
            }
            const float tmax = fmaxf(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3])), fmaxf(fmaxf(t[4], t[5]), fmaxf(t[6], t[7])));
            if (__any(tmax > m_ref + slack)) {     // (rare after the first tiles) move the head's reference, rescale its sums
                float tm = fmaxf(tmax, __shfl_xor(tmax, 16));
                tm = fmaxf(tm, __shfl_xor(tm, 32));
                const float m_new = fmaxf(m_ref, tm);
                const float corr = __builtin_amdgcn_exp2f((m_ref - m_new) * c1);
                l_run *= corr;
                m_ref = m_new;
                if (q4 == 0u) lds_corr[wave][n16] = corr;
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
                const float4 c4 = *reinterpret_cast<const float4 *>(&lds_corr[wave][4u * q4]);
                asm volatile("" ::: "memory");
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    acc[c][0] *= c4.x; acc[c][1] *= c4.y; acc[c][2] *= c4.z; acc[c][3] *= c4.w;
                }
            }
            const float bias = P_SHIFT - m_ref * c1;
            float ps[8];
            float lsum = 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                ps[j] = __builtin_amdgcn_exp2f(fmaf(t[j], c1, bias));     // p * 2^P_SHIFT, p <= 2^SLACK_LOG2
                if constexpr (!FULL) {   // a zero query makes every exponent 0: masked tokens need an explicit zero
                    if (32u * u + 16u * (j / 4) + 4u * q4 + (j % 4) >= n_tok) ps[j] = 0.f;
                }
                lsum += ps[j];
            }
            l_run += lsum;
            // ---- weights p_j |v_j| / 2^ev_ref: slice j of lane (., q4) = token 32 u + 4 q4 + j (j < 4), 32 u + 16 + 4 q4 + j - 4
            const uint32_t tok_a = 32u * u + 4u * q4, tok_b = tok_a + 16u;
            tq_u4 pa[PT];
            if constexpr (PT == 1) {
                const tq_u2 vn_a = *reinterpret_cast<const tq_u2 *>(&lds_vn[wave][tok_a]);
                const tq_u2 vn_b = *reinterpret_cast<const tq_u2 *>(&lds_vn[wave][tok_b]);
                const tq_u4 nrm = {vn_a[0], vn_a[1], vn_b[0], vn_b[1]};
                tq_half8 h;
#pragma unroll
                for (int j = 0; j < 8; ++j) h[j] = (_Float16)ps[j];
                h = h * __builtin_bit_cast(tq_half8, nrm);
                pa[0] = __builtin_bit_cast(tq_u4, h);
            } else {
                const float4 va = *reinterpret_cast<const float4 *>(&lds_vn[wave][tok_a]), vb = *reinterpret_cast<const float4 *>(&lds_vn[wave][tok_b]);
                float x[8] = {ps[0] * va.x, ps[1] * va.y, ps[2] * va.z, ps[3] * va.w, ps[4] * vb.x, ps[5] * vb.y, ps[6] * vb.z, ps[7] * vb.w};
#pragma unroll
                for (int k = 0; k < PT; ++k)
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        const auto two = __builtin_amdgcn_cvt_pkrtz(x[2 * d], x[2 * d + 1]);
                        pa[k][d] = __builtin_bit_cast(uint32_t, two);
                        x[2 * d] -= (float)two[0];
                        x[2 * d + 1] -= (float)two[1];
                    }
            }
            auto columns = [&](auto n_tag, int c0) __attribute__((always_inline)) {
                constexpr int N = decltype(n_tag)::value;
                uint32_t dec[8][N / 2];      // per token: N coordinates of the lane as fp16
                const uint32_t first = value_coord<D>(n16, c0);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    decode_values<IPBV, N>(vcodes + ((j < 4 ? tok_a : tok_b) + (uint32_t)(j % 4)) * GBV, first, lut_v, dec[j]);
#pragma unroll
                for (int c = 0; c < N; ++c) {
                    tq_u4 bt;
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        bt[d] = __builtin_amdgcn_perm(dec[2 * d + 1][c / 2], dec[2 * d][c / 2], (c & 1) ? 0x07060302u : 0x05040100u);
#pragma unroll
                    for (int k = 0; k < PT; ++k) acc[c0 + c] = mfma16_f16(pa[k], bt, acc[c0 + c]);
                }
            };
            if constexpr (D == 64) columns(std::integral_constant<int, 4>{}, 0);
            else if constexpr (D == 96) { columns(std::integral_constant<int, 4>{}, 0); columns(std::integral_constant<int, 2>{}, 4); }
            else if constexpr (D == 128) columns(std::integral_constant<int, 8>{}, 0);
            else { columns(std::integral_constant<int, 8>{}, 0); __builtin_amdgcn_sched_barrier(0); columns(std::integral_constant<int, 8>{}, 8); }
        }
    };

    // one trip: stage the run held in register set B, start the loads of the next run into the other set, compute
    // The two waves of a SIMD (w and w + 4) are kept level: the one that is ahead yields.  Left alone the older of the two is
    // served first, and the other one ends its runs without anybody to cover its waits: of a row of 16384 tokens the first
    // waves had done their 32 runs after 69 us and waited 22 us for the others; now all take 84 us and wait one
    // (512 rows, the launch, median over eight layers in turn: 208 -> 200-204 us).  Which wave takes which run stays fixed, so the sums do too.
    uint32_t trips = 0u;
    auto keep_level = [&]() __attribute__((always_inline)) {
        ++trips;
        volatile uint32_t *count = lds_trips;
        if (lane == 0u) count[wave] = trips;
        if (trips > tq_uniform32(count[wave ^ 4u])) __builtin_amdgcn_s_setprio(0); else __builtin_amdgcn_s_setprio(1);
    };
    auto trip = [&](auto bsel, auto full_tag, uint32_t t0) __attribute__((always_inline)) {
        constexpr int B = decltype(bsel)::value;
        keep_level();
        constexpr bool FULL = decltype(full_tag)::value;
        const uint32_t n_tok = FULL ? (uint32_t)RUN : t_end - t0;
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
            const uint32_t piece = p * 64u + lane;
            if (VPIECES % 64 == 0 || piece < VPIECES) {
                if constexpr (VPB == 16) *reinterpret_cast<tq_u4 *>(vcodes + piece * 16u) = vpiece_buf[B][p];
                else *reinterpret_cast<tq_u2 *>(vcodes + piece * 8u) = tq_u2{vpiece_buf[B][p][0], vpiece_buf[B][p][1]};
            }
        }
        {
            const _Float16 kh = __builtin_bit_cast(_Float16, kn_buf[B]);
            if (RUN == 64 || lane < (uint32_t)RUN) lds_kn[wave][lane] = (float)kh;     // one token per lane
            // does a value norm of this run exceed the reference exponent?  (a vote; a handful of times per wave)
            uint32_t e = ((uint32_t)vn_buf[B] >> 10) & 31u;
            if (__any((int)max(e, 1u) - 15 > ev_ref)) {
                // largest exponent field of the run: row-wise running maximum, then the four row ends
                e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x111, 0xf, 0xf, true));
                e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x112, 0xf, 0xf, true));
                e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x114, 0xf, 0xf, true));
                e = max(e, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)e, 0x118, 0xf, 0xf, true));
                const uint32_t emax = max(max((uint32_t)__builtin_amdgcn_readlane((int)e, 15), (uint32_t)__builtin_amdgcn_readlane((int)e, 31)),
                                          max((uint32_t)__builtin_amdgcn_readlane((int)e, 47), (uint32_t)__builtin_amdgcn_readlane((int)e, 63)));
                const int ev = (int)max(emax, 1u) - 15;
                const float f = ldexpf(1.f, ev_ref - ev);
#pragma unroll
                for (int c = 0; c < NC; ++c) acc[c] *= f;
                ev_ref = ev;
            }
            const _Float16 vh = __builtin_bit_cast(_Float16, vn_buf[B]);
            const float vs = ldexpf((float)vh, -ev_ref);
            if (RUN == 64 || lane < (uint32_t)RUN) {
                if constexpr (PT == 1) lds_vn[wave][lane] = __builtin_bit_cast(uint16_t, (_Float16)vs);
                else lds_vn[wave][lane] = vs;
            }
        }
        const uint32_t t_next = t0 + RUN * DW;
        constexpr auto nsel = std::integral_constant<int, SETS == 2 ? 1 - B : 0>{};
        if constexpr (FULL) {
            if (t_next + RUN <= t_end) {
                if constexpr (SETS == 2) issue_keys(nsel, std::true_type{}, t_next);
                issue_values(nsel, std::true_type{}, t_next);
            } else if (t_next < t_end) {
                if constexpr (SETS == 2) issue_keys(nsel, std::false_type{}, t_next);
                issue_values(nsel, std::false_type{}, t_next);
            }
        }
        asm volatile("" ::: "memory");    // staged with one access width, read back with others (LDS serves a wave in order)
        __builtin_amdgcn_wave_barrier();
        run(bsel, full_tag, n_tok, t_next);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        return t_next;
    };
    {
        // whole runs in the loop, the partial one (a wave has one at most) behind it: with both kinds in one loop body the
        // accumulators are copied where they meet and registers spill
        uint32_t t0 = t_first;
        while (t0 + RUN <= t_end) {
            t0 = trip(std::integral_constant<int, 0>{}, std::true_type{}, t0);
            if constexpr (SETS == 2) {
                if (t0 + RUN > t_end) {       // what has been loaded last moves to the set the partial run is taken from
#pragma unroll
                    for (int u = 0; u < SUB; ++u)
#pragma unroll
                        for (int b = 0; b < 2; ++b)
#pragma unroll
                            for (int i = 0; i < NWK; ++i) kraw_buf[0][u][b][i] = kraw_buf[SETS - 1][u][b][i];
#pragma unroll
                    for (int p = 0; p < NVP; ++p) vpiece_buf[0][p] = vpiece_buf[SETS - 1][p];
                    kn_buf[0] = kn_buf[SETS - 1];
                    vn_buf[0] = vn_buf[SETS - 1];
                    break;
                }
                t0 = trip(std::integral_constant<int, SETS - 1>{}, std::true_type{}, t0);
            }
        }
        if (t0 < t_end) trip(std::integral_constant<int, 0>{}, std::false_type{}, t0);
        if (lane == 0u) *(volatile uint32_t *)&lds_trips[wave] = 0xffffffffu;
        __builtin_amdgcn_s_setprio(0);
    }
    asm volatile("" ::: "memory");

    // ---- the waves' sums of HR heads at a time meet in LDS: record [head][largest natural score, sum, D sums] of the split
    float *dst = a.partial + ((size_t)row * splits + split) * G * PART;
    float l_all = l_run + __shfl_xor(l_run, 16);
    l_all = (l_all + __shfl_xor(l_all, 32)) * (1.0f / (float)(1 << P_SHIFT));
    const float out_scale = ldexpf(1.f, ev_ref - P_SHIFT);
    for (uint32_t h0 = 0; h0 < G; h0 += HR) {
        float *res = reinterpret_cast<float *>(lds_area[wave]);
        if (h0) __syncthreads();
        if (q4 == 0u && n16 >= h0 && n16 < h0 + HR) {
            res[(n16 - h0) * PART] = m_ref * rowscale;
            res[(n16 - h0) * PART + 1u] = l_all;
        }
        if (4u * q4 >= h0 && 4u * q4 < h0 + HR) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    res[(4u * q4 + r - h0) * PART + 2u + value_coord<D>(n16, c)] = acc[c][r] * out_scale;
        }
        __syncthreads();
        const uint32_t total = min((uint32_t)HR, G - h0) * PART;
        for (uint32_t i = tid; i < total; i += DTHREADS) {
            const uint32_t g = i / PART, j = i % PART;
            float mw[DW], mall = -3.0e38f;
#pragma unroll
            for (int w = 0; w < DW; ++w) {
                mw[w] = reinterpret_cast<const float *>(lds_area[w])[g * PART];
                mall = fmaxf(mall, mw[w]);
            }
            float v = mall;
            if (j != 0u) {
                v = 0.f;
#pragma unroll
                for (int w = 0; w < DW; ++w) v += __expf(mw[w] - mall) * reinterpret_cast<const float *>(lds_area[w])[g * PART + j];
            }
            put_record(splits > 1u, (TQ_GLOBAL float *)dst + h0 * PART + i, v);
        }
    }

    // ---- the last block of the row finishes it
    // (the records were stored at device scope: once every wave has waited for its own stores, which the barrier by itself does not
    // do, thread 0 may count the block as done, see put_record)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (splits > 1u) {
        if (tid == 0u) {
            const bool last = __hip_atomic_fetch_add(a.arrived + row, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == splits - 1u;
            if (last) __hip_atomic_store(a.arrived + row, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            lds_last = last ? 1u : 0u;
        }
        __syncthreads();
        if (!lds_last) return;
    }
    const TQ_GLOBAL float *part = (const TQ_GLOBAL float *)a.partial + (size_t)row * splits * G * PART;
    const TQ_GLOBAL float *wpart = (const TQ_GLOBAL float *)a.win_part + (size_t)row * win_tiles * G * PART;
    // rows of Pi_v for the rotation back: thread (four columns, part) takes ROTK of them
    const uint32_t rc = (tid % (D / 4)) * 4u, rp = tid / (D / 4);
    constexpr int RH = ROTK > 8 ? 8 : ROTK;           // held at a time
    tq_u4 pv[RH];
    auto load_pv = [&](int k0) {
        if (rp < (uint32_t)ROTP) {
#pragma unroll
            for (int k = 0; k < RH; ++k) pv[k] = tq_gload16(reinterpret_cast<const uint8_t *>(a.pi_v + (size_t)(rp * ROTK + k0 + k) * D + rc));
        }
    };
    if constexpr (ROTK == RH) load_pv(0);
    float *ysum = reinterpret_cast<float *>(&lds_area[0][0]);     // [head][D]: sums in the rotated space
    float *wsum = ysum + MAX_GROUP * D;                           // [head][D]: the window's, plain
    auto merge = [&](auto across_tag) __attribute__((always_inline)) {
        constexpr bool ACROSS = decltype(across_tag)::value;
        // weights of the records: exp(reference - largest reference of the head)
        float *wgt = reinterpret_cast<float *>(lds_lut_k);            // [head][splits + window tiles]
        const uint32_t nrec = splits + win_tiles;
        for (uint32_t g = wave; g < G; g += DW) {
            float m = -3.0e38f;
            for (uint32_t s = lane; s < nrec; s += 64u) {
                const float x = get_record<ACROSS>(s < splits ? part + ((size_t)s * G + g) * PART : wpart + ((size_t)(s - splits) * G + g) * PART);
                m = fmaxf(m, x);
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
            float den = 0.f;
            for (uint32_t s = lane; s < nrec; s += 64u) {
                const TQ_GLOBAL float *r = s < splits ? part + ((size_t)s * G + g) * PART : wpart + ((size_t)(s - splits) * G + g) * PART;
                const float f = __expf(get_record<ACROSS>(r) - m);
                wgt[g * nrec + s] = f;
                den = fmaf(f, get_record<ACROSS>(r + 1), den);
            }
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) den += __shfl_xor(den, d);
            if (lane == 0u) lds_den[g] = den;
        }
        __syncthreads();
        for (uint32_t p = tid; p < G * D; p += DTHREADS) {
            const uint32_t g = p / D, j = p % D;
            const float *f = wgt + g * nrec;
            float y = 0.f, w = 0.f;
#pragma unroll 8
            for (uint32_t s = 0; s < splits; ++s) y = fmaf(f[s], get_record<ACROSS>(part + ((size_t)s * G + g) * PART + 2u + j), y);
#pragma unroll 4
            for (uint32_t s = 0; s < win_tiles; ++s) w = fmaf(f[splits + s], get_record<ACROSS>(wpart + ((size_t)s * G + g) * PART + 2u + j), w);
            ysum[p] = y;
            wsum[p] = w;
        }
        __syncthreads();
    };
    if (splits > 1u) merge(std::true_type{}); else merge(std::false_type{});
    // out = (ysum @ Pi_v + wsum) / den, four heads at a time
    float *parts = reinterpret_cast<float *>(lds_lut_v);          // [part][4][D]
    for (uint32_t g0 = 0; g0 < G; g0 += 4u) {
        float x[4][4];
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[g][c] = 0.f;
#pragma unroll 1
        for (int k0 = 0; k0 < ROTK; k0 += RH) {
            if constexpr (ROTK != RH) load_pv(k0);
            if (rp < (uint32_t)ROTP) {
#pragma unroll
                for (int k = 0; k < RH; ++k)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const float y = ysum[(g0 + g) * D + rp * ROTK + k0 + k];     // (heads past the last one: whatever lies there, not stored)
#pragma unroll
                        for (int c = 0; c < 4; ++c) x[g][c] = fmaf(y, __uint_as_float(pv[k][c]), x[g][c]);
                    }
            }
        }
        if (g0) __syncthreads();
        if (rp < (uint32_t)ROTP) {
#pragma unroll
            for (int g = 0; g < 4; ++g) *reinterpret_cast<float4 *>(parts + (rp * 4u + g) * D + rc) = make_float4(x[g][0], x[g][1], x[g][2], x[g][3]);
        }
        __syncthreads();
        for (uint32_t p = tid; p < min(4u, G - g0) * D; p += DTHREADS) {
            const uint32_t g = p / D, j = p % D;
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < ROTP; ++q) v += parts[((uint32_t)q * 4u + g) * D + j];
            v = (v + wsum[(g0 + g) * D + j]) / lds_den[g0 + g];
            TQ_GLOBAL uint16_t *o = (TQ_GLOBAL uint16_t *)a.out + ((size_t)row * G + g0 + g) * D + j;
            if (a.bf16) { const __bf16 h = (__bf16)v; *o = __builtin_bit_cast(uint16_t, h); }
            else { const _Float16 h = (_Float16)v; *o = __builtin_bit_cast(uint16_t, h); }
        }
    }
}

// ---- append: compress the token that leaves the window, put the new one into its slot ---------------------------------
struct AppendArgs {
    const uint8_t *fresh[2];         // new keys, values: row r at element r * new_stride
    uint8_t *win[2];                 // row r, slot s at element r * win_stride + s * D
    const uint8_t *table[2];
    uint8_t *idx[2];                 // packed store, advanced to the slot of row 0
    uint16_t *norms[2];
    long long new_stride[2], win_stride;
    uint32_t packed_row_stride, rows, evict, put, bf16, compress;
    int ipb[2];
};

// Block (32 rows, tensor) of D / 32 waves, one vector per row: wave w produces the rotated coordinates [32 w, 32 w + 32) of
// the 32 vectors and their codes.  A step has one vector per row, so nothing is shared between blocks or reused: operands, vectors
// and the quantiser's cells come straight from memory (the cells of a lane's 16 coordinates as 16 loads in flight together)
// and the launch lasts as long as that chain of loads.  Products and sums run in the order of the kernels that compress whole
// tensors of this head dimension, so the bytes are theirs.
template <int D, bool BF>
__global__ __launch_bounds__(D / 32 * TQ_WAVE) void tq_decode_append_kernel(AppendArgs a) {
    constexpr int STEPS = D / 16, THREADS = D / 32 * TQ_WAVE;
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = tq_uniform32(tid >> 6), which = blockIdx.y;
    const uint32_t n = lane & 31u, hk = lane >> 5;
    const uint32_t row0 = blockIdx.x * 32u;
    const uint8_t *fresh = a.fresh[which];
    uint8_t *win = a.win[which];
    // the new tokens of the block's rows: 16-byte pieces (another slot than the one read below)
    for (uint32_t i = tid; i < 32u * (D / 8); i += THREADS) {
        const uint32_t r = row0 + i / (D / 8), piece = i % (D / 8);
        if (r < a.rows)
            tq_gstore16(win + ((size_t)r * a.win_stride + (size_t)a.put * D) * 2u + piece * 16u, tq_gload16(fresh + (size_t)r * a.new_stride[which] * 2u + piece * 16u));
    }
    if (!a.compress) return;
    const uint8_t *table = a.table[which];
    const TqTableHeader *hd = reinterpret_cast<const TqTableHeader *>(table);
    const uint32_t r = min(row0 + n, a.rows - 1u);
    const uint8_t *src = win + ((size_t)r * a.win_stride + (size_t)a.evict * D) * 2u + 16u * hk;
    const uint8_t *asrc = table + (BF ? hd->off_a_bf16 : hd->off_a_f16) + ((size_t)wave * STEPS * 64u + lane) * 16u;
    const uint32_t step0 = D == 128 ? 2u * wave : 0u;      // the 128-wide kernel starts the contraction at the wave's own quarter
    tq_u4 x[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) x[s] = tq_gload16(src + 32 * s);
    tq_f16v acc = tq_zero16();
    if constexpr (D == 128) {
        tq_u4 p[2][STEPS], xs[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const uint32_t sg = (s + step0) & 7u;
            p[0][s] = tq_gload16(asrc + (size_t)sg * 1024u);
            p[1][s] = tq_gload16(asrc + TQ_OPERAND_BYTES_FOR(D) + (size_t)sg * 1024u);
            xs[s] = tq_gload16(src + 32u * sg);
        }
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
#pragma unroll
            for (int t = 0; t < 2; ++t) acc = BF ? mfma_bf16(p[t][s], xs[s], acc) : mfma_f16(p[t][s], xs[s], acc);
    } else {
        constexpr int CH = STEPS < 8 ? STEPS : 8;
        for (int s0 = 0; s0 < STEPS; s0 += CH) {
            tq_u4 p[2][CH];
#pragma unroll
            for (int s = 0; s < CH; ++s) {
                if (s0 + s < STEPS) {
                    p[0][s] = tq_gload16(asrc + (size_t)(s0 + s) * 1024u);
                    p[1][s] = tq_gload16(asrc + TQ_OPERAND_BYTES_FOR(D) + (size_t)(s0 + s) * 1024u);
                }
            }
#pragma unroll
            for (int s = 0; s < CH; ++s) {
                if (s0 + s < STEPS) {
                    const tq_u4 xv = STEPS > CH ? tq_gload16(src + 32u * (s0 + s)) : x[s];
#pragma unroll
                    for (int t = 0; t < 2; ++t) acc = BF ? mfma_bf16(p[t][s], xv, acc) : mfma_f16(p[t][s], xv, acc);
                }
            }
        }
    }
    // ---- sum of squares: lane (n, hk) holds pieces 2 s + hk of its vector
    float ss;
    constexpr int DT = BF ? TQ_BF16 : TQ_F16;
    if constexpr (D == 128) {        // per quarter: two pieces as one chain, the halves added; the quarters pairwise
        float share[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            share[q] = sumsq8<DT>(x[2 * q + 1], sumsq8<DT>(x[2 * q], 0.f));
            share[q] += __shfl_xor(share[q], 32);
        }
        ss = (share[0] + share[1]) + (share[2] + share[3]);
    } else {
        float even[STEPS], odd[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const float own = sumsq8<DT>(x[s], 0.f), other = __shfl_xor(own, 32);
            even[s] = hk ? other : own;
            odd[s] = hk ? own : other;
        }
        if constexpr (D == 256) {    // a tree over the pieces
#pragma unroll
            for (int s = 0; s < STEPS; ++s) even[s] += odd[s];
#pragma unroll
            for (int m = 1; m < STEPS; m <<= 1)
#pragma unroll
                for (int s = 0; s < STEPS; s += 2 * m) even[s] += even[s + m];
            ss = even[0];
        } else {                     // in order
            ss = 0.f;
#pragma unroll
            for (int s = 0; s < STEPS; ++s) { ss += even[s]; ss += odd[s]; }
        }
    }
    const float nrm = tq_norm_from_sumsq(ss);
    float inv = __builtin_amdgcn_rcpf(nrm + 1e-8f);
    if (!BF) inv *= 1.0f / (float)(1 << TQ_F16_PI_SHIFT);
    const float inv_cell = inv * hd->grid_scale, grid_bias = hd->grid_bias;
    // ---- code search: lane (n, hk) holds coordinates 32 w + 16 hk + r
    const uint8_t *grid = table + hd->off_grid;
    tq_u2 cell[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) cell[q] = tq_gload8(grid + (__float_as_uint(fmaf(acc[q], inv_cell, grid_bias)) & TQ_GRID_ADDR_MASK));
    uint32_t code[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) code[q] = cell[q][1] + (~__float_as_uint(fmaf(acc[q], inv, -__uint_as_float(cell[q][0]))) >> 31);
    if (row0 + n >= a.rows) return;
    const int ipb = a.ipb[which];
    const size_t slot = (size_t)r * a.packed_row_stride;
    uint8_t *dst = a.idx[which] + slot * (uint32_t)(D / ipb) + (2u * wave + hk) * (uint32_t)(16 / ipb);
    auto pack = [&](auto ipb_tag) __attribute__((always_inline)) {       // most significant code of a byte first
        constexpr int I = decltype(ipb_tag)::value, BITS = 8 / I, NB = 16 / I, NW = NB < 4 ? 1 : NB / 4;
        uint32_t w[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) w[k] = 0u;
        const uint32_t width = hd->bits;       // 3-bit codes sit two to a byte, three bits apart
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int byte = q / I, k = q % I;
            const uint32_t shift = I == 2 ? width * (uint32_t)(I - 1 - k) : (uint32_t)(BITS * (I - 1 - k));
            w[byte / 4] |= code[q] << (8 * (byte % 4) + shift);
        }
        if constexpr (NB == 2) tq_gstore2(reinterpret_cast<uint16_t *>(dst), (uint16_t)w[0]);
        else if constexpr (NB == 4) *reinterpret_cast<TQ_GLOBAL uint32_t *>((TQ_GLOBAL uint8_t *)dst) = w[0];
        else if constexpr (NB == 8) tq_gstore8(dst, tq_u2{w[0], w[1]});
        else tq_gstore16(dst, tq_u4{w[0], w[1], w[2], w[3]});
    };
    if (ipb == 8) pack(std::integral_constant<int, 8>{});
    else if (ipb == 4) pack(std::integral_constant<int, 4>{});
    else if (ipb == 2) pack(std::integral_constant<int, 2>{});
    else pack(std::integral_constant<int, 1>{});
    if (wave == 0u && hk == 0u) {
        const _Float16 hn = (_Float16)nrm;
        tq_gstore2(a.norms[which] + slot, __builtin_bit_cast(uint16_t, hn));
    }
}

// ---- host side --------------------------------------------------------------------------------------------------------
bool decode_supported(int head_dim, int bits_k, int bits_v) {
    if (bits_k < 1 || bits_k > 8 || bits_v < 1 || bits_v > 8) return false;
    if (head_dim == 128) return true;
    return (head_dim == 64 || head_dim == 96 || head_dim == 256) && bits_k > 1 && bits_v > 1;
}

template <int D, int IPBK>
int launch_decode(int ipbv, dim3 grid, hipStream_t s, const DecodeArgs &a) {
    const dim3 block(DTHREADS);
    switch (ipbv) {
        case 8:
            if constexpr (D == 128) { hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, 8>), grid, block, 0, s, a); break; }
            return TQ_ERR_BITS;
        case 4: hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, 4>), grid, block, 0, s, a); break;
        case 2: hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, 2>), grid, block, 0, s, a); break;
        default: hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, 1>), grid, block, 0, s, a); break;
    }
    return (int)hipGetLastError();
}
template <int D>
int launch_decode(int ipbk, int ipbv, dim3 grid, hipStream_t s, const DecodeArgs &a) {
    switch (ipbk) {
        case 8:
            if constexpr (D == 128) return launch_decode<D, 8>(ipbv, grid, s, a);
            return TQ_ERR_BITS;
        case 4: return launch_decode<D, 4>(ipbv, grid, s, a);
        case 2: return launch_decode<D, 2>(ipbv, grid, s, a);
        default: return launch_decode<D, 1>(ipbv, grid, s, a);
    }
}

template <int D>
void launch_append(dim3 grid, hipStream_t s, const AppendArgs &a) {
    const dim3 block(D / 32 * TQ_WAVE);
    if (a.bf16) hipLaunchKernelGGL((tq_decode_append_kernel<D, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((tq_decode_append_kernel<D, false>), grid, block, 0, s, a);
}

// splits of the token range per row
int decode_splits(long long rows, long long tokens) {
    if (rows <= 0 || tokens <= 0) return 1;
    int cus = 0;
    if (tq_device_cus(cus)) cus = 256;
    // One block is resident per compute unit.  A launch takes as many rounds of blocks as rows * splits fill the chip, each as
    // long as a block's tokens (in trips of its eight waves) plus about what 1000 tokens take for tables, query rotation and
    // result, and what 600 more take where the splits of a row have to be merged.
    long long most = (tokens + 64 * DW - 1) / (64 * DW);
    if (most > MAX_SPLITS) most = MAX_SPLITS;
    long long best = 1, best_cost = 0;
    for (long long s = 1; s <= most; ++s) {
        const long long rounds = (rows * s + cus - 1) / cus;
        const long long trips = ((tokens + s - 1) / s + 64 * DW - 1) / (64 * DW);
        const long long cost = rounds * (trips * 64 * DW + 1000 + (s > 1 ? 600 : 0));
        if (s == 1 || cost < best_cost) { best = s; best_cost = cost; }
        if (rounds > 16 && s > 1) break;
    }
    return (int)best;
}

long long scratch_floats(long long rows, int group, int head_dim, int splits, long long n_win) {
    return rows * group * (head_dim + 2) * (splits + (n_win + WIN_TILE - 1) / WIN_TILE);
}

// what both calls ask of the layer's record
int check_layer(const tq_decode_layer *l) {
    if (!l) return TQ_ERR_NULL;
    if (l->dtype != TQ_F16 && l->dtype != TQ_BF16) return TQ_ERR_DTYPE;
    if (l->bits_k < 1 || l->bits_k > 8 || l->bits_v < 1 || l->bits_v > 8) return TQ_ERR_BITS;
    if (!decode_supported(l->head_dim, l->bits_k, l->bits_v)) return TQ_ERR_HEAD_DIM;
    if (l->rows < 0 || l->rows > 65535 || l->win_stride < 0) return TQ_ERR_SIZE;
    if (l->rows && (l->packed_row_stride < 0 || l->packed_row_stride > (long long)0x7fffffff / l->rows)) return TQ_ERR_SIZE;
    if (!l->table_k || !l->table_v || !l->pi_v) return TQ_ERR_NULL;
    if (((uintptr_t)l->table_k & 15u) || ((uintptr_t)l->table_v & 15u) || ((uintptr_t)l->pi_v & 15u) || ((uintptr_t)l->k_win & 15u) ||
        ((uintptr_t)l->v_win & 15u) || (l->win_stride & 7) || ((uintptr_t)l->k_idx & (tq_packed_alignment(l->head_dim, l->bits_k) - 1u)) ||
        ((uintptr_t)l->v_idx & (tq_packed_alignment(l->head_dim, l->bits_v) - 1u)) || ((uintptr_t)l->k_norms & 1u) || ((uintptr_t)l->v_norms & 1u))
        return TQ_ERR_ALIGN;
    return TQ_OK;
}

}  // namespace

extern "C" int tq_decode_supported(int head_dim, int dtype, int bits_k, int bits_v) {
    return (dtype == TQ_F16 || dtype == TQ_BF16) && decode_supported(head_dim, bits_k, bits_v) ? 1 : 0;
}

extern "C" long long tq_decode_scratch_floats(long long rows, int group, int head_dim, long long tokens, long long n_win) {
    if (rows < 0 || rows > 65535 || group < 1 || group > MAX_GROUP || tokens < 0 || n_win < 0 || n_win > MAX_WINDOW) return TQ_ERR_SIZE;
    return scratch_floats(rows, group, head_dim, decode_splits(rows, tokens), n_win);
}

extern "C" int tq_decode_attend(const tq_decode_layer *layer, const void *queries, int group, float scale, long long win_first, long long n_win,
                                long long tokens, float *scratch, long long scratch_size, uint32_t *arrived, void *out, void *stream) {
    const int rc = check_layer(layer);
    if (rc) return rc;
    const int D = layer->head_dim;
    const long long rows = layer->rows;
    if (group < 1 || group > MAX_GROUP || n_win < 0 || n_win > MAX_WINDOW || win_first < 0 || tokens < 0 || (tokens == 0 && n_win == 0)) return TQ_ERR_SIZE;
    if (rows == 0) return TQ_OK;
    if (!queries || !scratch || !arrived || !out) return TQ_ERR_NULL;
    if (tokens && (!layer->k_idx || !layer->k_norms || !layer->v_idx || !layer->v_norms)) return TQ_ERR_NULL;
    if (n_win && (!layer->k_win || !layer->v_win)) return TQ_ERR_NULL;
    if (n_win && layer->win_stride < (win_first + n_win) * D) return TQ_ERR_SIZE;
    if (tokens > (layer->packed_row_stride ? layer->packed_row_stride : (rows == 1 ? tokens : 0))) return TQ_ERR_SIZE;
    if (((uintptr_t)queries & 15u) || ((uintptr_t)scratch & 3u) || ((uintptr_t)arrived & 3u) || ((uintptr_t)out & 1u)) return TQ_ERR_ALIGN;
    const int splits = decode_splits(rows, tokens);
    if (scratch_size < scratch_floats(rows, group, D, splits, n_win)) return TQ_ERR_CAPACITY;
    DecodeArgs a;
    a.queries = static_cast<const uint8_t *>(queries);
    a.k_idx = layer->k_idx; a.v_idx = layer->v_idx; a.k_norms = layer->k_norms; a.v_norms = layer->v_norms;
    a.table_k = static_cast<const uint8_t *>(layer->table_k);
    a.table_v = static_cast<const uint8_t *>(layer->table_v);
    a.pi_v = layer->pi_v;
    a.k_win = static_cast<const uint8_t *>(layer->k_win) + win_first * D * 2;
    a.v_win = static_cast<const uint8_t *>(layer->v_win) + win_first * D * 2;
    a.partial = scratch;
    a.win_part = scratch + (size_t)rows * splits * group * (D + 2);
    a.arrived = arrived;
    a.out = static_cast<uint8_t *>(out);
    a.win_stride = layer->win_stride;
    a.scale = scale;
    a.tokens = (uint32_t)tokens;
    a.packed_row_stride = (uint32_t)layer->packed_row_stride;
    a.group = (uint32_t)group;
    a.chunk = (uint32_t)(((tokens + splits - 1) / splits + 63) / 64 * 64);
    a.n_win = (uint32_t)n_win;
    a.bf16 = layer->dtype == TQ_BF16 ? 1u : 0u;
    const dim3 grid((unsigned)splits, (unsigned)rows, 1);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int ik = 8 / layer->bits_k, iv = 8 / layer->bits_v;
    switch (D) {
        case 64: return launch_decode<64>(ik, iv, grid, s, a);
        case 96: return launch_decode<96>(ik, iv, grid, s, a);
        case 128: return launch_decode<128>(ik, iv, grid, s, a);
        default: return launch_decode<256>(ik, iv, grid, s, a);
    }
}

extern "C" int tq_decode_append(const tq_decode_layer *layer, const void *k_new, const void *v_new, long long k_new_stride, long long v_new_stride,
                                long long evict, long long put, long long packed_slot, void *stream) {
    const int rc = check_layer(layer);
    if (rc) return rc;
    const int D = layer->head_dim;
    const long long rows = layer->rows;
    if (put < 0 || evict < -1 || evict == put || packed_slot < 0) return TQ_ERR_SIZE;
    if (layer->win_stride < (put + 1) * D || layer->win_stride < (evict + 1) * D) return TQ_ERR_SIZE;
    if (rows > 1 && (k_new_stride < D || v_new_stride < D)) return TQ_ERR_SIZE;
    if (rows == 0) return TQ_OK;
    if (!k_new || !v_new || !layer->k_win || !layer->v_win) return TQ_ERR_NULL;
    if (((uintptr_t)k_new & 15u) || ((uintptr_t)v_new & 15u) || (rows > 1 && ((k_new_stride & 7) || (v_new_stride & 7)))) return TQ_ERR_ALIGN;
    AppendArgs a{};
    if (evict >= 0) {
        const long long prs = layer->packed_row_stride ? layer->packed_row_stride : 1;
        if (packed_slot >= prs) return TQ_ERR_SIZE;
        if (!layer->k_idx || !layer->k_norms || !layer->v_idx || !layer->v_norms) return TQ_ERR_NULL;
        a.ipb[0] = 8 / layer->bits_k; a.ipb[1] = 8 / layer->bits_v;
        a.table[0] = static_cast<const uint8_t *>(layer->table_k); a.table[1] = static_cast<const uint8_t *>(layer->table_v);
        a.idx[0] = layer->k_idx + packed_slot * (D / a.ipb[0]); a.idx[1] = layer->v_idx + packed_slot * (D / a.ipb[1]);
        a.norms[0] = layer->k_norms + packed_slot; a.norms[1] = layer->v_norms + packed_slot;
        a.packed_row_stride = (uint32_t)prs;
        a.evict = (uint32_t)evict;
        a.compress = 1u;
    }
    a.fresh[0] = static_cast<const uint8_t *>(k_new); a.fresh[1] = static_cast<const uint8_t *>(v_new);
    a.win[0] = static_cast<uint8_t *>(layer->k_win); a.win[1] = static_cast<uint8_t *>(layer->v_win);
    a.new_stride[0] = k_new_stride; a.new_stride[1] = v_new_stride;
    a.win_stride = layer->win_stride;
    a.rows = (uint32_t)rows;
    a.put = (uint32_t)put;
    a.bf16 = layer->dtype == TQ_BF16 ? 1u : 0u;
    const dim3 grid((unsigned)((rows + 31) / 32), 2, 1);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    switch (D) {
        case 64: launch_append<64>(grid, s, a); break;
        case 96: launch_append<96>(grid, s, a); break;
        case 128: launch_append<128>(grid, s, a); break;
        default: launch_append<256>(grid, s, a); break;
    }
    return (int)hipGetLastError();
}
