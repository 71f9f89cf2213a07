// The kernel behind tq_decode_attend (tq_decode.hip) and what launches it.  One source file per head dimension instantiates it
// (tq_decode_d64.hip ... tq_decode_d256.hip; 128 in two), so that they compile side by side.
#pragma once
#include <type_traits>

#include "tq_decode.h"
#include "tq_lut.h"

namespace {

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
// 8 rows x 32768 tokens took 32.0 us with fences and 30.0 this way when it was made, one of 32 rows x 6000 tokens, 64 wide, 27.3 and 24.7.  A row with one split keeps
// its records in its own block: they stay cached (512 rows x 16384 tokens: 2 % longer otherwise).
// No release and acquire of the language stand behind this order, all accesses are relaxed: it rests on the hardware, where a
// store of device scope counts in vmcnt until every compute unit sees it, and on both sides going through put_record and
// Records.  Plain accesses to a record of a row with several splits would be a race.
__device__ __forceinline__ void put_record(bool across, TQ_GLOBAL float *p, float v) {
    if (across) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
// Two neighbours in one access (the pair need not be one value to the other side, only each half of it).
template <bool ACROSS>
__device__ __forceinline__ void put_record2(TQ_GLOBAL float *p, float a, float b) {
    const tq_u2 v = {__float_as_uint(a), __float_as_uint(b)};
    if constexpr (ACROSS) __hip_atomic_store(reinterpret_cast<TQ_GLOBAL uint64_t *>(p), __builtin_bit_cast(uint64_t, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *reinterpret_cast<TQ_GLOBAL tq_u2 *>(p) = v;
}
// Records of a row, from the first float of the first one, as a buffer: four (or two) neighbours in one access of device scope (the
// cache-policy bits of a load can be given to the buffer form only), and what lies past the last record reads as zero.
struct Records {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ Records(const float *p, uint32_t floats) : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), 0, floats * 4u, 0x00020000)) {}
    template <bool ACROSS> __device__ __forceinline__ tq_u4 load4(uint32_t at) const { return __builtin_amdgcn_raw_buffer_load_b128(rsrc, at * 4u, 0, ACROSS ? 16 : 0); }
    template <bool ACROSS> __device__ __forceinline__ tq_u2 load2(uint32_t at) const { return __builtin_amdgcn_raw_buffer_load_b64(rsrc, at * 4u, 0, ACROSS ? 16 : 0); }
};

// Lanes L apart exchanged between two registers (L = 32: upper half of a with lower half of b; 16: the odd quarters of a with the
// even ones of b) and added: a summed over both where b's half (quarter) does not lie, b where it does.
template <int L>
__device__ __forceinline__ float fold(float a, float b) {
    const auto two = L == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                             : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(two[0]) + __uint_as_float(two[1]);
}

// Tokens a wave takes per trip: 32 where registers are short, and with a byte per code from 96 on (64 fit by now, but take longer: 128 x 8192
// tokens, K6/V4, 4 heads 393 -> 404 us for eight layers, K8/V8 474 -> 489; 96 wide, K8/V8, 7 heads 255 -> 277).
constexpr int decode_run(int d, int ipbk, int ipbv) { return d == 256 || (d > 64 && (ipbk == 1 || ipbv == 1)) ? 32 : 64; }

// Rotated queries of a row, q_rot[g][j] = scale * sum_i Pi[j][i] q[g][i]: a wave's 32 coordinates on the matrix cores, from the operands
// of the key codec's table (Pi as three bf16 terms that add up to its float32 value, or for fp16 queries as two fp16 terms, 22 bits).
// Loads and products apart, so that other loads can be under way between them.  A row has 16 heads at most: two tiles of 16 x 16, which
// take half the time of one of 32 x 32 (the table's operands are for that one: lane (row i, half hk) of step s has inputs 16 s + 8 hk ...;
// here a lane picks the pieces that it needs).
template <int D, bool BF>
struct Rotation {
    static constexpr int STEPS = D / 32, CH = STEPS < 4 ? STEPS : 4, TERMS = BF ? 3 : 2;     // CH: steps whose operands are in flight together
    static_assert(STEPS % CH == 0, "whole chunks");
    tq_u4 q[CH], p[2][TERMS][CH];
    const uint8_t *qsrc, *asrc;
    __device__ __forceinline__ void fetch(int s0) {
#pragma unroll
        for (int s = 0; s < CH; ++s) {
            q[s] = tq_gload16(qsrc + (s0 + s) * 64);
#pragma unroll
            for (int t = 0; t < TERMS; ++t)
#pragma unroll
                for (int b = 0; b < 2; ++b) p[b][t][s] = tq_gload16(asrc + (size_t)t * TQ_OPERAND_BYTES_FOR(D) + (size_t)(s0 + s) * 2048u + 256u * b);
        }
    }
    // queries: the row's, [group][D]
    __device__ __forceinline__ void load(const uint8_t *queries, uint32_t group, const uint8_t *table_k, uint32_t tile, uint32_t lane) {
        const uint32_t n16 = lane & 15u, q4 = lane >> 4;
        qsrc = queries + ((size_t)(n16 < group ? n16 : 0u) * D + 8u * q4) * 2u;
        asrc = table_k + (BF ? TQ_OFF_A_BF16(D) : TQ_OFF_A_F16) + ((size_t)tile * (D / 16 * 64u) + q4 * 32u + n16) * 16u;
        fetch(0);
    }
    // qrot: [MAX_GROUP] rows of `stride` floats
    __device__ __forceinline__ void finish(float *qrot, uint32_t stride, float scale, uint32_t tile, uint32_t lane) {
        const uint32_t n16 = lane & 15u, q4 = lane >> 4;
        tq_f4v acc[2] = {tq_f4v{0.f, 0.f, 0.f, 0.f}, tq_f4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll 1
        for (int s0 = 0;;) {
#pragma unroll
            for (int s = 0; s < CH; ++s)
#pragma unroll
                for (int t = 0; t < TERMS; ++t)
#pragma unroll
                    for (int b = 0; b < 2; ++b) acc[b] = BF ? mfma16_bf16(p[b][t][s], q[s], acc[b]) : mfma16_f16(p[b][t][s], q[s], acc[b]);
            s0 += CH;
            if (s0 >= STEPS) break;
            fetch(s0);
        }
        const float f = BF ? scale : scale * (1.0f / (float)(1 << TQ_F16_PI_SHIFT));
#pragma unroll
        for (int b = 0; b < 2; ++b)       // row i of the table's 32 holds coordinate 16 (i / 4 % 2) + 4 (i / 8) + i % 4
            *reinterpret_cast<float4 *>(qrot + n16 * stride + 32u * tile + 16u * (q4 & 1u) + 8u * b + 4u * (q4 >> 1)) =
                make_float4(acc[b][0] * f, acc[b][1] * f, acc[b][2] * f, acc[b][3] * f);
    }
};

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
__device__ __forceinline__ void decode_values(const uint8_t *codes, uint32_t first, const uint8_t *lut, uint32_t slot, uint32_t (&out)[N / 2]) {
    if constexpr (IPB == 8) {
        static_assert(N == 8, "whole bytes");
        const tq_u4 v = lut_entry<0, tq_u4>(lut, codes[first / 8u], slot);
        out[0] = v[0]; out[1] = v[1]; out[2] = v[2]; out[3] = v[3];
    } else if constexpr (IPB == 4) {
        if constexpr (N == 8) {
            const uint32_t two = *reinterpret_cast<const uint16_t *>(codes + first / 4u);
            const tq_u2 a = lut_entry<0, tq_u2>(lut, two, slot), b = lut_entry<1, tq_u2>(lut, two, slot);
            out[0] = a[0]; out[1] = a[1]; out[2] = b[0]; out[3] = b[1];
        } else if constexpr (N == 4) {
            const tq_u2 a = lut_entry<0, tq_u2>(lut, codes[first / 4u], slot);
            out[0] = a[0]; out[1] = a[1];
        } else {        // half a byte
            out[0] = lut_entry<0, uint32_t>(lut, codes[first / 4u], slot + 2u * (first & 3u));
        }
    } else if constexpr (IPB == 2) {
        uint32_t raw;
        if constexpr (N == 8) raw = *reinterpret_cast<const uint32_t *>(codes + first / 2u);
        else if constexpr (N == 4) raw = *reinterpret_cast<const uint16_t *>(codes + first / 2u);
        else raw = codes[first / 2u];
        out[0] = lut_entry<0, uint32_t>(lut, raw, slot);
        if constexpr (N >= 4) out[1] = lut_entry<1, uint32_t>(lut, raw, slot);
        if constexpr (N == 8) {
            out[2] = lut_entry<2, uint32_t>(lut, raw, slot);
            out[3] = lut_entry<3, uint32_t>(lut, raw, slot);
        }
    } else {
        uint32_t raw[2] = {0u, 0u};
        if constexpr (N == 8) { const tq_u2 v = *reinterpret_cast<const tq_u2 *>(codes + first); raw[0] = v[0]; raw[1] = v[1]; }
        else if constexpr (N == 4) raw[0] = *reinterpret_cast<const uint32_t *>(codes + first);
        else raw[0] = *reinterpret_cast<const uint16_t *>(codes + first);
#pragma unroll
        for (int i = 0; i < N / 2; i += 2) {
            out[i] = (uint32_t)lut_entry<0, uint16_t>(lut, raw[i / 2], slot) | ((uint32_t)lut_entry<1, uint16_t>(lut, raw[i / 2], slot) << 16);
            if constexpr (N > 2) out[i + 1] = (uint32_t)lut_entry<2, uint16_t>(lut, raw[i / 2], slot) | ((uint32_t)lut_entry<3, uint16_t>(lut, raw[i / 2], slot) << 16);
        }
    }
}

// 32 tokens of a row's uncompressed window: raw 16-bit keys and queries multiply exactly; probabilities enter the value product as three
// bf16 terms that add up to their float32 value, fp16 values as two that add up to theirs (two fp16 terms of a probability lie on a
// grid of 2^-38 of the largest one: at 2^-30 of it eight bits were left).  Record: [head][largest score, sum, D sums].  The values are
// loaded with the keys: their latency is the same, and a step of few rows waits for both.
template <int D, bool BF>
struct WindowTile {
    static constexpr int SK = D / 32, NC = D / 16;
    static constexpr int VW = D == 256 ? 0 : NC / 2;         // words of a token's columns held from the start (256: registers are short)
    tq_u4 q[SK], k[SK][2];
    uint32_t v[8][VW ? VW : 1];
    const uint8_t *kw, *vw;
    uint32_t left;

    static __device__ __forceinline__ uint32_t token(int j, uint32_t q4) { return 16u * (j / 4) + 4u * q4 + (uint32_t)(j % 4); }
    template <int N> __device__ __forceinline__ void load_columns(uint32_t (&dst)[8][N / 2], uint32_t lane, int c0) const {
        const uint32_t first = value_coord<D>(lane & 15u, c0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {      // past the end the last token is read again and not used
            const uint8_t *src = vw + (size_t)min(token(j, lane >> 4), left - 1u) * (2 * D) + 2u * first;
            if constexpr (N == 8) { const tq_u4 x = tq_gload16(src); dst[j][0] = x[0]; dst[j][1] = x[1]; dst[j][2] = x[2]; dst[j][3] = x[3]; }
            else if constexpr (N == 4) { const tq_u2 x = tq_gload8(src); dst[j][0] = x[0]; dst[j][1] = x[1]; }
            else dst[j][0] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)src);
        }
    }
    __device__ __forceinline__ void load(const TqDecodeArgs &a, uint32_t row, uint32_t wt, uint32_t lane) {
        const uint32_t n16 = lane & 15u, q4 = lane >> 4, t0 = wt * WIN_TILE;
        left = min((uint32_t)WIN_TILE, a.n_win - t0);
        kw = a.k_win + ((size_t)row * a.win_stride + (size_t)t0 * D) * 2u;
        vw = a.v_win + ((size_t)row * a.win_stride + (size_t)t0 * D) * 2u;
        const uint8_t *qs = a.queries + (((size_t)row * a.group + (n16 < a.group ? n16 : 0u)) * D + 8u * q4) * 2u;
#pragma unroll
        for (int s = 0; s < SK; ++s) {
            q[s] = tq_gload16(qs + 64 * s);
#pragma unroll
            for (int b = 0; b < 2; ++b) k[s][b] = tq_gload16(kw + (size_t)min(16u * b + n16, left - 1u) * (2 * D) + 64 * s + 16u * q4);
        }
        if constexpr (D == 64 || D == 128) load_columns<NC>(v, lane, 0);
        else if constexpr (D == 96) {
            uint32_t two[8][2], one[8][1];
            load_columns<4>(two, lane, 0);
            load_columns<2>(one, lane, 4);
#pragma unroll
            for (int j = 0; j < 8; ++j) { v[j][0] = two[j][0]; v[j][1] = two[j][1]; v[j][VW - 1] = one[j][0]; }
        }
    }
    __device__ __forceinline__ void finish(const TqDecodeArgs &a, TQ_GLOBAL float *rec, bool across, uint32_t lane) {
        constexpr int PART = D + 2;
        const uint32_t n16 = lane & 15u, q4 = lane >> 4, G = a.group;
        auto mm = [](tq_u4 x, tq_u4 y, tq_f4v c) { return BF ? mfma16_bf16(x, y, c) : mfma16_f16(x, y, c); };
        tq_f4v sc[2] = {tq_f4v{0.f, 0.f, 0.f, 0.f}, tq_f4v{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < SK; ++s)
#pragma unroll
            for (int b = 0; b < 2; ++b) sc[b] = mm(k[s][b], q[s], sc[b]);
        float t[8], m = -3.0e38f, l = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            t[j] = sc[j / 4][j % 4] * a.scale;       // token(j) of the tile, head n16
            if (token(j, q4) >= left) t[j] = -3.0e38f;
            m = fmaxf(m, t[j]);
        }
        m = reduce_rows(m, OpMax());
        float p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            p[j] = token(j, q4) < left ? __expf(t[j] - m) : 0.f;
            l += p[j];
        }
        l = reduce_rows(l, OpAdd());
        tq_u4 pa[3];
        split_f32x8(p, pa[0], pa[1], pa[2]);
        if (q4 == 0u && n16 < G) { put_record(across, rec + n16 * PART, m); put_record(across, rec + n16 * PART + 1u, l); }
        // columns in chunks of 8 (or 4, 2): the same element of token pairs side by side, one operand per coordinate
        auto columns = [&](auto n_tag, int c0, const auto &w, int w0) __attribute__((always_inline)) {
            constexpr int N = decltype(n_tag)::value;
            const uint32_t first = value_coord<D>(n16, c0);
            float odd = 0.f;         // NaN once a sum is not finite
            auto column = [&](tq_u4 bt, tq_f4v acc) __attribute__((always_inline)) {
                tq_u4 hi = bt, lo;
                if constexpr (!BF) split_f16x8(bt, hi, lo);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    acc = mfma16_bf16(pa[i], hi, acc);
                    if constexpr (!BF) acc = mfma16_bf16(pa[i], lo, acc);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) odd = fmaf(acc[r], 0.f, odd);
                return acc;
            };
            tq_f4v sum[N];
#pragma unroll
            for (int c = 0; c < N; ++c) {
                tq_u4 bt;
#pragma unroll
                for (int d = 0; d < 4; ++d)
                    bt[d] = __builtin_amdgcn_perm(w[2 * d + 1][w0 + c / 2], w[2 * d][w0 + c / 2], (c & 1) ? 0x07060302u : 0x05040100u);
                sum[c] = column(bt, tq_f4v{0.f, 0.f, 0.f, 0.f});
            }
            auto store = [&](auto across_tag) __attribute__((always_inline)) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (4u * q4 + r < G) {
#pragma unroll
                        for (int c = 0; c < N; c += 2) put_record2<decltype(across_tag)::value>(rec + (4u * q4 + r) * PART + 2u + first + c, sum[c][r], sum[c + 1][r]);
                    }
                }
            };
            if (across) store(std::true_type{}); else store(std::false_type{});
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
                        for (int i = 0; i < 2; ++i) {
                            const uint32_t tt = 16u * (d / 2) + 4u * q4 + 2u * (d % 2) + i;
                            if (tt < left) pair |= (uint32_t)tq_gload2(reinterpret_cast<const uint16_t *>(vw + (size_t)tt * (2 * D)) + first + c) << (16 * i);
                        }
                        constexpr uint32_t EXPO = BF ? 0x7f807f80u : 0x7c007c00u, ONE = BF ? 0x00800080u : 0x04000400u;
                        const uint32_t mask = ((((pair & EXPO) + ONE) >> 15) & 0x00010001u) * 0xffffu;     // exponent all ones
                        wild[d] = pair & mask;
                        if constexpr (!BF)
                            wild[d] = (wild[d] & 0x80008000u) | (mask & 0x7f807f80u) | ((((wild[d] & 0x03ff03ffu) + 0x03ff03ffu) >> 4) & 0x00400040u);
                        bt[d] = pair & ~mask;
                    }
                    const tq_f4v again = column(bt, mfma16_bf16(pa[0], wild, tq_f4v{0.f, 0.f, 0.f, 0.f}));
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (4u * q4 + r < G) put_record(across, rec + (4u * q4 + r) * PART + 2u + first + c, again[r]);
                }
            }
        };
        if constexpr (D == 64) columns(std::integral_constant<int, 4>{}, 0, v, 0);
        else if constexpr (D == 96) { columns(std::integral_constant<int, 4>{}, 0, v, 0); columns(std::integral_constant<int, 2>{}, 4, v, 2); }
        else if constexpr (D == 128) columns(std::integral_constant<int, 8>{}, 0, v, 0);
        else {
#pragma unroll 1
            for (int c0 = 0; c0 < NC; c0 += 8) {
                uint32_t w[8][4];
                load_columns<8>(w, lane, c0);
                columns(std::integral_constant<int, 8>{}, c0, w, 0);
            }
        }
    }
};

// Block (split, row), eight waves.  The main loop is the one of tq_attend_kernel (tq_attend.hip): a wave takes runs of 32 or 64
// tokens of the split, loaded one run ahead; scores transposed (A = decoded keys, B = rotated queries, heads in the 16
// columns), softmax in base 2 against a lazily moved per-head reference, probabilities times value norms as the A operand
// of the value product, whose B operand is built in the lanes from the staged codes.  Around it, in the same launch:
//   * waves 0 .. D/32 - 1 rotate the row's queries on the matrix cores (Rotation), the other waves attend to the window, 32 tokens
//     each (WindowTile);
//   * the waves' sums meet in LDS; with several splits per row the block that arrives last at the row's counter merges the
//     records of all splits and of the window, rotates the value sums back and stores the result.
// With few rows that is a chain of latencies, and what keeps it short (8 rows x 32768 tokens, K4/V2, 4 heads; clock stamps of a launch in 22
// splits, which the rule of then took, before / after; it takes 32 now): all loads of the start issued at once in the order of their use, tables found without their header, queries
// rotated by 4.2 / 2.5 us; the window's values loaded with its keys and its sums stored without a branch for each, 7.0 / 4.5; the block's
// tokens dealt out evenly; records merged with one trip to memory and a code of a few hundred bytes (code that runs once is fetched from
// the L2 as it goes: 1 us for 2.4 KiB of it), last arrival to result 5.5 / 3.4.
// A tile of the window used to stand before the block's barrier: everybody in it waited 2.3 us (256 wide 4.4) for the wave that had it, and the row for the
// block.  It is finished behind the barrier now; records are merged without loops around their loads.  us a layer, 4 heads, K4/V2: 8 rows x 32768
// tokens 21.0 -> 20.3; 4 x 6000 16.4 -> 15.0; 64 wide, 32 x 6000 15.8 -> 14.8; 256 wide, 8 x 16384 35.3 -> 33.0.
// Where the 16 us of a launch of 8 rows x 32768 tokens lie now (clock stamps, medians of the last block; together 15.1, the rest is before the first stamp and behind the
// last): 3.6 until the first tables and operands are
// there and the barrier is passed, 0.5 the queries' operands, 4.7 two runs a wave (what reading 26 MB takes), 1.0 the 8 tokens over, 1.2 the waves' sums, 0.9 stores and
// count, 2.3 the records of 32 blocks, 0.9 back through Pi_v.  What moved it last, a layer with its append: counters apart and Pi_v early 21.7 -> 20.9,
// history past the caches 19.8, products of 16 x 16 and tables in fewer loads 19.3.  (One loop body for whole and partial runs: a trip of it takes
// 2.05 us for 1.9 and the partial one still 1.0, a chain of latencies.  All waves rotating, or a barrier between the operands and the history: nothing
// at 128, 1 % longer at 96.)
// Before that, whole step of 32 layers 948 -> 778 us (734 since the append asks for all of its loads at once, see tq_decode.hip); 64 wide, 32 rows x 6000 tokens, K6/V4, 16 layers 394 -> 336; 512 rows x 16384 tokens, 8 layers 1565 -> 1404.
// The matrix products have 16 columns and a row of the cache seldom 16 query heads.  C blocks of 16 tokens share them (C = 4 for up to 4
// heads, 2 for up to 8): every block's scores are computed for the heads repeated C times, a lane keeps those of its own column's
// block, and the weights of the other blocks are zeros in its column of the value product.  The softmax of a token then costs 1 / C
// of what it did; columns of one head are added at the end.  With table addresses as one instruction: 512 rows x 16384
// tokens, K4/V2, 4 heads 202 -> 194 us; 64 wide, K6/V4, 512 rows x 32768 tokens, 4 heads 387 -> 357 us; 8 heads even (107 us at 256 rows).  Runs of
// 32 tokens have no room for C = 4.
// At 128 queries (against 8-bit keys: two terms) and weights enter the packed products as one fp16 term, as in tq_attend_kernel:
// their 2^-12 roundings stay under what the fp16 centroids cost.  The other head dimensions are as exact as float32 arithmetic:
//   * queries enter as two fp16 terms, Pi of fp16 caches as well (22 bits each).  Logits that come about by cancellation, where the
//     roundings show, are off by 0.5 to 0.8 of what the same products in float32 are off by (rotation and score, 64 to 256 wide).
//   * weights enter as three fp16 terms of p * 2^P_SHIFT * (value norm / 2^ev_ref) <= 2^15: 24 bits or more down to 2^-10 of the
//     reference weight times the largest value norm's binade, a grid of 2^-34 of that below (the smaller SLACK_LOG2, the finer).
//     Two terms on a grid of 2^-30 lost up to 2^-8 of weights around 2^-22 of the reference, a short history behind one token
//     that takes nearly everything.  The third one costs 4 to 5 % where rows are many (96 wide, 512 rows x 8000 tokens: 102 -> 107 us).
template <int D, int IPBK, int IPBV, int C, bool STREAM>
__global__ __launch_bounds__(DTHREADS, DW / 4) void tq_decode_kernel(TqDecodeArgs a) {
    static_assert(DTHREADS == LUT_THREADS, "threads that stage the tables");
    constexpr int QT = D != 128 || IPBK == 1 ? 2 : 1;    // fp16 terms of a rotated query
    constexpr int QREG = D == 256 && (IPBK == 1 || IPBV == 1) ? 1 : QT;      // terms held in registers, the others in LDS (see below)
    constexpr int PT = D != 128 ? 3 : 1;                 // fp16 terms of a weight
    constexpr int PART = D + 2;
    constexpr int TILES = D / 32;                        // waves that rotate queries
    constexpr int SK = D / 32;                           // score product: steps of 32 coordinates, 8 per lane
    constexpr int NC = D / 16;                           // value coordinates per lane
    constexpr int KB = D / 4 / IPBK;                     // key bytes per lane and token (D / 4 coordinates)
    constexpr int NWK = (KB + 3) / 4;
    constexpr int GBV = D / IPBV;                        // value bytes per vector
    constexpr int RUN = decode_run(D, IPBK, IPBV);       // tokens per wave and trip
    constexpr int SUB = RUN / 32;
    constexpr int HEADS = MAX_GROUP / C;                 // heads that the columns hold side by side for each of C blocks of tokens
    constexpr int UNIT = C == 4 ? 64 : 32;               // tokens of a softmax round
    constexpr int SPL = C == 1 ? 8 : 4;                  // their scores in a lane
    static_assert(UNIT <= RUN, "a round of softmax lies within a run");
    constexpr int VPB = GBV % 16 ? 8 : 16;               // value codes are staged in pieces of this size
    constexpr int VBYTES = RUN * GBV, VPIECES = VBYTES / VPB, NVP = (VPIECES + 63) / 64;
    constexpr int SLACK_LOG2 = PT == 1 ? 8 : 4;          // (several terms: the smaller it is, the finer the grid of small weights)
    constexpr int P_SHIFT = 14 - SLACK_LOG2;             // p * 2^P_SHIFT * (value norm / 2^ev_ref < 2) <= 2^15 fits fp16
    constexpr int HR = D == 256 && C == 1 ? 8 : HEADS;   // heads per round of the merge through LDS
    constexpr int AREA = VBYTES > HR * PART * 4 ? VBYTES : HR * PART * 4;    // per wave: staged value codes, later its sums
    constexpr bool EARLY_PV = D <= 128 && C > 1;         // rows of Pi_v asked for by every block that may be the last (see there)
    constexpr int QROW = D + 4;                          // rotated queries in LDS, floats per head
    constexpr int ROTP = DTHREADS / (D / 4) >= 16 ? 16 : DTHREADS / (D / 4);     // parts of the contraction when rotating back
    constexpr int ROTK = D / ROTP;                       // rows of Pi_v per part
    static_assert(DW * AREA >= 2 * MAX_GROUP * D * 4, "LDS area too small");

    __shared__ __attribute__((aligned(1024))) uint8_t lds_lut[65536];      // (the strictest alignment: lies at address 0, where no base has to be added)
    __shared__ __attribute__((aligned(16))) uint8_t lds_area[DW][AREA];
    __shared__ __attribute__((aligned(16))) float lds_kn[DW][RUN];
    __shared__ __attribute__((aligned(16))) std::conditional_t<PT == 1, uint16_t, float> lds_vn[DW][RUN];     // value norms / 2^ev_ref (uint16_t: as fp16)
    __shared__ __attribute__((aligned(16))) tq_u4 lds_q[QT > QREG ? (QT - QREG) * SK : 1][TQ_WAVE];
    __shared__ __attribute__((aligned(16))) float lds_qrot[MAX_GROUP][QROW];
    __shared__ __attribute__((aligned(16))) float lds_corr[DW][16];
    __shared__ float lds_den[MAX_GROUP];
    __shared__ uint32_t lds_last;
    __shared__ uint32_t lds_trips[DW];                   // runs a wave has begun

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = tq_uniform32(tid >> 6);
    const uint32_t row = blockIdx.y, split = blockIdx.x, splits = gridDim.x;
    const uint32_t n16 = lane & 15u, q4 = lane >> 4;
    const uint32_t G = a.group;
    const uint32_t head = n16 % HEADS, cls = n16 / HEADS;
    const bool live = head < G;

    const uint32_t win_tiles = (a.n_win + WIN_TILE - 1u) / WIN_TILE;     // tile w goes to the block of split w % splits
    // (the same cut of the history whatever the window holds: a sum in other parts is another rounding)
    const uint32_t t_begin = min(a.tokens, split * a.chunk);
    const uint32_t t_end = min(a.tokens, t_begin + a.chunk);
    const size_t slot0 = (size_t)row * a.packed_row_stride;
    uint8_t *vcodes = lds_area[wave];
    // Runs of a wave: in every whole round of the block one of RUN tokens; what is left of the block's tokens is dealt out evenly, in
    // blocks of 16 tokens, so that no wave works on a whole run alone at the end.
    const uint32_t rounds = (t_end - t_begin) / (RUN * DW);
    const uint32_t rest0 = t_begin + rounds * (RUN * DW);
    const uint32_t share = (t_end - rest0 + 16u * DW - 1u) / (16u * DW) * 16u;
    const uint32_t tail0 = min(t_end, rest0 + wave * share), n_tail = min(t_end, tail0 + share) - tail0;
    auto run_start = [&](uint32_t i) { return i < rounds ? t_begin + (i * DW + wave) * RUN : tail0; };
    auto run_tokens = [&](uint32_t i) { return i < rounds ? (uint32_t)RUN : i == rounds ? n_tail : 0u; };

    // Loads of a run, issued one run ahead: values and norms again as soon as the run has been staged, keys when its scores are done.
    // (A second register set, with keys issued a little earlier, made two copies of the loop: no faster with many rows, and with few every
    // copy is fetched for the first time, 512 rows x 16384 tokens 171 against 171 us, 128 rows x 4182 tokens 24.6 against 25.1.)
    uint32_t kraw[SUB][2][NWK];
    tq_u4 vpiece[NVP];
    uint16_t kn_raw, vn_raw;
    // n_tok >= 1: what lies past the last token is read as that token.  One form for whole and partial runs: with a branch between two
    // the registers are merged behind it, and that waits for the loads just issued.
    constexpr bool KEYS = STREAM && !(IPBK == 1 && (D == 256 || (D == 128 && C == 1)));      // keys streamed as well (see launch_decode)
    auto load16 = [](const uint8_t *p, auto hint) __attribute__((always_inline)) { return decltype(hint)::value ? tq_gload16_stream(p) : tq_gload16(p); };
    auto load8 = [](const uint8_t *p, auto hint) __attribute__((always_inline)) { return decltype(hint)::value ? tq_gload8_stream(p) : tq_gload8(p); };
    constexpr std::integral_constant<bool, KEYS> key_hint{};
    constexpr std::integral_constant<bool, STREAM> value_hint{};
    auto issue_keys = [&](uint32_t t0, uint32_t n_tok) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < SUB; ++u)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                const uint32_t tl = 32u * u + 16u * b + n16;
                const uint8_t *src = a.k_idx + (slot0 + t0) * (4 * KB) + min(tl, n_tok - 1u) * (4 * KB) + q4 * KB;
                if constexpr (KB % 16 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 16; ++p) {
                        const tq_u4 v = load16(src + 16 * p, key_hint);
#pragma unroll
                        for (int i = 0; i < 4; ++i) kraw[u][b][4 * p + i] = v[i];
                    }
                } else if constexpr (KB % 8 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 8; ++p) {
                        const tq_u2 v = load8(src + 8 * p, key_hint);
                        kraw[u][b][2 * p] = v[0]; kraw[u][b][2 * p + 1] = v[1];
                    }
                } else if constexpr (KB % 4 == 0) {
#pragma unroll
                    for (int p = 0; p < KB / 4; ++p)
                        kraw[u][b][p] = KEYS ? tq_gload4_stream(src + 4 * p) : tq_gload4(src + 4 * p);
                } else {
                    static_assert(KB % 2 == 0, "key bytes of a lane");
                    uint32_t h[KB / 2];
#pragma unroll
                    for (int p = 0; p < KB / 2; ++p) h[p] = tq_gload2(reinterpret_cast<const uint16_t *>(src) + p);
#pragma unroll
                    for (int p = 0; p < NWK; ++p) kraw[u][b][p] = h[2 * p] | (2 * p + 1 < KB / 2 ? h[2 * p + 1 < KB / 2 ? 2 * p + 1 : 0] << 16 : 0u);
                }
            }
    };
    auto issue_values = [&](uint32_t t0, uint32_t n_tok) __attribute__((always_inline)) {
        const uint8_t *vsrc = a.v_idx + (slot0 + t0) * GBV;
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
            const uint32_t piece = min(p * 64u + lane, min((uint32_t)VPIECES, n_tok * (GBV / VPB)) - 1u);
            if constexpr (VPB == 16) vpiece[p] = load16(vsrc + piece * 16u, value_hint);
            else { const tq_u2 v = load8(vsrc + piece * 8u, value_hint); vpiece[p][0] = v[0]; vpiece[p][1] = v[1]; }
        }
        const uint32_t own = min(lane, n_tok - 1u);       // (lanes past the end: see trip)
        kn_raw = tq_gload2(a.k_norms + slot0 + t0 + own);
        vn_raw = tq_gload2(a.v_norms + slot0 + t0 + own);
    };

    // ---- start: loads in the order in which their data is used, nothing waits for what it does not need.  Tables, then the operands of
    // the query rotation (the first waves) or a tile of the window (from the last wave down), then the first run; a wave that has no run
    // reads the row's first token (of a row without history, what the host put there instead).
    uint32_t wt = DW - 1u - wave;
    TQ_GLOBAL float *wrec = (TQ_GLOBAL float *)a.win_part + (size_t)row * win_tiles * G * PART;
    if (tid < (uint32_t)DW) lds_trips[tid] = 0u;
    Lut<IPBK> table_k;
    Lut<IPBV> table_v;
    table_k.load(a.table_k + TQ_OFF_LUT(D), tid);
    table_v.load(a.table_v + TQ_OFF_LUT(D), tid);
    __builtin_amdgcn_sched_barrier(0);
    auto first_run = [&]() __attribute__((always_inline)) {
        const uint32_t n0 = run_tokens(0u), t0 = n0 ? run_start(0u) : 0u;
        __builtin_amdgcn_sched_barrier(0);
        issue_keys(t0, max(n0, 1u));
        issue_values(t0, max(n0, 1u));
        __builtin_amdgcn_sched_barrier(0);
        table_k.store(lds_lut, tid);
        table_v.store(lds_lut + 128, tid);
    };
    // The barrier stands where rotated queries and tables are complete.  What is left of the window comes behind it: its waves, and nobody
    // else, begin their runs later.
    auto window = [&](auto bf_tag) __attribute__((always_inline)) {
#pragma unroll 1
        for (; split + wt * splits < win_tiles; wt += DW) {
            WindowTile<D, decltype(bf_tag)::value> w;
            w.load(a, row, split + wt * splits, lane);
            w.finish(a, wrec + (size_t)(split + wt * splits) * G * PART, splits > 1u, lane);
        }
    };
    auto start = [&](auto bf_tag) __attribute__((always_inline)) {
        constexpr bool BF = decltype(bf_tag)::value;
        if (wave < (uint32_t)TILES) {
            Rotation<D, BF> r;
            r.load(a.queries + (size_t)row * G * D * 2u, G, a.table_k, wave, lane);
            first_run();
            r.finish(&lds_qrot[0][0], QROW, a.scale, wave, lane);
            // (256 wide a tile takes several runs' time, and where every split has one or more it is better spent together: 128 rows x 4000
            // tokens, K8/V8, 8 heads, eight layers 809 us, behind the barrier 857)
            if (D == 256 && win_tiles > splits) window(bf_tag);
            __syncthreads();
        } else if (split + wt * splits < win_tiles) {
            WindowTile<D, BF> w;
            w.load(a, row, split + wt * splits, lane);
            first_run();
            __syncthreads();
            w.finish(a, wrec + (size_t)(split + wt * splits) * G * PART, splits > 1u, lane);
            wt += DW;
        } else {
            first_run();
            __syncthreads();
        }
    };
    if (a.bf16) { start(std::true_type{}); window(std::true_type{}); } else { start(std::false_type{}); window(std::false_type{}); }

    // ---- B operand of the score product: fp16 of q * 2^(10 - e), e = binary exponent of the head's largest magnitude.  At 256 with
    // 8-bit codes on either side registers run out (28 spilled with 8-bit keys and values): the low term, the same in every wave, lies
    // in LDS and serves both blocks of a step (128 rows x 8000 tokens, K8/V8: 211 -> 156 us).
    tq_u4 qb[QREG][SK];
    float c1;                // score in base-2 units = t * c1, t = accumulator * key norm
    float rowscale;          // natural score = t * rowscale
    {
        const float *q = &lds_qrot[head][(D / 4) * q4];
        float x[D / 4];
#pragma unroll
        for (int i = 0; i < D / 4; i += 4) {
            const float4 f = *reinterpret_cast<const float4 *>(q + i);
            x[i] = f.x; x[i + 1] = f.y; x[i + 2] = f.z; x[i + 3] = f.w;
        }
        float big = 0.f;
#pragma unroll
        for (int i = 0; i < D / 4; ++i) big = fmaxf(big, fabsf(x[i]));
        big = reduce_rows(big, OpMax());
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
            for (int k = QREG; k < QT; ++k)         // the same in every wave, and each writes it: none waits for another
                lds_q[(k - QREG) * SK + s][lane] = __builtin_bit_cast(tq_u4, term[k]);
        }
    }
    const uint32_t slot_k = RepLut<IPBK>::lane_offset(lane), slot_v = 128u + RepLut<IPBV>::lane_offset(lane);
    tq_f4v acc[NC];          // weighted value sums: register r = column 4 q4 + r of the scores (head and block of tokens), c = coordinate value_coord(n16, c)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = tq_f4v{0.f, 0.f, 0.f, 0.f};
    // Softmax reference of this lane's head, in units of t (the lanes of a head agree): it moves only when a score
    // exceeds it by more than SLACK_LOG2 binary orders, so the common tile needs no exchange between lanes.
    float m_ref = -1e30f;
    float l_run = 0.f;       // running sum of p * 2^P_SHIFT over this lane's tokens
    const float slack = live ? (float)SLACK_LOG2 / c1 : 3.0e38f;
    int ev_ref = -100;       // largest binary exponent of a value norm this wave has seen; the sums are in units of 2^ev_ref

    // one run of staged tokens; FULL: all of them exist.  The score products of all its tiles come first, so that a later
    // tile's matrix work runs under an earlier one's softmax.
    auto run = [&](auto full_tag, uint32_t n_tok, uint32_t t_next, uint32_t n_next) __attribute__((always_inline)) {
        constexpr bool FULL = decltype(full_tag)::value;
        tq_f4v sc[SUB][2];   // register r of block b = token 32 u + 16 b + 4 q4 + r
#pragma unroll
        for (int u = 0; u < SUB; ++u) {
            sc[u][0] = sc[u][1] = tq_f4v{0.f, 0.f, 0.f, 0.f};
            if (!FULL && 32u * u >= n_tok) continue;       // uniform
            auto step = [&](int b, int s, const tq_u4 (&q)[QT]) __attribute__((always_inline)) {
                const tq_u4 kd = decode_keys<IPBK, NWK>(kraw[u][b], s, lds_lut, slot_k);
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
        if constexpr (FULL) issue_keys(t_next, n_next);
#pragma unroll
        for (int u = 0; u < RUN / UNIT; ++u) {
            if (!FULL && (uint32_t)(UNIT * u) >= n_tok) break;  // uniform
            // tokens of this lane: tok .. tok + 3 (C = 1: and tok + 16 .. tok + 19)
            const uint32_t tok = (uint32_t)(UNIT * u) + 16u * cls + 4u * q4;
            float t[SPL];
#pragma unroll
            for (int b = 0; b < SPL / 4; ++b) {
                tq_f4v own = sc[(UNIT / 32) * u][b];
                if constexpr (C > 1) {
#pragma unroll
                    for (int k = 1; k < C; ++k) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) own[r] = cls == (uint32_t)k ? sc[(UNIT / 32) * u + k / 2][k % 2][r] : own[r];
                    }
                }
                const float4 k4 = *reinterpret_cast<const float4 *>(&lds_kn[wave][tok + 16u * b]);
                t[4 * b + 0] = own[0] * k4.x; t[4 * b + 1] = own[1] * k4.y;
                t[4 * b + 2] = own[2] * k4.z; t[4 * b + 3] = own[3] * k4.w;
            }
            if constexpr (!FULL) {
#pragma unroll
                for (int j = 0; j < SPL; ++j)
                    if (tok + 16u * (j / 4) + (j % 4) >= n_tok) t[j] = -1e30f;
            }
            float tmax = fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]));
            if constexpr (SPL == 8) tmax = fmaxf(tmax, fmaxf(fmaxf(t[SPL - 4], t[SPL - 3]), fmaxf(t[SPL - 2], t[SPL - 1])));
            if (__any(tmax > m_ref + slack)) {     // (rare after the first tiles) move the head's reference, rescale its sums
                float tm = tmax;
#pragma unroll
                for (int d = HEADS; d < 64; d <<= 1) tm = fmaxf(tm, __shfl_xor(tm, d));
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
            float ps[SPL];
            float lsum = 0.f;
#pragma unroll
            for (int j = 0; j < SPL; ++j) {
                ps[j] = __builtin_amdgcn_exp2f(fmaf(t[j], c1, bias));     // p * 2^P_SHIFT, p <= 2^SLACK_LOG2
                if constexpr (!FULL) {   // a zero query makes every exponent 0: masked tokens need an explicit zero
                    if (tok + 16u * (j / 4) + (j % 4) >= n_tok) ps[j] = 0.f;
                }
                lsum += ps[j];
            }
            l_run += lsum;
            // ---- weights p_j |v_j| / 2^ev_ref of the lane's own tokens, in pairs
            uint32_t w[PT][SPL / 2];
#pragma unroll
            for (int b = 0; b < SPL / 4; ++b) {
                if constexpr (PT == 1) {
                    const tq_u2 nrm = *reinterpret_cast<const tq_u2 *>(&lds_vn[wave][tok + 16u * b]);
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        const tq_half2 two = tq_half2{(_Float16)ps[4 * b + 2 * d], (_Float16)ps[4 * b + 2 * d + 1]} * __builtin_bit_cast(tq_half2, (uint32_t)nrm[d]);
                        w[0][2 * b + d] = __builtin_bit_cast(uint32_t, two);
                    }
                } else {
                    const float4 vn = *reinterpret_cast<const float4 *>(&lds_vn[wave][tok + 16u * b]);
                    float x[4] = {ps[4 * b] * vn.x, ps[4 * b + 1] * vn.y, ps[4 * b + 2] * vn.z, ps[4 * b + 3] * vn.w};
#pragma unroll
                    for (int k = 0; k < PT; ++k)
#pragma unroll
                        for (int d = 0; d < 2; ++d) {
                            const auto two = __builtin_amdgcn_cvt_pkrtz(x[2 * d], x[2 * d + 1]);
                            w[k][2 * b + d] = __builtin_bit_cast(uint32_t, two);
                            x[2 * d] -= (float)two[0];
                            x[2 * d + 1] -= (float)two[1];
                        }
                }
            }
#pragma unroll
            for (int tile = 0; tile < UNIT / 32; ++tile) {
                if (!FULL && (uint32_t)(UNIT * u + 32 * tile) >= n_tok) break;  // uniform
                // slice j of lane (., q4) = token tok_a + j (j < 4), tok_b + j - 4; a column holds the weights of its own block of tokens
                const uint32_t tok_a = (uint32_t)(UNIT * u + 32 * tile) + 4u * q4, tok_b = tok_a + 16u;
                tq_u4 pa[PT];
#pragma unroll
                for (int k = 0; k < PT; ++k)
#pragma unroll
                    for (int d = 0; d < 4; ++d)
                        pa[k][d] = C == 1 ? w[k][d % (SPL / 2)] : (cls == (uint32_t)(2 * tile + d / 2) ? w[k][d % 2] : 0u);
                auto columns = [&](auto n_tag, int c0) __attribute__((always_inline)) {
                    constexpr int N = decltype(n_tag)::value;
                    uint32_t dec[8][N / 2];      // per token: N coordinates of the lane as fp16
                    const uint32_t first = value_coord<D>(n16, c0);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        decode_values<IPBV, N>(vcodes + ((j < 4 ? tok_a : tok_b) + (uint32_t)(j % 4)) * GBV, first, lds_lut, slot_v, dec[j]);
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
        }
    };

    // one trip: stage the run that has been loaded, start the loads of the next one, compute
    // The two waves of a SIMD (w and w + 4) are kept level: the one that is ahead yields.  Left alone the older of the two is
    // served first, and the other one ends its runs without anybody to cover its waits: of a row of 16384 tokens the first
    // waves had done their 32 runs after 69 us and waited 22 us for the others; now all take 84 us and wait one
    // (512 rows, the launch, median over eight layers in turn: 208 -> 200-204 us).  Which wave takes which run stays fixed, so the sums do too.
    uint32_t trips = 0u;
    auto keep_level = [&]() __attribute__((always_inline)) {
        ++trips;
        volatile __attribute__((address_space(3))) uint32_t *count = (__attribute__((address_space(3))) uint32_t *)lds_trips;
        if (lane == 0u) count[wave] = trips;
        if (trips > tq_uniform32(count[wave ^ 4u])) __builtin_amdgcn_s_setprio(0); else __builtin_amdgcn_s_setprio(1);
    };
    auto trip = [&](auto full_tag, uint32_t i) __attribute__((always_inline)) {
        keep_level();
        constexpr bool FULL = decltype(full_tag)::value;
        const uint32_t n_tok = FULL ? (uint32_t)RUN : run_tokens(i);
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
            const uint32_t piece = p * 64u + lane;
            if (VPIECES % 64 == 0 || piece < VPIECES) {
                if constexpr (VPB == 16) *reinterpret_cast<tq_u4 *>(vcodes + piece * 16u) = vpiece[p];
                else *reinterpret_cast<tq_u2 *>(vcodes + piece * 8u) = tq_u2{vpiece[p][0], vpiece[p][1]};
            }
        }
        {
            const _Float16 kh = __builtin_bit_cast(_Float16, kn_raw);
            if (RUN == 64 || lane < (uint32_t)RUN) lds_kn[wave][lane] = (float)kh;     // one token per lane
            // does a value norm of this run exceed the reference exponent?  (a vote; a handful of times per wave)
            const uint16_t vn = (FULL && RUN == 64) || lane < n_tok ? vn_raw : (uint16_t)0;   // tokens past the end weigh nothing
            uint32_t e = ((uint32_t)vn >> 10) & 31u;
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
            const _Float16 vh = __builtin_bit_cast(_Float16, vn);
            const float vs = ldexpf((float)vh, -ev_ref);
            if (RUN == 64 || lane < (uint32_t)RUN) {
                if constexpr (PT == 1) lds_vn[wave][lane] = __builtin_bit_cast(uint16_t, (_Float16)vs);
                else lds_vn[wave][lane] = vs;
            }
        }
        // (behind the last run the row's first token is read again)
        const uint32_t n_more = run_tokens(i + 1u), t_next = n_more ? run_start(i + 1u) : 0u, n_next = max(n_more, 1u);
        if constexpr (FULL) issue_values(t_next, n_next);
        asm volatile("" ::: "memory");    // staged with one access width, read back with others (LDS serves a wave in order)
        __builtin_amdgcn_wave_barrier();
        run(full_tag, n_tok, t_next, n_next);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    };
    {
        // whole runs in the loop, the partial one (a wave has one at most) behind it: with both kinds in one loop body the
        // accumulators are copied where they meet and registers spill
        uint32_t i = 0u;
        while (run_tokens(i) == (uint32_t)RUN) trip(std::true_type{}, i++);
        if (run_tokens(i)) trip(std::false_type{}, i);
        if (lane == 0u) *(volatile __attribute__((address_space(3))) uint32_t *)&lds_trips[wave] = 0xffffffffu;
        __builtin_amdgcn_s_setprio(0);
    }
    asm volatile("" ::: "memory");

    // ---- the waves' sums of HR heads at a time meet in LDS: record [head][largest natural score, sum, D sums] of the split
    float *dst = a.partial + ((size_t)row * splits + split) * G * PART;
    float l_all = l_run;
#pragma unroll
    for (int d = HEADS; d < 64; d <<= 1) l_all += __shfl_xor(l_all, d);
    l_all *= 1.0f / (float)(1 << P_SHIFT);
    const float out_scale = ldexpf(1.f, ev_ref - P_SHIFT);
    for (uint32_t h0 = 0; h0 < G; h0 += HR) {
        float *res = reinterpret_cast<float *>(lds_area[wave]);
        if (h0) __syncthreads();
        if (q4 == 0u && cls == 0u && n16 >= h0 && n16 < h0 + HR) {
            res[(n16 - h0) * PART] = m_ref * rowscale;
            res[(n16 - h0) * PART + 1u] = l_all;
        }
        if constexpr (C == 1) {
            if (4u * q4 >= h0 && 4u * q4 < h0 + HR) {
#pragma unroll
                for (int c = 0; c < NC; ++c)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        res[(4u * q4 + r - h0) * PART + 2u + value_coord<D>(n16, c)] = acc[c][r] * out_scale;
            }
        } else {
            // The blocks of tokens lie in lanes 32 apart (C = 4: and 16 apart): two registers exchange halves and are added, which
            // leaves the sum of one in each half (then the same with quarters).
            static_assert(HR >= HEADS, "one round");
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float half[NC / 2];
#pragma unroll
                for (int c = 0; c < NC; c += 2) half[c / 2] = fold<32>(acc[c][r], acc[c + 1][r]);
                if constexpr (C == 2) {
#pragma unroll
                    for (int c = 0; c < NC; c += 2)
                        res[(4u * (q4 & 1u) + r) * PART + 2u + value_coord<D>(n16, c + (int)(q4 >> 1))] = half[c / 2] * out_scale;
                } else {
#pragma unroll
                    for (int c = 0; c < NC; c += 4) {
                        const bool pair = c + 2 < NC;     // (96: the last two columns stand alone, both quarters hold them)
                        const float sum = fold<16>(half[c / 2], half[pair ? c / 2 + 1 : c / 2]);
                        res[r * PART + 2u + value_coord<D>(n16, c + (int)((pair ? 2u * (q4 & 1u) : 0u) + (q4 >> 1)))] = sum * out_scale;
                    }
                }
            }
        }
        __syncthreads();
        for (uint32_t i = 2u * tid; i < min((uint32_t)HR, G - h0) * D; i += 2u * DTHREADS) {
            const uint32_t g = i / D, j = i % D;
            const float *rec = reinterpret_cast<const float *>(lds_area[0]) + g * PART;      // wave w: AREA bytes further
            float f[DW], mall = -3.0e38f, v0 = 0.f, v1 = 0.f;
#pragma unroll
            for (int w = 0; w < DW; ++w) {
                f[w] = rec[w * (AREA / 4)];
                mall = fmaxf(mall, f[w]);
            }
#pragma unroll
            for (int w = 0; w < DW; ++w) {
                f[w] = __expf(f[w] - mall);
                const float2 two = *reinterpret_cast<const float2 *>(rec + w * (AREA / 4) + 2u + j);
                v0 += f[w] * two.x;
                v1 += f[w] * two.y;
            }
            TQ_GLOBAL float *out = (TQ_GLOBAL float *)dst + (h0 + g) * PART;
            if (splits > 1u) put_record2<true>(out + 2u + j, v0, v1); else put_record2<false>(out + 2u + j, v0, v1);
            if (j == 0u) {
                float l = 0.f;
#pragma unroll
                for (int w = 0; w < DW; ++w) l += f[w] * rec[w * (AREA / 4) + 1];
                if (splits > 1u) put_record2<true>(out, mall, l); else put_record2<false>(out, mall, l);
            }
        }
    }

    // ---- the last block of the row finishes it
    // (the records were stored at device scope: once every wave has waited for its own stores, which the barrier by itself does not
    // do, thread 0 may count the block as done, see put_record)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // Rows of Pi_v for the rotation back: thread (four columns, part) takes ROTK of them.  Where registers allow they are asked for right behind
    // the atomic, by every block, so that they arrive while its answer is on its way and only the records are left to wait for: 8 rows x
    // 32768 tokens, from the last block's count to merged sums 2.9 -> 2.3 us (the other blocks drop them: 64 KB of the L2 each at 128).
    // At 256 (four times as much) and for more than eight heads they are loaded behind the records.
    const uint32_t rc = (tid % (D / 4)) * 4u, rp = tid / (D / 4);
    tq_u4 pv[ROTK];
    auto load_pv = [&]() __attribute__((always_inline)) {
        const uint8_t *src = reinterpret_cast<const uint8_t *>(a.pi_v + (size_t)(min(rp, (uint32_t)ROTP - 1u) * ROTK) * D + rc);
#pragma unroll
        for (int k = 0; k < ROTK; ++k) pv[k] = tq_gload16(src + k * (D * 4));
    };
    if (splits > 1u) {
        uint32_t before = 0u;
        if (tid == 0u) before = __hip_atomic_fetch_add(a.arrived + (size_t)row * a.arrived_stride, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if constexpr (EARLY_PV) {
            __builtin_amdgcn_sched_barrier(0);
            load_pv();
            __builtin_amdgcn_sched_barrier(0);
        }
        if (tid == 0u) {
            const bool last = before == splits - 1u;
            if (last) __hip_atomic_store(a.arrived + (size_t)row * a.arrived_stride, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            lds_last = last ? 1u : 0u;
        }
        __syncthreads();
        if (!lds_last) return;
    }
    float *ysum = reinterpret_cast<float *>(&lds_area[0][0]);     // [head][D]: sums in the rotated space
    float *wsum = ysum + MAX_GROUP * D;                           // [head][D]: the window's, plain
    // Where few records meet there is one trip to memory: references and sums of exp of a head's records (a lane each), the sums (four columns
    // a lane, every fourth record; the quarters of a wave are added in registers) and, if they are not on their way already, the rows of Pi_v,
    // which are needed last, are under way together.  No loop holds a load there: behind one the compiler waits for everything in flight, the rows of Pi_v among it (32 rows x 6000
    // tokens, 64 wide, from the last arrival to merged sums: 1.9 us with loops, now 1.4).  What is left grows with the records: one compute unit reads
    // what other dies wrote at some 27 KB/us (8 rows x 32768, 66 KB: 2.4 us; 256 wide, 8 x 9906, 120 KB and 256 KB of Pi_v: 5.2).  Little code: it runs once and is fetched for the first time
    // (33 loads a lane, written out: 2.0 us from the first to the last of them, now 0.4).
    // Two heads a wave where a row has more than eight: they went through the loops of `many` (16 heads, 32 rows x 6000 tokens, us: 64 wide
    // 20.4, this way 18.2, 128 wide 28.7 / 25.8).  `many` takes the references with as few loads as there are records for, and asks for a further 32
    // records only where there are any (2 rows x 20000 tokens, about 40 splits, 128 wide, 8 heads 21.9 / 20.9, 16 heads 29.7 / 27.3).
    auto merge = [&](auto across_tag) __attribute__((always_inline)) {
        constexpr bool ACROSS = decltype(across_tag)::value;
        const uint32_t step = G * PART, nrec = splits + win_tiles;    // (a row's records lie within 4.5 MiB)
        const Records part(a.partial + (size_t)row * splits * step, splits * step), wpart(a.win_part + (size_t)row * win_tiles * step, win_tiles * step);
        // weights of the records: exp(reference - largest reference of the head)
        float *wgt = reinterpret_cast<float *>(lds_lut);              // [head][splits, then window tiles: each up to a multiple of 4, zeros behind]
        const uint32_t wfirst = (splits + 3u) / 4u * 4u, wrow = wfirst + (win_tiles + 3u) / 4u * 4u;
        auto place = [&](uint32_t s) { return s < splits ? s : wfirst + s - splits; };
        auto fetch = [&](auto &y, uint32_t off, uint32_t s0) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < (int)(sizeof(y) / sizeof(y[0])); ++s) y[s] = part.load4<ACROSS>((s0 + 4u * s + q4) * step + off);
        };
        float ys[4], ws[4];
        auto add_records = [&](const auto &y, const float *f, uint32_t s0) __attribute__((always_inline)) {
#pragma unroll
            for (int s = 0; s < (int)(sizeof(y) / sizeof(y[0])); ++s) {
                if (s0 + 4u * s >= splits) break;     // (uniform)
                const float fs = f[s0 + 4 * s];       // (zero for what lies past the last record)
#pragma unroll
                for (int c = 0; c < 4; ++c) ys[c] = fmaf(fs, __uint_as_float(y[s][c]), ys[c]);
            }
        };
        auto add_window = [&](tq_u4 w, float f) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 4; ++c) ws[c] = fmaf(f, __uint_as_float(w[c]), ws[c]);
        };
        auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 4; ++c) ys[c] = ws[c] = 0.f;
        };
        auto put_sums = [&](uint32_t p) __attribute__((always_inline)) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                ys[c] = reduce_rows(ys[c], OpAdd());
                ws[c] = reduce_rows(ws[c], OpAdd());
            }
            if (q4 == 0u) {
                *reinterpret_cast<float4 *>(ysum + p) = make_float4(ys[0], ys[1], ys[2], ys[3]);
                *reinterpret_cast<float4 *>(wsum + p) = make_float4(ws[0], ws[1], ws[2], ws[3]);
            }
        };
        const uint32_t col = (wave * 16u + n16) * 4u;                 // + DTHREADS: further heads
        // references and sums of exp of head g's records, R x 64 of them, a lane each (of either kind: where there is none of one it reads as zero)
        auto load_heads = [&](auto &ml, uint32_t g) __attribute__((always_inline)) {
#pragma unroll
            for (int k = 0; k < (int)(sizeof(ml) / sizeof(ml[0])); ++k) {
                const uint32_t s = 64u * k + lane;
                const tq_u2 hs = part.load2<ACROSS>(s * step + g * PART), hw = wpart.load2<ACROSS>((s - splits) * step + g * PART);
                ml[k] = s < splits ? hs : hw;
            }
        };
        auto weigh = [&](const auto &ml, uint32_t g) __attribute__((always_inline)) {
            constexpr int R = sizeof(ml) / sizeof(ml[0]);
            float m = -3.0e38f, den = 0.f;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t s = 64u * k + lane;
                if (s < nrec) m = fmaxf(m, __uint_as_float(ml[k][0]));
                if (s < wrow) wgt[g * wrow + s] = 0.f;       // (the LDS serves a wave in order)
            }
            m = reduce_wave(m, OpMax());
            asm volatile("" ::: "memory");
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const uint32_t s = 64u * k + lane;
                if (s < nrec) {
                    const float f = __expf(__uint_as_float(ml[k][0]) - m);
                    wgt[g * wrow + place(s)] = f;
                    den = fmaf(f, __uint_as_float(ml[k][1]), den);
                }
            }
            den = reduce_wave(den, OpAdd());
            if (lane == 0u) lds_den[g] = den;
        };
        auto few = [&](auto passes) __attribute__((always_inline)) {
            constexpr int N = decltype(passes)::value;                // of 512 columns
            constexpr int H = C == 1 ? 2 : 1;                         // heads a wave weighs
            tq_u4 y[N][8], w[N];
            tq_u2 ml[H][1];
#pragma unroll
            for (int h = 0; h < H; ++h) load_heads(ml[h], wave + h * DW);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const uint32_t p = col + k * DTHREADS, off = p / D * PART + 2u + p % D;
                fetch(y[k], off, 0u);
                w[k] = wpart.load4<ACROSS>(q4 * step + off);
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (N <= 2 && !(ACROSS && EARLY_PV)) load_pv();                          // (more columns leave no registers for them yet)
#pragma unroll
            for (int h = 0; h < H; ++h)
                if (wave + h * DW < G) weigh(ml[h], wave + h * DW);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const uint32_t p = col + k * DTHREADS;
                if (p >= G * D) break;
                const float *f = wgt + p / D * wrow + q4;
                clear();
                add_records(y[k], f, 0u);
                if (win_tiles) add_window(w[k], f[wfirst]);
                put_sums(p);
            }
            if constexpr (N > 2 && !(ACROSS && EARLY_PV)) load_pv();
            __syncthreads();
        };
        if (splits <= 32u && win_tiles <= 4u) {      // (launched for at most HEADS heads, HEADS = 16 for 9 at least, see launch_decode)
            constexpr int LEAST = C == 1 ? 9 : 1;
            if constexpr (LEAST * D <= DTHREADS) {
                if (G * D <= (uint32_t)DTHREADS) { few(std::integral_constant<int, 1>{}); return; }
            }
            if constexpr (HEADS * D > DTHREADS && LEAST * D <= 2 * DTHREADS) {
                if (G * D <= 2u * DTHREADS) { few(std::integral_constant<int, 2>{}); return; }
            }
            if constexpr (HEADS * D > 2 * DTHREADS && HEADS * D <= 4 * DTHREADS) { few(std::integral_constant<int, 4>{}); return; }
        }
        auto many = [&](auto reads) __attribute__((always_inline)) {      // of 64 records' references each
            tq_u4 y[8], w;
            tq_u2 ml[decltype(reads)::value];
            load_heads(ml, wave);
            fetch(y, col / D * PART + 2u + col % D, 0u);
            w = wpart.load4<ACROSS>(q4 * step + col / D * PART + 2u + col % D);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (D <= 128 && !(ACROSS && EARLY_PV)) load_pv();
            for (uint32_t g = wave; g < G; g += DW) {
                if (g != wave) load_heads(ml, g);
                weigh(ml, g);
            }
            __syncthreads();
            for (uint32_t p = col; p < G * D; p += DTHREADS) {
                const uint32_t g = p / D, off = g * PART + 2u + p % D;
                const float *f = wgt + g * wrow + q4;
                if (p != col) {
                    fetch(y, off, 0u);
                    w = wpart.load4<ACROSS>(q4 * step + off);
                }
                clear();
                uint32_t s0 = 0;
                for (; s0 + 32u < splits; s0 += 32u) {       // the next 32 records under way while these are added
                    tq_u4 z[8];
                    fetch(z, off, s0 + 32u);
                    add_records(y, f, s0);
#pragma unroll
                    for (int s = 0; s < 8; ++s) y[s] = z[s];
                }
                add_records(y, f, s0);
                if (win_tiles) add_window(w, f[wfirst]);
                for (uint32_t t = 4u; t < win_tiles; t += 4u) add_window(wpart.load4<ACROSS>((t + q4) * step + off), f[wfirst + t]);
                put_sums(p);
            }
            if constexpr (D > 128) load_pv();
            __syncthreads();
        };
        if (wrow <= 64u) many(std::integral_constant<int, 1>{});
        else many(std::integral_constant<int, (MAX_SPLITS + MAX_WINDOW / WIN_TILE + 63) / 64>{});
    };
    if (splits > 1u) merge(std::true_type{}); else merge(std::false_type{});
    // out = (ysum @ Pi_v + wsum) / den, eight heads at a time as long as more than four are left, then four: eight are twice the work where a
    // row has four (at 256 3.4 us for 2.0), and every pass costs two barriers (all in fours / this, 4 rows x 6000 tokens, us: 64 wide, 16 heads
    // 18.8 / 18.1, 8 heads 13.5 / 13.2; 128 wide 25.6 / 25.1, 17.9 / 17.7)
    float *parts = reinterpret_cast<float *>(lds_lut);            // [part][RG][D]
    auto rotate_back = [&](auto heads, uint32_t g0) __attribute__((always_inline)) {
        constexpr int RG = decltype(heads)::value;
        static_assert(ROTP * RG * D * 4 <= 65536, "LDS area too small");
        float x[RG][4];
#pragma unroll
        for (int g = 0; g < RG; ++g)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[g][c] = 0.f;
        if (rp < (uint32_t)ROTP) {
#pragma unroll
            for (int k = 0; k < ROTK; k += 2)
#pragma unroll
                for (int g = 0; g < RG; ++g) {
                    // (heads past the last one: whatever lies there, not stored)
                    const float2 y = *reinterpret_cast<const float2 *>(ysum + (g0 + g) * D + rp * ROTK + k);
#pragma unroll
                    for (int c = 0; c < 4; ++c) x[g][c] = fmaf(y.y, __uint_as_float(pv[k + 1][c]), fmaf(y.x, __uint_as_float(pv[k][c]), x[g][c]));
                }
        }
        if (g0) __syncthreads();
        if (rp < (uint32_t)ROTP) {
#pragma unroll
            for (int g = 0; g < RG; ++g) *reinterpret_cast<float4 *>(parts + (rp * RG + g) * D + rc) = make_float4(x[g][0], x[g][1], x[g][2], x[g][3]);
        }
        __syncthreads();
        for (uint32_t p = tid; p < min((uint32_t)RG, G - g0) * D; p += DTHREADS) {
            const uint32_t g = p / D, j = p % D;
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < ROTP; ++q) v += parts[((uint32_t)q * RG + g) * D + j];
            v = (v + wsum[(g0 + g) * D + j]) / lds_den[g0 + g];
            TQ_GLOBAL uint16_t *o = (TQ_GLOBAL uint16_t *)a.out + ((size_t)row * G + g0 + g) * D + j;
            if (a.bf16) { const __bf16 h = (__bf16)v; *o = __builtin_bit_cast(uint16_t, h); }
            else { const _Float16 h = (_Float16)v; *o = __builtin_bit_cast(uint16_t, h); }
        }
    };
    uint32_t g0 = 0;
    if constexpr (C != 4)
        for (; G - g0 > 4u && g0 < G; g0 += 8u) rotate_back(std::integral_constant<int, 8>{}, g0);
    if (g0 < G) rotate_back(std::integral_constant<int, 4>{}, g0);
}

// STREAM (a.stream, see CACHE_STREAMED): the history read with the non-temporal hint.  What is used once then no longer drives out what every block of the next
// launch reads (tables, operands, code), and few rows start and merge sooner.  us a pass without / with it, 128 wide unless stated: 32 layers of
// 8 x 32768 tokens 669 / 635, 16 of 32 x 6000 at 64 276 / 264, 24 of 128 x 4182 642 / 620, 8 of 512 x 16384 1378 / 1355.  Norms, and 2-bit keys at 96 (six
// bytes a lane, in loads of two), are read without it.
// Keys of a byte a code at 256 (KEYS) are read without it too, and so they are at 128 for more than eight heads: a lane takes a line of theirs in several loads with
// other lines between, and what the hint lets go in the meantime is fetched again.  Time with the hint on keys and values / on values alone, over plain loads:
// 256 wide, K8/V4, 24 layers of 2 x 13512 tokens 1.044 / 0.957, 8 of 8 x 13512 1.021 / 0.941, 6 of 256 x 1140 1.066 / 0.992; 128 wide, K8/V4, 16 heads, 6 of
// 256 x 2256 1.036 / 0.967.  With two codes a byte at 256, and with a byte a code at 64 and 96, the keys gain by it as well: 256 wide, K4/V2, 6 of
// 32 x 18055 0.938 / 0.997, 8 of 128 x 1671 0.902 / 0.989; 64 wide, K8/V4, 16 heads, 6 of 256 x 4423 0.985 / 1.043.
template <int D, int IPBK, int IPBV, int C>
int launch_decode(dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    if (a.stream) hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, IPBV, C, true>), grid, dim3(DTHREADS), 0, s, a);
    else hipLaunchKernelGGL((tq_decode_kernel<D, IPBK, IPBV, C, false>), grid, dim3(DTHREADS), 0, s, a);
    return (int)hipGetLastError();
}
template <int D, int IPBK, int IPBV>
int launch_decode(dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    if constexpr (decode_run(D, IPBK, IPBV) == 64) {
        if (a.group <= 4u) return launch_decode<D, IPBK, IPBV, 4>(grid, s, a);
    }
    return a.group <= 8u ? launch_decode<D, IPBK, IPBV, 2>(grid, s, a) : launch_decode<D, IPBK, IPBV, 1>(grid, s, a);
}
template <int D, int IPBK>
int launch_decode(int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a) {
    switch (ipbv) {
        case 8:
            if constexpr (D == 128) return launch_decode<D, IPBK, 8>(grid, s, a);
            return TQ_ERR_BITS;
        case 4: return launch_decode<D, IPBK, 4>(grid, s, a);
        case 2: return launch_decode<D, IPBK, 2>(grid, s, a);
        default: return launch_decode<D, IPBK, 1>(grid, s, a);
    }
}

}  // namespace
