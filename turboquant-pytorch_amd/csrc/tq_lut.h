// What the kernels that attend to packed codes with blocks of 512 threads share: 16x16x32 matrix instructions, the decode tables
// spread over the banks of the LDS, reductions over the lanes of a wave.
#pragma once
#include "tq_device.h"

namespace {

typedef float tq_f4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ tq_f4v mfma16_f16(tq_u4 a, tq_u4 b, tq_f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(tq_half8, a), __builtin_bit_cast(tq_half8, b), c, 0, 0, 0);
}
__device__ __forceinline__ tq_f4v mfma16_bf16(tq_u4 a, tq_u4 b, tq_f4v c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(tq_bf8, a), __builtin_bit_cast(tq_bf8, b), c, 0, 0, 0);
}

// Over the lanes of a wave: within rows of 16 by rotation, then rows, then halves (no trip through the LDS as __shfl_xor takes).
template <typename Op>
__device__ __forceinline__ float reduce_rows(float x, Op op) {       // over the four lanes 16 apart
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return op(__uint_as_float(h[0]), __uint_as_float(h[1]));
}
template <typename Op>
__device__ __forceinline__ float reduce_wave(float x, Op op) {
    x = op(x, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x128, 0xf, 0xf, true)));
    x = op(x, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x124, 0xf, 0xf, true)));
    x = op(x, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x122, 0xf, 0xf, true)));
    x = op(x, __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x121, 0xf, 0xf, true)));
    return reduce_rows(x, op);
}
struct OpMax { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
struct OpAdd { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };

constexpr int LUT_THREADS = 512;     // threads of the block that stages the tables

// The byte -> centroids tables of keys and values, spread over the banks (RepLut), side by side: 256 rows of 256 bytes, the
// keys' entry in the first half of a row and the values' in the second.  The address of a lane's slot of an entry is then the byte,
// moved up by eight bits, with the lane's offset below it: one v_perm_b32, where 128-byte rows took two or three instructions (and
// v_dot4_u32_u8, one as well, is followed by idle cycles before its result can be used as an address).
// Eight consecutive threads write the 128 bytes of a table's half row, so the writes are free of conflicts; they read the same four entries
// with one or two loads (a load for each entry, eight of them a thread for keys and values, stood in front of the other loads of a
// block's start: 32 layers of 8 x 32768 tokens, K4/V2 628 -> 617 us, 16 of 32 x 6000 at 64 260 -> 258, 16 of 4 x 25627 266 -> 263).
template <int B, typename T>
__device__ __forceinline__ T lut_entry(const uint8_t *lut, uint32_t raw, uint32_t slot) {      // entry <byte B of raw>
    return *reinterpret_cast<const T *>(lut + __builtin_amdgcn_perm(raw, slot, 0x0c0c0000u | ((4u + B) << 8)));
}
template <int IPB>
struct Lut {
    static constexpr int ES = 2 * IPB, ROWS = 256 * 8 / LUT_THREADS;        // a thread has ROWS entries in a row, which it loads together
    static constexpr int WORDS = ROWS * ES / 4;
    static_assert(ROWS == 4, "entries of a thread");
    uint32_t v[WORDS];
    __device__ __forceinline__ void load(const uint8_t *src, uint32_t tid) {
        const uint8_t *g = src + (tid >> 3) * (ROWS * ES);
        if constexpr (WORDS == 2) { const tq_u2 x = tq_gload8(g); v[0] = x[0]; v[1] = x[1]; }
        else {
#pragma unroll
            for (int k = 0; k < WORDS; k += 4) {
                const tq_u4 x = tq_gload16(g + 4 * k);
                v[k] = x[0]; v[k + 1] = x[1]; v[k + 2] = x[2]; v[k + 3] = x[3];
            }
        }
    }
    __device__ __forceinline__ void store(uint8_t *lds, uint32_t tid) {
#pragma unroll
        for (int k = 0; k < ROWS; ++k) {
            tq_u4 x;
            if constexpr (ES == 2) { const uint32_t e = (v[k / 2] >> (16 * (k % 2))) & 0xffffu; x = tq_u4{e, e, e, e}; }
            else if constexpr (ES == 4) x = tq_u4{v[k], v[k], v[k], v[k]};
            else if constexpr (ES == 8) x = tq_u4{v[2 * k], v[2 * k + 1], v[2 * k], v[2 * k + 1]};
            else x = tq_u4{v[4 * k], v[4 * k + 1], v[4 * k + 2], v[4 * k + 3]};
            *reinterpret_cast<tq_u4 *>(lds + ((tid >> 3) * ROWS + k) * 256u + (tid & 7u) * 16u) = x;
        }
    }
};

// The eight coordinates of step s among a lane's key bytes -> fp16 operand.
template <int IPB, int NW>
__device__ __forceinline__ tq_u4 decode_keys(const uint32_t (&raw)[NW], int s, const uint8_t *lut, uint32_t slot) {
    tq_u4 out;
    if constexpr (IPB == 1) {
#pragma unroll
        for (int d = 0; d < 2; ++d) {
            const uint32_t r = raw[2 * s + d];
            out[2 * d] = (uint32_t)lut_entry<0, uint16_t>(lut, r, slot) | ((uint32_t)lut_entry<1, uint16_t>(lut, r, slot) << 16);
            out[2 * d + 1] = (uint32_t)lut_entry<2, uint16_t>(lut, r, slot) | ((uint32_t)lut_entry<3, uint16_t>(lut, r, slot) << 16);
        }
    } else if constexpr (IPB == 2) {
        out[0] = lut_entry<0, uint32_t>(lut, raw[s], slot);
        out[1] = lut_entry<1, uint32_t>(lut, raw[s], slot);
        out[2] = lut_entry<2, uint32_t>(lut, raw[s], slot);
        out[3] = lut_entry<3, uint32_t>(lut, raw[s], slot);
    } else if constexpr (IPB == 4) {
        const uint32_t r = raw[s / 2];
        const tq_u2 v0 = s % 2 ? lut_entry<2, tq_u2>(lut, r, slot) : lut_entry<0, tq_u2>(lut, r, slot);
        const tq_u2 v1 = s % 2 ? lut_entry<3, tq_u2>(lut, r, slot) : lut_entry<1, tq_u2>(lut, r, slot);
        out = tq_u4{v0[0], v0[1], v1[0], v1[1]};
    } else {
        const uint32_t r = raw[s / 4];
        out = s % 4 == 0 ? lut_entry<0, tq_u4>(lut, r, slot) : s % 4 == 1 ? lut_entry<1, tq_u4>(lut, r, slot) : s % 4 == 2 ? lut_entry<2, tq_u4>(lut, r, slot) : lut_entry<3, tq_u4>(lut, r, slot);
    }
    return out;
}

}  // namespace
