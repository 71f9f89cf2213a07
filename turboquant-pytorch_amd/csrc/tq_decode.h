// What tq_decode.hip (host side of the decode step) and the sources that instantiate its attention kernel share.
#pragma once
#include "tq_device.h"

struct TqDecodeArgs {
    const uint8_t *queries;          // [rows, group, D] 16-bit elements, contiguous
    const uint8_t *k_idx, *v_idx;
    const uint16_t *k_norms, *v_norms;
    const uint8_t *table_k, *table_v;
    const float *pi_v;               // [D, D] rotation of the value codec
    const uint8_t *k_win, *v_win;    // row r, token t at element r * win_stride + t * D
    float *partial;                  // [rows, splits, group, D + 2]: reference score, sum of exp, D sums in the rotated value space
    float *win_part;                 // [rows, window tiles, group, D + 2]: the same over 32 window tokens, sums in the plain space
    uint32_t *arrived;               // row r: [r * arrived_stride] blocks of the row that are done; zero before and after every launch (splits > 1)
    uint8_t *out;                    // [rows, group, D]
    long long win_stride;
    float scale;
    uint32_t tokens, packed_row_stride, group, chunk, n_win, bf16, arrived_stride, stream;
};

namespace {

constexpr int DW = 8;                // waves per block: one block per compute unit (two waves per SIMD), its waves share the tables
constexpr int DTHREADS = DW * TQ_WAVE;
constexpr int MAX_GROUP = 16;
constexpr int WIN_TILE = 32;
constexpr int MAX_WINDOW = 512;
constexpr int MAX_SPLITS = 256;     // (the merge keeps a weight per record and head in 32 KiB of LDS)
static_assert(MAX_GROUP * (MAX_SPLITS + MAX_WINDOW / WIN_TILE) * 4 <= 32768, "weights of the records");    // (both multiples of a batch)

}  // namespace

// Launches tq_decode_kernel for one head dimension (128: for 1- and 2-bit keys, and for wider ones); ipbk, ipbv = codes per byte.
int tq_decode_launch_d64(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a);
int tq_decode_launch_d96(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a);
int tq_decode_launch_d128_narrow(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a);
int tq_decode_launch_d128_wide(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a);
int tq_decode_launch_d256(int ipbk, int ipbv, dim3 grid, hipStream_t s, const TqDecodeArgs &a);
