// compress and decompress for the head dimensions 96, 160, 192 and 224 with 16-bit elements: the structure of the
// 256-wide kernels (csrc/tq_anydim.hip) with the dimension as a template argument.  Upstream
// turboquant/compressors_v3.py:37-43 builds rotation and codebook for whatever head_dim it is given; :46-81
// compress, :84-105 decompress.
//
// A block is D/32 waves that share tiles of 32 vectors; wave w keeps the rows [32w, 32w+32) of the rotation (compress:
// two 16-bit terms of Pi; decompress: the leading fp16 term of Pi^T) resident in registers as MFMA A operands for all
// D/16 steps of the contraction, so nothing of the table is read again after a block's first tile.  Tiles are fetched
// one ahead with coalesced loads, parked in a double-buffered LDS tile (one barrier per tile) and read back by every
// wave as B operands.  A row of such a tile is D*2 bytes, an odd multiple of 64: rows are rotated by their index
// (piece p of row v sits at position (p + v) mod D/8), which spreads the eight rows a 16-byte LDS access touches over all
// banks.  Same arithmetic, in the same order, as the run-time-dimension kernels: a vector gets the same bytes whichever
// of the two compresses it (fp32 elements go there).  The RAGGED instantiations take a head dimension dl that is not a
// multiple of 32 as the next multiple D, the way the run-time-dimension kernels do: the table holds the rotation extended
// by zeros, elements a vector does not have are staged as zeros, coordinates it does not have get the code 0 and are
// neither decoded nor stored; whole 16-byte pieces at aligned addresses take the wide loads and stores, the rest moves
// element by element.
// One source file per dimension instantiates them (tq_wide_d96.hip ... tq_wide_d224.hip), so that they compile side by side.
#pragma once
#include <mutex>
#include <type_traits>

#include "tq_wide.h"

namespace {

template <int D>
struct Wide {
    static_assert(D % 32 == 0 && D > 64 && D < 256 && D != 128, "96, 160, 192, 224");
    static constexpr int WAVES = D / 32, THREADS = 64 * WAVES, STEPS = D / 16, PIECES = D / 8;
    static constexpr int ROW = D * 2, TILE_BYTES = 32 * ROW;
    // waves per SIMD the compress kernel is compiled for: three (168 registers) at 96, where a compute unit's LDS holds
    // four blocks of three waves; from 160 on the resident rotation takes D/2 registers and the kernel 228 to 256 (held
    // to 168 it spills 60 to 80 of them and runs at half the rate), so one block of D/32 waves is resident per unit
    static constexpr int COMPRESS_WAVES_PER_SIMD = D == 96 ? 3 : 2;
    // compress: quantiser grid | two tiles | per-piece sums of squares of three tiles
    static constexpr uint32_t COMPRESS_LDS = TQ_GRID_LDS_BYTES + 2 * TILE_BYTES + 3 * 32 * PIECES * 4;
    // decompress: byte -> centroids table | two tiles of centroids | output tile | norms of two tiles
    // waves per SIMD the restore of a layer is compiled for: as many as the per-tensor kernel has.  Left alone its bodies and the piece
    // of the window took 136 registers at 224, where a block is seven waves and one instead of two were resident (8 x 16384 tokens, K4/V2, no
    // window: per tensor 41 us, 44.5 that way, 40.0 this way), and four waves instead of five at 96
    static constexpr int RESTORE_WAVES_PER_SIMD = D == 96 ? 5 : 4;
    static constexpr uint32_t DECOMPRESS_LDS = 4096 + 3 * TILE_BYTES + 2 * 32 * 4;
};

// How a head dimension dl fills the D coordinates worked on
enum Fit {
    FULL,       // dl == D
    CHUNKS,     // dl < D in chunks of 16 coordinates, rows, vectors and packed bytes aligned for their pieces: a lane's pieces and codes are
                // all there or all missing, and every load is one unconditional load of a clamped address
    ELEMENTS    // dl < D, anything else: element by element and byte by byte where a piece is not whole or not aligned
};
// CHUNKS for this job?  (The loads of ELEMENTS sit behind conditions, where the compiler waits for one before it writes the zeros of the
// other lanes, so nothing is in flight while a tile is worked on: 32 rows x 5873 tokens at 80, 4-bit, keys and values, compress / decompress
// 40 / 27 us that way, 31 / 23 us this way, 28.6 / 21.9 us with TqTileWalk instead of a division an address, 26.5 /
// 21.1 us since that looks for whole tiles first.)
__device__ __forceinline__ bool in_chunks(const TqDevJob &job, uint32_t dl, uint32_t packed_bytes) {
    return dl % 16u == 0u && (((uintptr_t)job.states | (uintptr_t)job.row_stride | (uintptr_t)job.token_stride) & 15u) == 0u &&
           ((uintptr_t)job.idx_bytes & (uintptr_t)(packed_bytes - 1u)) == 0u;
}

// position of piece p in row v of a tile
template <int D>
__device__ __forceinline__ uint32_t rotated_piece(uint32_t p, uint32_t v) {
    return (p + v) % (uint32_t)Wide<D>::PIECES;
}

template <int DTYPE, int BITS, int D, int FIT>
__device__ __forceinline__ void wide_compress_tiles(const TqDevJob &job, TqBlock blk, uint32_t dl, uint8_t *lds) {
    static_assert(DTYPE == TQ_F16 || DTYPE == TQ_BF16, "16-bit inputs");
    using W = Wide<D>;
    constexpr int STEPS = W::STEPS, PIECES = W::PIECES, ROW = W::ROW, THREADS = W::THREADS;
    constexpr int IPB = 8 / BITS, NB = 16 / IPB, NW = NB < 4 ? 1 : NB / 4;
    constexpr int CPS = (16 + STEPS - 1) / STEPS;      // coordinates searched per step of the contraction

    uint8_t *lds_grid = lds;                                                        // single copy, bases unshifted
    uint8_t (*lds_stage)[W::TILE_BYTES] = reinterpret_cast<uint8_t (*)[W::TILE_BYTES]>(lds + TQ_GRID_LDS_BYTES);
    float (*lds_part)[32][PIECES] = reinterpret_cast<float (*)[32][PIECES]>(lds + TQ_GRID_LDS_BYTES + 2 * W::TILE_BYTES);   // [3]

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = tq_uniform32(tid >> 6);
    const uint32_t n = lane & 31u, hk = lane >> 5;
    const uint32_t n_tiles = (job.n_vec + 31u) / 32u;
    if (blk.x >= n_tiles) return;        // also: an empty job of a batch, whose table may be NULL
    const TqTableHeader *hd = reinterpret_cast<const TqTableHeader *>(job.table);

    // loads of a tile: piece i = l * THREADS + tid of the tile's 32 * PIECES is piece i % PIECES of vector i / PIECES;
    // vectors past the end read the tile's first piece (never stored)
    uint32_t ld_vec[2], ld_piece[2];
#pragma unroll
    for (int l = 0; l < 2; ++l) {
        const uint32_t i = l * THREADS + tid;
        ld_vec[l] = i / PIECES;
        ld_piece[l] = i % PIECES;
    }
    long long ld_own[2];
#pragma unroll
    for (int l = 0; l < 2; ++l) ld_own[l] = (long long)ld_vec[l] * job.token_stride + (FIT != CHUNKS || ld_piece[l] * 8u < dl ? ld_piece[l] * 16u : 0u);
    tq_u4 pre[2];
    auto issue_loads = [&](const TqTileWalk &t) {
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            const uint8_t *piece = job.states + t.offset(job, ld_vec[l], ld_own[l]);
            if constexpr (FIT == ELEMENTS) {
                const uint32_t e0 = t.v + ld_vec[l] < job.n_vec ? ld_piece[l] * 8u : 0u;
                const TQ_GLOBAL uint8_t *src = (const TQ_GLOBAL uint8_t *)piece - 2u * e0;
                if (e0 + 8u <= dl && (((uintptr_t)src + 2u * e0) & 15u) == 0u) {      // a whole piece at an aligned address
                    pre[l] = *reinterpret_cast<const TQ_GLOBAL tq_u4 *>(src + 2u * e0);
                } else {                                                              // element by element; past the end: zero
                    tq_u4 q = {0u, 0u, 0u, 0u};
#pragma unroll
                    for (uint32_t k = 0; k < 8u; ++k)
                        if (e0 + k < dl) q[k / 2] |= (uint32_t)*reinterpret_cast<const TQ_GLOBAL uint16_t *>(src + 2u * (e0 + k)) << (16 * (k & 1));
                    pre[l] = q;
                }
            } else {
                pre[l] = tq_gload16(piece);
            }
        }
    };
    TqTileWalk ahead(job, blk.x, blk.grid), done = ahead;      // of the tile fetched next, of the tile searched next
    issue_loads(ahead);

    tq_u4 areg[2][STEPS];
    {
        const uint8_t *src = job.table + (DTYPE == TQ_F16 ? TQ_OFF_A_F16 : TQ_OFF_A_BF16(D));
#pragma unroll
        for (int term = 0; term < 2; ++term)
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                areg[term][s] = tq_gload16(src + (size_t)term * TQ_OPERAND_BYTES_FOR(D) + (((size_t)wave * STEPS + s) * 64 + lane) * 16);
    }
    tq_stage_in_lds<TQ_GRID_LDS_BYTES, THREADS>(lds_grid, job.table + TQ_OFF_GRID(D), tid);
    const float grid_scale = hd->grid_scale, grid_bias = hd->grid_bias;

    // park the prefetched tile in buffer b and leave the pieces' sums of squares in slot `slot`
    uint32_t park_off[2];
#pragma unroll
    for (int l = 0; l < 2; ++l) park_off[l] = ld_vec[l] * ROW + (rotated_piece<D>(ld_piece[l], ld_vec[l]) << 4);
    auto park = [&](uint32_t b, uint32_t slot) {
#pragma unroll
        for (int l = 0; l < 2; ++l) {
            if (FIT == CHUNKS && ld_piece[l] * 8u >= dl) pre[l] = tq_u4{0u, 0u, 0u, 0u};
            *reinterpret_cast<tq_u4 *>(lds_stage[b] + park_off[l]) = pre[l];
            lds_part[slot][ld_vec[l]][ld_piece[l]] = sumsq8<DTYPE>(pre[l], 0.f);
        }
    };
    // B operand of step s: piece 2 s + hk of row n
    uint32_t op_off[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) op_off[s] = n * ROW + (rotated_piece<D>(2u * s + hk, n) << 4);
    const uint32_t g_bytes = FIT != FULL ? (dl + IPB - 1u) / IPB : (uint32_t)(D / IPB);      // packed bytes per vector

    // iteration j: rotate tile j into acc_new, search tile j-1 from acc_old
    auto iteration = [&](auto rot_tag, auto search_tag, uint32_t j, tq_f16v &acc_new, const tq_f16v &acc_old) {
        constexpr bool ROT = decltype(rot_tag)::value, SEARCH = decltype(search_tag)::value;
        const uint8_t *stage = lds_stage[j & 1u];
        float nrm = 0.f, inv = 0.f, inv_cell = 0.f;
        if constexpr (SEARCH) {
            // pieces added in index order, as the run-time-dimension kernel adds them: tile j-1 sits in slot (j-1) % 3
            const float4 *pp = reinterpret_cast<const float4 *>(&lds_part[(j + 2u) % 3u][n][0]);
            float ss = 0.f;
#pragma unroll
            for (int q = 0; q < PIECES / 4; ++q) {
                const float4 f = pp[q];
                ss += f.x; ss += f.y; ss += f.z; ss += f.w;
            }
            nrm = tq_norm_from_sumsq(ss);
            inv = __builtin_amdgcn_rcpf(nrm + 1e-8f);
            if (DTYPE == TQ_F16) inv *= 1.0f / (float)(1 << TQ_F16_PI_SHIFT);
            inv_cell = inv * grid_scale;
        }
        if constexpr (ROT) acc_new = tq_zero16();
        uint32_t words[NW];
#pragma unroll
        for (int w = 0; w < NW; ++w) words[w] = 0u;
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            if constexpr (ROT) {
                const tq_u4 bop = *reinterpret_cast<const tq_u4 *>(stage + op_off[s]);
                acc_new = (DTYPE == TQ_F16) ? mfma_f16(areg[0][s], bop, acc_new) : mfma_bf16(areg[0][s], bop, acc_new);
                acc_new = (DTYPE == TQ_F16) ? mfma_f16(areg[1][s], bop, acc_new) : mfma_bf16(areg[1][s], bop, acc_new);
            }
            if constexpr (SEARCH) {     // coordinates 32 w + 16 hk + c of vector n, CPS of them behind every step
#pragma unroll
                for (int c = s * CPS; c < (s + 1) * CPS && c < 16; ++c) {
                    const float a = acc_old[c];
                    const uint32_t addr = __float_as_uint(fmaf(a, inv_cell, grid_bias)) & TQ_GRID_ADDR_MASK;
                    const tq_u2 cell = *reinterpret_cast<const tq_u2 *>(lds_grid + addr);
                    const float t = fmaf(a, inv, -__uint_as_float(cell[0]));
                    uint32_t code = cell[1] + (~__float_as_uint(t) >> 31);                // base + !(rho < threshold)
                    if constexpr (FIT == ELEMENTS) code = 32u * wave + 16u * hk + (uint32_t)c < dl ? code : 0u;
                    const int byte = c / IPB, k = c % IPB;                                // most significant code of a byte first
                    words[byte / 4] |= code << (8 * (byte % 4) + BITS * (IPB - 1 - k));
                }
            }
            if (s % 2 == 1) __builtin_amdgcn_sched_barrier(0);      // keep the steps in this order (register pressure)
        }
        if constexpr (SEARCH) {
            if (done.v + n < job.n_vec && (FIT != CHUNKS || 32u * wave + 16u * hk < dl)) {
                const uint32_t slot = done.slot(job, n);
                uint8_t *dst = job.idx_bytes + (size_t)slot * g_bytes + (2u * wave + hk) * NB;
                bool bytewise = false;
                if constexpr (FIT == ELEMENTS) bytewise = (2u * wave + hk) * NB + NB > g_bytes || ((uintptr_t)dst & (uintptr_t)(NB - 1));
                if (bytewise) {
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        if ((2u * wave + hk) * NB + (uint32_t)b < g_bytes)
                            *((TQ_GLOBAL uint8_t *)dst + b) = (uint8_t)(words[b / 4] >> (8 * (b % 4)));
                } else if constexpr (NB == 2) tq_gstore2(reinterpret_cast<uint16_t *>(dst), (uint16_t)words[0]);
                else if constexpr (NB == 4) *reinterpret_cast<TQ_GLOBAL uint32_t *>((TQ_GLOBAL uint8_t *)dst) = words[0];
                else if constexpr (NB == 8) { const tq_u2 o = {words[0], words[1]}; tq_gstore8(dst, o); }
                else { const tq_u4 o = {words[0], words[1], words[2], words[3]}; tq_gstore16(dst, o); }
                if (wave == 0u && hk == 0u) {
                    const _Float16 hn = (_Float16)nrm;
                    tq_gstore2(job.vec_norms + slot, __builtin_bit_cast(uint16_t, hn));
                }
            }
            done.next(job);
        }
    };

    const uint32_t m = (n_tiles - blk.x + blk.grid - 1u) / blk.grid;     // this block's tiles
    // one trip: the tile after this one sets out while this one is rotated, and is parked behind the trip's work
    auto trip = [&](auto rot_tag, auto search_tag, uint32_t j, tq_f16v &acc_new, const tq_f16v &acc_old) {
        const bool more = j + 1u < m;
        if (more) {
            ahead.next(job);
            issue_loads(ahead);
        }
        __syncthreads();        // tile j and its sums are parked, and nobody reads buffer (j + 1) & 1 any more
        iteration(rot_tag, search_tag, j, acc_new, acc_old);
        if (more) park((j + 1u) & 1u, (j + 1u) % 3u);
    };
    using T = std::true_type;
    using F = std::false_type;
    park(0u, 0u);
    tq_f16v acc_a, acc_b;       // tiles with an even index rotate into acc_a, the others into acc_b
    trip(T{}, F{}, 0u, acc_a, acc_a);
    uint32_t j = 1;
    for (; j + 1u < m; j += 2u) {
        trip(T{}, T{}, j, acc_b, acc_a);
        trip(T{}, T{}, j + 1u, acc_a, acc_b);
    }
    if (j < m) {
        trip(T{}, T{}, j, acc_b, acc_a);
        ++j;
    }
    if (m & 1u) trip(F{}, T{}, m, acc_b, acc_a);        // the last tile's codes
    else trip(F{}, T{}, m, acc_a, acc_b);
}

template <int DTYPE, int BITS, int D, bool RAGGED>
__device__ __forceinline__ void wide_compress_job(const TqDevJob &job, TqBlock blk, uint32_t dl, uint8_t *lds) {
    if constexpr (!RAGGED) wide_compress_tiles<DTYPE, BITS, D, FULL>(job, blk, dl, lds);
    else if (in_chunks(job, dl, 16 / (8 / BITS))) wide_compress_tiles<DTYPE, BITS, D, CHUNKS>(job, blk, dl, lds);
    else wide_compress_tiles<DTYPE, BITS, D, ELEMENTS>(job, blk, dl, lds);
}

template <int DTYPE, int BITS, int D, bool RAGGED>
__global__ __launch_bounds__(Wide<D>::THREADS, Wide<D>::COMPRESS_WAVES_PER_SIMD) void tq_wide_compress_kernel(TqDevJob job0, const tq_job *jobs, uint32_t dl) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    wide_compress_job<DTYPE, BITS, D, RAGGED>(tq_uniform_job(tq_load_job(job0, jobs, blockIdx.y, 2)), TqBlock{blockIdx.x, gridDim.x}, dl, lds);
}

// keys and values of a layer
template <int DTYPE, int D, bool RAGGED>
__global__ __launch_bounds__(Wide<D>::THREADS, Wide<D>::COMPRESS_WAVES_PER_SIMD) void tq_wide_compress_layer_kernel(TqLayer l, uint32_t dl) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t which = tq_layer_job(l);
    const TqDevJob job = tq_uniform_job(which ? l.job[1] : l.job[0]);
    const TqBlock blk = tq_layer_block(l, which);
    switch (which ? l.bits[1] : l.bits[0]) {
        case 1: wide_compress_job<DTYPE, 1, D, RAGGED>(job, blk, dl, lds); break;
        case 2: wide_compress_job<DTYPE, 2, D, RAGGED>(job, blk, dl, lds); break;
        case 3: wide_compress_job<DTYPE, 3, D, RAGGED>(job, blk, dl, lds); break;
        case 4: wide_compress_job<DTYPE, 4, D, RAGGED>(job, blk, dl, lds); break;
        default: wide_compress_job<DTYPE, 8, D, RAGGED>(job, blk, dl, lds); break;
    }
}

// decompress: wave w keeps the rows [32w, 32w+32) of Pi^T (leading fp16 term).  The packed bytes of a tile are fetched
// one tile ahead (every thread the bytes of 16 codes), turned into fp16 centroids through the byte -> centroids table and
// parked in a double-buffered LDS tile that all waves read as B operands; the scaled, rounded results go through a
// second LDS tile so that the stores are D*2 contiguous bytes per vector.
template <int DTYPE, int IPB, int D, int FIT>
__device__ __forceinline__ void wide_decompress_tiles(const TqDevJob &job, TqBlock blk, uint32_t dl, uint8_t *lds) {
    static_assert(DTYPE == TQ_F16 || DTYPE == TQ_BF16, "16-bit outputs");
    using W = Wide<D>;
    constexpr int STEPS = W::STEPS, PIECES = W::PIECES, ROW = W::ROW, THREADS = W::THREADS, WAVES = W::WAVES;
    constexpr int ENTRY = 2 * IPB;                 // bytes of a table entry: the fp16 centroids of one packed byte
    constexpr int RAW = 16 / IPB;                  // packed bytes of a thread's 16 codes: 2, 4, 8, 16

    uint8_t *lds_lut = lds;
    uint8_t (*lds_y)[W::TILE_BYTES] = reinterpret_cast<uint8_t (*)[W::TILE_BYTES]>(lds + 4096);
    uint8_t *lds_out = lds + 4096 + 2 * W::TILE_BYTES;
    float (*lds_norm)[32] = reinterpret_cast<float (*)[32]>(lds + 4096 + 3 * W::TILE_BYTES);       // [2][32]

    uint8_t *out_base = const_cast<uint8_t *>(job.states);
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = tq_uniform32(tid >> 6);
    const uint32_t n = lane & 31u, hk = lane >> 5;
    const uint32_t n_tiles = (job.n_vec + 31u) / 32u;
    if (blk.x >= n_tiles) return;
    const uint32_t g_bytes = FIT != FULL ? (dl + IPB - 1u) / IPB : (uint32_t)(D / IPB);      // packed bytes per vector in memory

    // a thread's share of a tile: codes [16 c, 16 c + 16) of vector dv, c = tid % (2 WAVES)
    const uint32_t dv = tid / (2u * WAVES), chunk = tid % (2u * WAVES);
    uint32_t raw[4] = {0u, 0u, 0u, 0u};
    uint16_t norm_bits = 0;
    auto issue_loads = [&](const TqTileWalk &t) {
        const uint32_t slot = t.slot(job, dv);
        const uint8_t *src = job.idx_bytes + (size_t)slot * g_bytes + (FIT != CHUNKS || 16u * chunk < dl ? chunk * RAW : 0u);
        bool bytewise = false;
        if constexpr (FIT == ELEMENTS) bytewise = chunk * RAW + RAW > g_bytes || ((uintptr_t)src & (uintptr_t)(RAW - 1));
        if (bytewise) {     // byte by byte; past the vector's last byte: zero (never decoded)
#pragma unroll
            for (int q = 0; q < 4; ++q) raw[q] = 0u;
#pragma unroll
            for (int b = 0; b < RAW; ++b)
                if (chunk * RAW + (uint32_t)b < g_bytes) raw[b / 4] |= (uint32_t)*((const TQ_GLOBAL uint8_t *)src + b) << (8 * (b % 4));
        } else if constexpr (RAW == 2) raw[0] = tq_gload2(reinterpret_cast<const uint16_t *>(src));
        else if constexpr (RAW == 4) raw[0] = *reinterpret_cast<const TQ_GLOBAL uint32_t *>((const TQ_GLOBAL uint8_t *)src);
        else if constexpr (RAW == 8) { const tq_u2 t = tq_gload8(src); raw[0] = t[0]; raw[1] = t[1]; }
        else { const tq_u4 t = tq_gload16(src); raw[0] = t[0]; raw[1] = t[1]; raw[2] = t[2]; raw[3] = t[3]; }
        if (chunk == 0u) norm_bits = tq_gload2(job.vec_norms + slot);
    };
    TqTileWalk ahead(job, blk.x, blk.grid), here = ahead;      // of the tile fetched next, of the tile stored
    issue_loads(ahead);

    tq_u4 areg[STEPS];
    {
        const uint8_t *src = job.table + TQ_OFF_AT_F16(D);
#pragma unroll
        for (int s = 0; s < STEPS; ++s) areg[s] = tq_gload16(src + (((size_t)wave * STEPS + s) * 64 + lane) * 16);
    }
    tq_stage_in_lds<256 * ENTRY, THREADS>(lds_lut, job.table + TQ_OFF_LUT(D), tid);
    __syncthreads();

    // the prefetched bytes -> 16 fp16 centroids = pieces 2 chunk, 2 chunk + 1 of row dv of buffer b.  In this tile the even
    // pieces of a row come first and the odd ones after them (piece 2 c + q at index q * PIECES/2 + c, then rotated by the
    // row like everywhere else): the threads that decode a row write neighbouring bank groups at a time instead of every
    // second one.
    const uint32_t y_off[2] = {dv * ROW + (rotated_piece<D>(chunk, dv) << 4), dv * ROW + (rotated_piece<D>(PIECES / 2 + chunk, dv) << 4)};
    auto decode = [&](uint32_t b) {
        uint32_t h[8];          // 16 halves
#pragma unroll
        for (int byte = 0; byte < RAW; ++byte) {
            const uint32_t v = (raw[byte / 4] >> (8 * (byte % 4))) & 0xffu;
            const uint8_t *e = lds_lut + v * ENTRY;
            if constexpr (IPB == 1) {
                const uint32_t c = *reinterpret_cast<const uint16_t *>(e);
                if (byte & 1) h[byte / 2] |= c << 16; else h[byte / 2] = c;
            } else if constexpr (IPB == 2) {
                h[byte] = *reinterpret_cast<const uint32_t *>(e);
            } else if constexpr (IPB == 4) {
                const tq_u2 c = *reinterpret_cast<const tq_u2 *>(e);
                h[2 * byte] = c[0]; h[2 * byte + 1] = c[1];
            } else {
                const tq_u4 c = *reinterpret_cast<const tq_u4 *>(e);
                h[4 * byte] = c[0]; h[4 * byte + 1] = c[1]; h[4 * byte + 2] = c[2]; h[4 * byte + 3] = c[3];
            }
        }
        if constexpr (FIT == ELEMENTS) {     // coordinates the vector does not have contribute nothing (CHUNKS: their operands are zero, the centroids finite)
#pragma unroll
            for (int k = 0; k < 16; ++k)
                if (16u * chunk + (uint32_t)k >= dl) h[k / 2] &= (k & 1) ? 0x0000ffffu : 0xffff0000u;
        }
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const tq_u4 o = {h[4 * q], h[4 * q + 1], h[4 * q + 2], h[4 * q + 3]};
            *reinterpret_cast<tq_u4 *>(lds_y[b] + y_off[q]) = o;
        }
        if (chunk == 0u) lds_norm[b][dv] = (float)__builtin_bit_cast(_Float16, norm_bits);
    };
    uint32_t op_off[STEPS];     // B operand of step s: piece 2 s + hk of row n, at index hk * PIECES/2 + s
#pragma unroll
    for (int s = 0; s < STEPS; ++s) op_off[s] = n * ROW + (rotated_piece<D>(hk * (PIECES / 2) + s, n) << 4);
    // lane (n, hk) ends up with elements 32 w + 16 hk + r of vector n: pieces 4 w + 2 hk + c of its output row
    const uint32_t out_off[2] = {n * ROW + (rotated_piece<D>(4u * wave + 2u * hk, n) << 4), n * ROW + (rotated_piece<D>(4u * wave + 2u * hk + 1u, n) << 4)};
    // the stores of a tile: piece i = k * THREADS + tid is piece i % PIECES of vector i / PIECES
    uint32_t st_vec[2], st_piece[2], st_off[2];
    long long st_own[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t i = k * THREADS + tid;
        st_vec[k] = i / PIECES;
        st_piece[k] = i % PIECES;
        st_own[k] = (long long)st_vec[k] * job.token_stride + st_piece[k] * 16u;
        st_off[k] = st_vec[k] * ROW + (rotated_piece<D>(st_piece[k], st_vec[k]) << 4);
    }

    const uint32_t m = (n_tiles - blk.x + blk.grid - 1u) / blk.grid;
    decode(0u);
    for (uint32_t j = 0; j < m; ++j) {
        if (j + 1u < m) {
            ahead.next(job);
            issue_loads(ahead);
        }
        __syncthreads();        // tile j is decoded; the output tile of the last iteration has been read
        const uint8_t *ys = lds_y[j & 1u];
        tq_f16v acc = tq_zero16();
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const tq_u4 b = *reinterpret_cast<const tq_u4 *>(ys + op_off[s]);
            acc = mfma_f16(areg[s], b, acc);
        }
        const float nrm = lds_norm[j & 1u][n];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            tq_u4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float x0 = acc[8 * c + 2 * e] * nrm, x1 = acc[8 * c + 2 * e + 1] * nrm;
                if constexpr (DTYPE == TQ_F16) {
                    const tq_half2 hh = {(_Float16)x0, (_Float16)x1};
                    o[e] = __builtin_bit_cast(uint32_t, hh);
                } else {
                    const tq_bf2 hh = {(__bf16)x0, (__bf16)x1};
                    o[e] = __builtin_bit_cast(uint32_t, hh);
                }
            }
            *reinterpret_cast<tq_u4 *>(lds_out + out_off[c]) = o;
        }
        __syncthreads();        // the output tile is complete
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const tq_u4 val = *reinterpret_cast<const tq_u4 *>(lds_out + st_off[k]);
            if (here.v + st_vec[k] >= job.n_vec) continue;
            uint8_t *dst = out_base + here.offset(job, st_vec[k], st_own[k]);
            if constexpr (FIT != FULL) {
                const uint32_t e0 = st_piece[k] * 8u;
                if (e0 >= dl) continue;
                if (FIT == ELEMENTS && (e0 + 8u > dl || ((uintptr_t)dst & 15u))) {       // element by element
#pragma unroll
                    for (uint32_t e = 0; e < 8u; ++e)
                        if (e0 + e < dl) *reinterpret_cast<TQ_GLOBAL uint16_t *>((TQ_GLOBAL uint8_t *)dst + 2u * e) = (uint16_t)(val[e / 2] >> (16 * (e & 1)));
                    continue;
                }
            }
            tq_gstore16_stream(dst, val);
        }
        here.next(job);
        if (j + 1u < m) decode((j + 1u) & 1u);
    }
}

template <int DTYPE, int IPB, int D, bool RAGGED>
__device__ __forceinline__ void wide_decompress_job(const TqDevJob &job, TqBlock blk, uint32_t dl, uint8_t *lds) {
    if constexpr (!RAGGED) wide_decompress_tiles<DTYPE, IPB, D, FULL>(job, blk, dl, lds);
    else if (in_chunks(job, dl, 16 / IPB)) wide_decompress_tiles<DTYPE, IPB, D, CHUNKS>(job, blk, dl, lds);
    else wide_decompress_tiles<DTYPE, IPB, D, ELEMENTS>(job, blk, dl, lds);
}

template <int DTYPE, int IPB, int D, bool RAGGED>
__global__ __launch_bounds__(Wide<D>::THREADS) void tq_wide_decompress_kernel(TqDevJob job0, const tq_job *jobs, uint32_t dl) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    wide_decompress_job<DTYPE, IPB, D, RAGGED>(tq_uniform_job(tq_load_job(job0, jobs, blockIdx.y, 2)), TqBlock{blockIdx.x, gridDim.x}, dl, lds);
}

// keys and values of a layer and its window
template <int DTYPE, int D, bool RAGGED>
__global__ __launch_bounds__(Wide<D>::THREADS, Wide<D>::RESTORE_WAVES_PER_SIMD) void tq_wide_restore_layer_kernel(TqLayer l, TqWindowCopy window, uint32_t dl) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t which = tq_layer_job(l);
    const TqDevJob job = tq_uniform_job(which ? l.job[1] : l.job[0]);
    const TqBlock blk = tq_layer_block(l, which);
    tq_with_window(window, [&]() __attribute__((always_inline)) {
        switch (8 / (which ? l.bits[1] : l.bits[0])) {
            case 8: wide_decompress_job<DTYPE, 8, D, RAGGED>(job, blk, dl, lds); break;
            case 4: wide_decompress_job<DTYPE, 4, D, RAGGED>(job, blk, dl, lds); break;
            case 2: wide_decompress_job<DTYPE, 2, D, RAGGED>(job, blk, dl, lds); break;
            default: wide_decompress_job<DTYPE, 1, D, RAGGED>(job, blk, dl, lds); break;
        }
    });
}

// ---- host side --------------------------------------------------------------------------

constexpr int MAX_DEVICES = 64;
std::mutex host_state_mutex;

// Blocks of `threads` threads with `lds` bytes of dynamic LDS that the current device holds at once (what the runtime says fits a
// compute unit, remembered per device in `slots`, the kernel's own); raises the kernel's LDS limit.
template <typename K>
int resident_blocks(K kernel, int (&slots)[MAX_DEVICES], uint32_t lds, uint32_t threads, int &resident) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES) return TQ_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lock(host_state_mutex);
    if (slots[dev] == 0) {
        e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
        int cus = 0, per_cu = 0;
        e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return (int)e;
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, (int)threads, lds);
        if (e != hipSuccess) return (int)e;
        slots[dev] = (cus > 0 ? cus : 1) * (per_cu > 0 ? per_cu : 1);
    }
    resident = slots[dev];
    return 0;
}

template <typename K>
int launch(K kernel, int (&slots)[MAX_DEVICES], uint32_t lds, uint32_t threads, const TqDevJob &job, const tq_job *jobs_dev,
           int n_jobs, uint32_t max_vec, uint32_t dl, hipStream_t stream) {
    int resident = 0;
    const int rc = resident_blocks(kernel, slots, lds, threads, resident);
    if (rc) return rc;
    const uint32_t tiles = (max_vec + 31u) / 32u;
    const uint32_t bx = tq_blocks_per_job(tiles, resident, n_jobs);
    hipLaunchKernelGGL(kernel, dim3(bx, (unsigned)n_jobs, 1), dim3(threads, 1, 1), lds, stream, job, jobs_dev, dl);
    return (int)hipGetLastError();
}

template <int DTYPE, int D, bool RAGGED>
int launch_compress_layer(TqLayer &l, uint32_t n_vec, uint32_t dl, hipStream_t s) {
    static int slots[MAX_DEVICES] = {};
    int resident = 0;
    const int rc = resident_blocks(&tq_wide_compress_layer_kernel<DTYPE, D, RAGGED>, slots, Wide<D>::COMPRESS_LDS, Wide<D>::THREADS, resident);
    if (rc) return rc;
    const uint32_t blocks = tq_layer_blocks(l, (n_vec + 31u) / 32u, (uint32_t)resident);
    hipLaunchKernelGGL((tq_wide_compress_layer_kernel<DTYPE, D, RAGGED>), dim3(blocks), dim3(Wide<D>::THREADS), Wide<D>::COMPRESS_LDS, s, l, dl);
    return (int)hipGetLastError();
}
template <int DTYPE, int D, bool RAGGED>
int launch_restore_layer(TqLayer &l, const TqWindowCopy &w, uint32_t n_vec, uint32_t dl, hipStream_t s) {
    static int slots[MAX_DEVICES] = {};
    int resident = 0;
    const int rc = resident_blocks(&tq_wide_restore_layer_kernel<DTYPE, D, RAGGED>, slots, Wide<D>::DECOMPRESS_LDS, Wide<D>::THREADS, resident);
    if (rc) return rc;
    const uint32_t blocks = tq_layer_blocks(l, (n_vec + 31u) / 32u, (uint32_t)resident);
    hipLaunchKernelGGL((tq_wide_restore_layer_kernel<DTYPE, D, RAGGED>), dim3(blocks), dim3(Wide<D>::THREADS), Wide<D>::DECOMPRESS_LDS, s, l, w, dl);
    return (int)hipGetLastError();
}
template <int DTYPE, int BITS, int D>
int launch_compress(const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec, uint32_t dl, hipStream_t s) {
    if (dl != (uint32_t)D) {
        static int slots_ragged[MAX_DEVICES] = {};
        return launch(&tq_wide_compress_kernel<DTYPE, BITS, D, true>, slots_ragged, Wide<D>::COMPRESS_LDS, Wide<D>::THREADS, job, jobs_dev, n_jobs, max_vec, dl, s);
    }
    static int slots[MAX_DEVICES] = {};
    return launch(&tq_wide_compress_kernel<DTYPE, BITS, D, false>, slots, Wide<D>::COMPRESS_LDS, Wide<D>::THREADS, job, jobs_dev, n_jobs, max_vec, dl, s);
}
template <int DTYPE, int D>
int compress_bits(int bits, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec, uint32_t dl, hipStream_t s) {
    switch (bits) {
        case 1: return launch_compress<DTYPE, 1, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 2: return launch_compress<DTYPE, 2, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 3: return launch_compress<DTYPE, 3, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 4: return launch_compress<DTYPE, 4, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 5: case 6: case 7: case 8:  // one code per byte: identical packing
            return launch_compress<DTYPE, 8, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        default: return TQ_ERR_BITS;
    }
}
template <int DTYPE, int IPB, int D>
int launch_decompress(const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec, uint32_t dl, hipStream_t s) {
    if (dl != (uint32_t)D) {
        static int slots_ragged[MAX_DEVICES] = {};
        return launch(&tq_wide_decompress_kernel<DTYPE, IPB, D, true>, slots_ragged, Wide<D>::DECOMPRESS_LDS, Wide<D>::THREADS, job, jobs_dev, n_jobs, max_vec, dl, s);
    }
    static int slots[MAX_DEVICES] = {};
    return launch(&tq_wide_decompress_kernel<DTYPE, IPB, D, false>, slots, Wide<D>::DECOMPRESS_LDS, Wide<D>::THREADS, job, jobs_dev, n_jobs, max_vec, dl, s);
}
template <int DTYPE, int D>
int decompress_bits(int bits, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec, uint32_t dl, hipStream_t s) {
    switch (8 / bits) {
        case 8: return launch_decompress<DTYPE, 8, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 4: return launch_decompress<DTYPE, 4, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 2: return launch_decompress<DTYPE, 2, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        case 1: return launch_decompress<DTYPE, 1, D>(job, jobs_dev, n_jobs, max_vec, dl, s);
        default: return TQ_ERR_BITS;
    }
}

}  // namespace

// The entry points of one dimension (tq_wide.h), `dl` of whose coordinates a vector has.
#define TQ_WIDE_DEFINE(D)                                                                                                                        \
    int tq_wide_compress_d##D(int dtype, int bits, uint32_t dl, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec,       \
                              hipStream_t s) {                                                                                                  \
        return dtype == TQ_F16 ? compress_bits<TQ_F16, D>(bits, job, jobs_dev, n_jobs, max_vec, dl, s)                                           \
                               : compress_bits<TQ_BF16, D>(bits, job, jobs_dev, n_jobs, max_vec, dl, s);                                         \
    }                                                                                                                                            \
    int tq_wide_decompress_d##D(int dtype, int bits, uint32_t dl, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec,     \
                                hipStream_t s) {                                                                                                \
        return dtype == TQ_F16 ? decompress_bits<TQ_F16, D>(bits, job, jobs_dev, n_jobs, max_vec, dl, s)                                         \
                               : decompress_bits<TQ_BF16, D>(bits, job, jobs_dev, n_jobs, max_vec, dl, s);                                       \
    }                                                                                                                                            \
    int tq_wide_compress_layer_d##D(int dtype, uint32_t dl, TqLayer &l, uint32_t n_vec, hipStream_t s) {       \
        if (dl != (uint32_t)D)                                                                                                                   \
            return dtype == TQ_F16 ? launch_compress_layer<TQ_F16, D, true>(l, n_vec, dl, s)                                     \
                                   : launch_compress_layer<TQ_BF16, D, true>(l, n_vec, dl, s);                                   \
        return dtype == TQ_F16 ? launch_compress_layer<TQ_F16, D, false>(l, n_vec, dl, s)                                        \
                               : launch_compress_layer<TQ_BF16, D, false>(l, n_vec, dl, s);                                      \
    }                                                                                                                                            \
    int tq_wide_restore_layer_d##D(int dtype, uint32_t dl, TqLayer &l, const TqWindowCopy &w, uint32_t n_vec,  \
                                   hipStream_t s) {                                                                                             \
        if (dl != (uint32_t)D)                                                                                                                   \
            return dtype == TQ_F16 ? launch_restore_layer<TQ_F16, D, true>(l, w, n_vec, dl, s)                                   \
                                   : launch_restore_layer<TQ_BF16, D, true>(l, w, n_vec, dl, s);                                 \
        return dtype == TQ_F16 ? launch_restore_layer<TQ_F16, D, false>(l, w, n_vec, dl, s)                                      \
                               : launch_restore_layer<TQ_BF16, D, false>(l, w, n_vec, dl, s);                                    \
    }
