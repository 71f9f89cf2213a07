// compress: per-vector L2 norm, rotation on the matrix cores, Lloyd-Max code search, bit packing.
// Replaces MSECompressor.compress (upstream turboquant/compressors_v3.py:46-81) with one kernel.
//
// Work decomposition (gfx950, wave64):
//   * a block is four waves that share tiles of 32 consecutive vectors; wave w keeps the quarter
//     of the rotation that produces coordinates [32w, 32w+32) resident in registers as MFMA A
//     operands (all 16-bit terms of the split: 64 registers), so the matrix pipe never waits for
//     operand loads and several waves fit on a SIMD;
//   * the tile is fetched with fully coalesced 16-byte loads (one instruction = 1 KiB of
//     consecutive memory, a quarter of them by each wave), parked in a double-buffered,
//     XOR-swizzled LDS buffer (one barrier per tile) and read back as the B operand of
//     v_mfma_f32_32x32x16 (vector n on MFMA column n);
//   * the rotation is pre-split on the host into 16-bit terms whose sum is Pi to ~2^-22 (fp16
//     path) / 2^-17 (bf16 path); inputs are exact in the MFMA input type (fp32 inputs are split
//     into three exact bf16 terms and use three Pi terms), accumulation is fp32, so the rotated
//     coordinates agree with an fp32 GEMM to ~1e-6 or better;
//   * the rotation is applied to the raw vector and scaled by 1 / (norm + 1e-8) afterwards
//     (linearity), so the norm reduction overlaps the MFMAs;
//   * every lane ends up with 16 consecutive rotated coordinates of one vector: the code search
//     is two fused multiply-adds, one 8-byte LDS lookup and a funnel shift per coordinate, and
//     the packed bytes of a lane are contiguous in memory;
//   * tiles whose 32 vectors all exist take a path without per-lane predicates: a fixed number
//     of loads and stores per iteration lets the compiler wait for the prefetched loads alone
//     (s_waitcnt vmcnt(n)) instead of draining the previous tile's stores on every iteration.
#include <mutex>
#include <type_traits>

#include "tq_anydim.h"
#include "tq_device.h"

namespace {

#ifndef TQ_C16_WAVES
#define TQ_C16_WAVES 3
#endif
// tiles of 16-bit input that a block keeps in LDS or on their way there (direct-to-LDS loads)
#ifndef TQ_RING
#define TQ_RING 4
#endif
#ifndef TQ_PIN_SCHEDULE
#define TQ_PIN_SCHEDULE 1
#endif
// log2 of the iterations a block keeps one issue priority before it moves to the next (0: priorities stay untouched)
#ifndef TQ_PRIO_SHIFT
#define TQ_PRIO_SHIFT 3
#endif
// Measurement build (never the shipped library): the pipelined path keeps its loads, LDS traffic, barriers, norm
// arithmetic and stores, and leaves out the matrix instructions and the code search (1), the matrix instructions only
// (2) or the code search only (3).  What it writes is garbage; its time is what the rest of the kernel costs on its own.
#ifndef TQ_SKELETON
#define TQ_SKELETON 0
#endif
#define TQ_SKEL_NO_MFMA (TQ_SKELETON == 1 || TQ_SKELETON == 2)
#define TQ_SKEL_NO_SEARCH (TQ_SKELETON == 1 || TQ_SKELETON == 3)
template <int DTYPE> struct InTraits;
template <> struct InTraits<TQ_F16> { static constexpr int ELEM = 2, TERMS = 2, MIN_WAVES = TQ_C16_WAVES; };
template <> struct InTraits<TQ_BF16> { static constexpr int ELEM = 2, TERMS = 2, MIN_WAVES = TQ_C16_WAVES; };
// fp32 input keeps three rotation terms resident and stages tiles as three bf16 terms, 24 KiB
template <> struct InTraits<TQ_F32> { static constexpr int ELEM = 4, TERMS = 3, MIN_WAVES = 2; };

constexpr int CWAVES = TQ_TILES;        // waves per block = MFMA row tiles
constexpr int CTHREADS = CWAVES * TQ_WAVE;

// calls step(k) for k = FROM .. TO-1 until one of them reports the end; true = ended
template <uint32_t FROM, uint32_t TO, typename F>
__device__ __forceinline__ bool run_tail(F &step) {
    if constexpr (FROM >= TO) {
        return false;
    } else {
        if (step(std::integral_constant<uint32_t, FROM>{})) return true;
        return run_tail<FROM + 1, TO>(step);
    }
}

// LDS of a block, the same arrays for every width (several bodies in one kernel share them).  Arrays of their own and not one structure:
// the compiler then knows that the tiles, the grid and the sums do not overlap, and orders their accesses freely (one structure: the
// pipelined loop waits more, compress launches of the 32-layer cache + 2 %).
template <int DTYPE>
struct CompressLds {
    static constexpr int ELEM = InTraits<DTYPE>::ELEM;
    static constexpr int RING = ELEM == 2 ? TQ_RING : 2;     // staged tiles
    using Grid = uint8_t[TQ_GRID_LDS_BYTES];
    using Stage = uint8_t[RING][32 * TQ_HEAD_DIM * (ELEM == 2 ? 2 : 6)];
    using Part = float[2][32][4];      // sum of squares of the tile's vectors, one share per wave (pipelined path)
    using Ss = float[2][32];           // the same, whole (16-bit inputs)
    using Ssh = float[ELEM == 2 ? 2 : 3][32][2];       // the same per half of a row (rows that are pairs of 64-wide vectors; fp32 inputs)
    using Tk = uint32_t[4];            // ticket k of the block sits in slot k % 4 (counter mode only)
    static __device__ __forceinline__ Grid &grid() { __shared__ __attribute__((aligned(16))) Grid a; return a; }
    static __device__ __forceinline__ Stage &stage() { __shared__ __attribute__((aligned(1024))) Stage a; return a; }
    static __device__ __forceinline__ Part &part() { __shared__ __attribute__((aligned(16))) Part a; return a; }
    static __device__ __forceinline__ Ss &ss() { __shared__ Ss a; return a; }
    static __device__ __forceinline__ Ssh &ssh() { __shared__ Ssh a; return a; }
    static __device__ __forceinline__ Tk &tk() { __shared__ Tk a; return a; }
};

// One block's share of a job; `workspace`: the job's two counters, or NULL.
template <int DTYPE, int BITS>
__device__ __forceinline__ void compress_job(const TqDevJob &job, TqBlock blk, uint32_t *workspace, uint32_t tshift, uint32_t paired) {
    using T = InTraits<DTYPE>;
    using P = Pack<BITS>;
    constexpr int ELEM = T::ELEM;
    constexpr int VEC_BYTES = TQ_HEAD_DIM * ELEM;      // 256 or 512
    constexpr int STAGE = 32 * VEC_BYTES;              // one tile
    constexpr int NLOAD = STAGE / 1024 / CWAVES;       // 16-byte loads per lane per tile (this wave's quarter)
    constexpr int PIECES = VEC_BYTES / 16;             // 16-byte pieces per vector
    constexpr int VEC_PER_LOAD = 64 / PIECES;          // vectors covered by one load instruction
    constexpr int NB = P::NB, NW = P::NW;
    constexpr int TERM = 32 * TQ_HEAD_DIM * 2;         // one bf16 term of a staged tile of fp32 inputs

    constexpr int RING = CompressLds<DTYPE>::RING;
    auto &lds_grid = CompressLds<DTYPE>::grid();
    auto &lds_stage = CompressLds<DTYPE>::stage();
    auto &lds_ss = CompressLds<DTYPE>::ss();
    auto &lds_ssh = CompressLds<DTYPE>::ssh();
    auto &lds_part = CompressLds<DTYPE>::part();
    auto &tk = CompressLds<DTYPE>::tk();

    // paired: the job's vectors are 64 wide and the kernel works on pairs of them as 128-wide rows (diag(Pi, Pi) from the
    // table's pair sections).  Everything is as for 128-wide vectors except the norm: one per half of a row; the
    // coordinates of wave w belong to half w / 2.

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63u;
    const uint32_t wave = tid >> 6;
    const uint32_t n_tiles = (job.n_vec + 31u) / 32u;
    if (n_tiles == 0u) return;    // an empty job of a batch: its table may be NULL, and its counters stay untouched (zero)
    const uint32_t n_full = job.n_vec / 32u;
    const bool one_row = job.tokens >= job.n_vec;
    // Which tiles a block works on.  Jobs of 16-bit elements (the pipelined path below) hand their tiles out
    // as tickets of 2^tshift consecutive tiles: block b starts with ticket b; its later tickets are b + grid, b + 2 grid, ...
    // (fixed assignment) or, with a workspace, come from a counter in device memory in the order in which the blocks
    // ask, so that compute units that run slower than others (the dies of this part do not all run at one pace) take
    // fewer tiles and all blocks of a job end together.  counter[0] = tiles handed out beyond every block's first ticket,
    // counter[1] = blocks of the job that are done; the last block to finish sets both back to zero, so a workspace
    // that was zero before a launch is zero after it (the contract of the decompress kernel's counters).
    // Every other job walks single tiles blk.x, blk.x + grid, ...
    // Several rows (a token slice of a [B, H, S, D] tensor, a window left behind): a tile is 32 vectors of the rows laid
    // end to end, so with at least 32 tokens a row it touches two rows at most; vectors of the second one lie `row_skip`
    // bytes further than the tile's own stride says.  The loads take 32-bit offsets from the tile's first vector, which
    // bounds token_stride and row_skip; rows that overlap or lie further apart take the plain loop.
    // Bound: as for one row (memory and the power limit); the plain loop it replaces for these jobs re-divided every
    // lane's index and waited for each tile.  4-bit bf16, all but the last 128 tokens of a row: 8 rows of 32768 tokens
    // 27.9 -> 25.8 us, 32 such rows 105 -> 92 us, 128 rows of 8192 100 -> 91 us (a dense tensor of that size: 91 us).
    const long long row_skip = one_row ? 0 : job.row_stride - (long long)job.tokens * job.token_stride;
    const bool ticket_job = ELEM == 2 && job.token_stride < (1ll << 26) &&
                            (one_row || (job.tokens >= 32u && row_skip >= 0 && row_skip < (1ll << 31)));
    // (a ticket has to outlast the pipeline's depth: the first drawn ticket is published one iteration after the start)
    uint32_t *counter = workspace && (1u << tshift) > (uint32_t)TQ_RING ? workspace : nullptr;
    auto report_done = [&]() {      // once per block of a non-empty job, after its last draw has been answered
        if (counter && tid == 0) {
            if (atomicAdd(counter + 1, 1u) == blk.grid - 1u) {
                atomicExch(counter, 0u);
                atomicExch(counter + 1, 0u);
            }
        }
    };
    uint32_t tile = ticket_job ? blk.x << tshift : blk.x;
    if (tile >= n_tiles) {        // whole block idle (uniform)
        report_done();
        return;
    }
    const uint32_t tile_stride = blk.grid;

    const TqTableHeader *hd = reinterpret_cast<const TqTableHeader *>(job.table);

    // ---- this wave's quarter of the rotation, resident for the whole kernel.  Wave w walks the 16-input
    // steps of the contraction in the order 2w, 2w+1, ... (mod 8): its first two steps then cover inputs
    // [32w, 32w+32), the share of the vector whose squares it sums in the pipelined path.
    const uint32_t step0 = ELEM == 2 ? 2u * wave : 0u;
    tq_u4 areg[T::TERMS][TQ_STEPS];
    // Rotation operands into registers and the quantiser grid into LDS (one copy per code position, base pre-shifted).
    // Every cell is fetched once and written to all its copies; the fetches of a thread are issued together.
    // Called once per block: behind the first tile loads on the pipelined path, so that their latencies overlap.  Sections are taken where every
    // table has them: the table's header in front was a trip to memory of its own (16 rows of 3968
    // tokens, K6/V4, compress and restore, which does the same: 32.0 -> 31.3 us).
    auto load_tables = [&]() {
        const uint8_t *src = job.table + (DTYPE == TQ_F16 ? TQ_OFF_A_F16 : TQ_OFF_A_BF16(TQ_HEAD_DIM));
        uint32_t grid = TQ_OFF_GRID(TQ_HEAD_DIM);
        if (paired) {      // (tables of 64-wide vectors: the pairs' section lies behind sections of the width)
            src = job.table + (DTYPE == TQ_F16 ? hd->off_pair_a_f16 : hd->off_pair_a_bf16);
            grid = TQ_OFF_GRID(TQ_HEAD_DIM / 2);
        }
#pragma unroll
        for (int term = 0; term < T::TERMS; ++term)
#pragma unroll
            for (int s = 0; s < TQ_STEPS; ++s)
                areg[term][s] = tq_gload16(src + (size_t)term * TQ_OPERAND_BYTES +
                                           (((size_t)wave * TQ_STEPS + ((s + step0) & 7u)) * 64 + lane) * 16);
        constexpr int CELL_TRIPS = (TQ_GRID_MAX_CELLS(BITS) + CTHREADS - 1) / CTHREADS;
        constexpr uint32_t cells = TQ_GRID_MAX_CELLS(BITS);      // (a table has room for as many: how many it uses need not be known)
        const uint8_t *gsrc = job.table + grid;
        tq_u2 cell[CELL_TRIPS];
#pragma unroll
        for (int k = 0; k < CELL_TRIPS; ++k) {
            const uint32_t q = tid + k * CTHREADS;
            cell[k] = tq_gload8(gsrc + 8u * (q < cells ? q : 0u));
        }
#pragma unroll
        for (int k = 0; k < CELL_TRIPS; ++k) {
            const uint32_t q = tid + k * CTHREADS;
            if (q < cells) {
#pragma unroll
                for (int c = 0; c < P::COPIES; ++c) {
                    const tq_u2 e = {cell[k][0], cell[k][1] << copy_shift_rt<BITS>(c)};
                    *reinterpret_cast<tq_u2 *>(lds_grid + c * P::COPY_STRIDE + 8u * q) = e;
                }
            }
        }
    };
    const float grid_scale = hd->grid_scale, grid_bias = hd->grid_bias;

    // Role in the loads, 16 bytes a lane.  16-bit inputs: piece ld_piece of vector ld_vec of every four.  fp32 inputs: eight lanes share a
    // vector; lane (vk, vq) has the eight elements of half vk of steps 2 vq and 2 vq + 1, pieces ld_piece + {0, 1, 4, 5} (see park).
    const uint32_t vk = (lane >> 2) & 1u, vq = lane & 3u;
    const uint32_t ld_vec = ELEM == 2 ? lane / PIECES : lane >> 3, ld_piece = ELEM == 2 ? lane % PIECES : 8u * vq + 2u * vk;
    const uint32_t n = lane & 31u, hk = lane >> 5;                    // role in the MFMA: column, half
    const uint32_t half = wave >> 1;                                  // paired rows: the 64-wide vector this wave's coordinates belong to

    // LDS offset of this lane's piece of load j of 16-bit inputs (computed where it is used: these paths are not the hot one)
    auto st_off = [&](int j) {
        const uint32_t vl = (wave * NLOAD + j) * VEC_PER_LOAD + ld_vec;
        return vl * VEC_BYTES + ((ld_piece ^ (vl & 15u)) << 4);
    };

    tq_u4 pre[NLOAD];
    // loads of this wave's quarter of tile `tl`, generic addressing (any strides, tail clamped)
    auto load_vector = [&](const uint8_t *at) {      // fp32 inputs
#pragma unroll
        for (int j = 0; j < NLOAD; ++j) pre[j] = tq_gload16(at + (j / 2) * 64 + (j % 2) * 16);
    };
    auto issue_loads = [&](auto full_tag, uint32_t tl) {
        constexpr bool FULL = decltype(full_tag)::value;
        const uint32_t v0 = tl * 32u + (wave * NLOAD) * VEC_PER_LOAD + ld_vec;
#pragma unroll
        for (int j = 0; j < (ELEM == 2 ? NLOAD : 1); ++j) {
            uint32_t v = v0 + j * VEC_PER_LOAD;
            if (!FULL) v = v < job.n_vec ? v : job.n_vec - 1u;   // tail: re-read the last vector, never stored
            const uint8_t *at = job.states + tq_vec_offset(job, v) + ld_piece * 16u;
            if constexpr (ELEM == 2) pre[j] = tq_gload16(at);
            else load_vector(at);
        }
    };

    // Park this wave's quarter of the prefetched tile in LDS (swizzled: the operand reads are conflict
    // free).  For 16-bit inputs the squares are summed here, where every element is touched once: the 16
    // lanes of a DPP row hold the 16 pieces of one vector.  The order of the additions is the one of the
    // pipelined path below (pieces 4w + h and 4w + 2 + h as one chain, the two chains of a wave's share
    // added, the shares added pairwise), so that a vector gets the same norm whichever path compresses it.
    auto row_shr = [](float v, auto n_tag) {
        constexpr int N = decltype(n_tag)::value;
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x110 + N, 0xf, 0xf, true));
    };
    // fp32 inputs are split into their terms here, once (by the waves that read the operands it took four times as many vector
    // instructions as everything else together).  Their squares are added in the order in which those waves walked a vector, which fixes the
    // last bit of the norm and with it the codes next to a boundary: four chains, over the even and the odd elements of either half (hk) of
    // the steps 0..7.  The eight lanes of a vector, two steps of a half each, hand the chains on from lane to lane.  The sum ends up in
    // element 1 of slot `slot`; pairs of 64-wide vectors, four steps each, use both.  (131168 vectors, 4-bit: 31.5 us.  Squares added by lanes
    // of whole loads, in an order of their own, 30.9; in this order from such loads, pieces exchanged through the LDS, 3 us more.)
    auto park = [&](uint32_t b, uint32_t slot, const tq_u4 (&src)[NLOAD]) {
        uint8_t *stage = lds_stage[b];
        if constexpr (ELEM == 2) {
#pragma unroll
            for (int j = 0; j < NLOAD; ++j) *reinterpret_cast<tq_u4 *>(stage + st_off(j)) = src[j];
#pragma unroll
            for (int j = 0; j < NLOAD; ++j) {
                const float own = sumsq8<DTYPE>(src[j], 0.f);
                const float chain = sumsq8<DTYPE>(src[j], row_shr(own, std::integral_constant<int, 2>{}));   // pieces p - 2, p
                const float share = chain + row_shr(chain, std::integral_constant<int, 1>{});               // at p % 4 == 3
                const float pair = share + row_shr(share, std::integral_constant<int, 4>{});                // at p == 7, 15
                const float total = pair + row_shr(pair, std::integral_constant<int, 8>{});                 // at p == 15
                if ((lane & 15u) == 15u) lds_ss[b][(wave * NLOAD + j) * VEC_PER_LOAD + ld_vec] = total;
                if ((lane & 7u) == 7u) lds_ssh[b][(wave * NLOAD + j) * VEC_PER_LOAD + ld_vec][(lane >> 3) & 1u] = pair;   // pieces 0..7, 8..15
            }
        } else {
            static_assert(NLOAD == 4 && VEC_PER_LOAD == 2, "eight vectors a wave, four pieces a lane");
            const bool first = vq == 0u || (paired && vq == 2u);
            auto handed_on = [&](float s) {      // from the lane before it in its quad
                const float t = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, s), 0x90, 0xf, 0xf, true));
                return first ? 0.f : t;
            };
            float s0 = 0.f, s1 = 0.f;
#pragma unroll
            for (int turn = 0; turn < 4; ++turn) {      // (after turn t the chains are right up to lane t of the quad)
                if (turn) {
                    s0 = handed_on(s0);
                    s1 = handed_on(s1);
                }
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    const tq_u4 &p = src[i / 4];
                    const float e = __uint_as_float(p[i % 4]), o = __uint_as_float(p[i % 4 + 1]);
                    s0 = fmaf(e, e, s0);
                    s1 = fmaf(o, o, s1);
                }
            }
            const float one = s0 + s1, both = one + row_shr(one, std::integral_constant<int, 4>{});       // at vk == 1
            if (vk == 1u && (vq & 1u)) lds_ssh[slot][wave * 8u + ld_vec][vq >> 1] = both;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                tq_u4 t[3];
#pragma unroll
                for (int d = 0; d < 4; ++d) {      // x = its three terms exactly: every term a truncation, every remainder exact
                    uint32_t r[2][3];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        const float f = __uint_as_float(src[2 * a + d / 2][d % 2 * 2 + i]);
                        const float r1 = f - __uint_as_float(__float_as_uint(f) & 0xffff0000u);
                        const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
                        r[i][0] = __float_as_uint(f); r[i][1] = __float_as_uint(r1); r[i][2] = __float_as_uint(r2);
                    }
#pragma unroll
                    for (int k = 0; k < 3; ++k) t[k][d] = __builtin_amdgcn_perm(r[1][k], r[0][k], 0x07060302u);
                }
                const uint32_t vl = wave * 8u + ld_vec, at = vl * (TQ_HEAD_DIM * 2) + (((4u * vq + 2u * a + vk) ^ (vl & 15u)) << 4);
#pragma unroll
                for (int k = 0; k < 3; ++k) *reinterpret_cast<tq_u4 *>(stage + k * TERM + at) = t[k];
            }
        }
    };

    // ---- the three stages of a tile ---------------------------------------------------------
    // (1) rotation step s of the tile parked in `stage`: acc[r] += sum over 16 inputs of
    //     Pi[32w + 16h + r][k] * x_n[k]  (raw, unnormalised)
    auto rotate_step = [&](const uint8_t *stage, int s, tq_f16v &acc) {
        const uint32_t sg = ((uint32_t)s + step0) & 7u;   // the step of the contraction that areg[.][s] belongs to
        const uint8_t *at = stage + n * (TQ_HEAD_DIM * 2) + (((2u * sg + hk) ^ (n & 15u)) << 4);
        if constexpr (ELEM == 2) {
            const tq_u4 bop = *reinterpret_cast<const tq_u4 *>(at);
#pragma unroll
            for (int term = 0; term < T::TERMS; ++term)
                acc = (DTYPE == TQ_F16) ? mfma_f16(areg[term][s], bop, acc) : mfma_bf16(areg[term][s], bop, acc);
        } else {
            // all products whose weight is >= 2^-24 of the leading one: (x term i, Pi term j), i + j <= 2
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const tq_u4 bop = *reinterpret_cast<const tq_u4 *>(at + i * TERM);
#pragma unroll
                for (int term = 0; term + i < 3; ++term) acc = mfma_bf16(areg[term][s], bop, acc);
            }
        }
    };

    // (2) norm of the lane's vector and the two scale factors of the code search
    struct Scale { float nrm, inv, inv_cell; };
    auto scale_from_ss = [&](float ss) {
        Scale sc;
        sc.nrm = tq_norm_from_sumsq(ss);
        // 1 / (norm + 1e-8): the reciprocal only scales the coordinates, one ulp is irrelevant
        sc.inv = __builtin_amdgcn_rcpf(sc.nrm + 1e-8f);
        if (DTYPE == TQ_F16) sc.inv *= 1.0f / (float)(1 << TQ_F16_PI_SHIFT);
        sc.inv_cell = sc.inv * grid_scale;   // grid_scale is a power of two: exact
        return sc;
    };
    auto scale_of = [&](uint32_t slot) {
        if constexpr (ELEM == 2) return scale_from_ss(paired ? lds_ssh[slot][n][half] : lds_ss[slot][n]);
        else return scale_from_ss(lds_ssh[slot][n][paired ? half : 1u]);
    };

    // (3) code search + packing.  Lane (n, hk) of wave w holds coordinates 32w + 16hk + r.
    // Per coordinate: cell address (fma, and), one 8-byte LDS lookup from the grid copy whose base
    // is pre-shifted to the code's bit position, exact comparison by fma, sign bit funnelled
    // into `lt`, bases OR-ed together.  code = base + !(rho < threshold).
    // The 16 coordinates of a lane are visited in the order q = 0..15 = (word, position in word).
    struct Search { uint32_t lt[NW], lo[NW], hi[NW]; };
    auto search_begin = [&](Search &z) {
#pragma unroll
        for (int w = 0; w < NW; ++w) z.lt[w] = z.lo[w] = z.hi[w] = 0u;
    };
    auto search_lookup = [&](int q, const tq_f16v &acc, const Scale &sc) {
        const int w = q / P::CPW, i = q % P::CPW;
        const float a = acc[P::local_code(w, i)];
        const uint32_t addr = __float_as_uint(fmaf(a, sc.inv_cell, grid_bias)) & TQ_GRID_ADDR_MASK;
        return *reinterpret_cast<const tq_u2 *>(lds_grid + P::copy_of(i) * P::COPY_STRIDE + addr);
    };
    auto search_apply = [&](Search &z, int q, const tq_f16v &acc, const Scale &sc, tq_u2 cell) {
        const int w = q / P::CPW, i = q % P::CPW;
        const float a = acc[P::local_code(w, i)];
        const float t = fmaf(a, sc.inv, -__uint_as_float(cell[0]));
        const int cursor = i == 0 ? 8 * P::WB : P::shift_of(i - 1);
        const int gap = cursor - (P::shift_of(i) + P::FIELD);
        if (gap > 0) z.lt[w] = __builtin_amdgcn_alignbit(z.lt[w], 0u, 32 - gap);
        z.lt[w] = __builtin_amdgcn_alignbit(z.lt[w], __float_as_uint(t), 32 - P::FIELD);
        if (P::IPB == 1 && P::byte_of(i) >= 2) z.hi[w] |= cell[1]; else z.lo[w] |= cell[1];
    };
    auto search_coord = [&](Search &z, int q, const tq_f16v &acc, const Scale &sc) {
        search_apply(z, q, acc, sc, search_lookup(q, acc, sc));
    };
    auto search_end = [&](const Search &z, uint32_t (&words)[NW]) {
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            const uint32_t bases = P::IPB == 1 ? (z.lo[w] | (z.hi[w] << 16)) : z.lo[w];
            const uint32_t ge = (~z.lt[w] & P::sign_mask()) >> (P::FIELD - 1);
            words[w] = bases + ge;
        }
    };

    // One tile, parked in buffer `b` and published by a barrier: rotate, then search.
    // Leaves the lane's packed words in `words` and the vector's norm in `nrm`.
    auto compute = [&](uint32_t b, uint32_t (&words)[NW], float &nrm) {
        tq_f16v acc = tq_zero16();
#pragma unroll
        for (int s = 0; s < TQ_STEPS; ++s) rotate_step(lds_stage[b], s, acc);
        const Scale sc = scale_of(b);
        Search z;
        search_begin(z);
#pragma unroll
        for (int q = 0; q < 16; ++q) search_coord(z, q, acc, sc);
        search_end(z, words);
        nrm = sc.nrm;
    };

    // the lane's NB packed bytes and (identical in all lanes of a vector) the fp16 norm
    auto store = [&](uint8_t *dst, uint16_t *ndst, const uint32_t (&words)[NW], float nrm) {
        if constexpr (NB == 2) {
            tq_gstore2(reinterpret_cast<uint16_t *>(dst), (uint16_t)words[0]);
        } else if constexpr (NB == 4) {
            *reinterpret_cast<TQ_GLOBAL uint32_t *>((TQ_GLOBAL uint8_t *)dst) = words[0];
        } else if constexpr (NB == 8) {
            tq_u2 o = {words[0], words[1]};
            tq_gstore8(dst, o);
        } else {
            tq_u4 o = {words[0], words[1], words[2], words[3]};
            tq_gstore16(dst, o);
        }
        // every lane of every wave holds the same norm for vector n: all store it (identical values
        // to one address) rather than predicating the store on a fraction of the lanes
        const _Float16 hn = (_Float16)nrm;
        tq_gstore2(ndst, __builtin_bit_cast(uint16_t, hn));
    };
    const uint32_t lane_slot = (2u * wave + hk) * NB;   // this lane's bytes inside a vector's G = 8 * NB
    auto norm_slot = [&](size_t slot) { return paired ? 2u * slot + half : slot; };     // where the norm of this wave's half of row `slot` goes

    uint32_t buf = 0;
    uint32_t words[NW];
    float nrm;
    // (the pipelined path addresses a tile's vectors with 32-bit offsets from a scalar base: the stride limit of ticket_job)
    const bool pipelined = ticket_job && tile < n_full;
    if (!pipelined && (ELEM == 2 || tile >= n_full)) load_tables();
    if (pipelined) {
        if constexpr (ELEM == 2) {
            // Jobs with 16-bit elements (the KV-cache case): a software pipeline over this block's full
            // tiles t_0 .. t_{m-1}.  Tiles travel from memory straight into a ring of RING LDS slots
            // (global_load_lds_dwordx4: no registers, no LDS write instructions); iteration j
            //   waits for its own loads of t_j (issued RING-1 iterations ago) and passes the barrier: t_j is complete
            //   in slot j % RING, and everybody has finished reading t_{j-1};
            //   starts the loads of t_{j+RING-1} into the slot that t_{j-1} has just left;
            //   rotates t_j on the matrix cores while it searches and packs the codes of t_{j-1}, whose rotated
            //   coordinates wait in the other accumulator set (two independent instruction streams: the VALU work
            //   fills the issue slots under the MFMAs); the scale of t_{j-1} comes from the four waves' shares of
            //   its sum of squares, written an iteration ago;
            //   sums the squares of its own share of t_j from the first two operands it feeds to the matrix cores;
            //   stores t_{j-1}.
            // The loads are invisible to the compiler (inline assembly), so it never waits for them; the explicit
            // s_waitcnt counts the younger vector-memory operations of the wave, which is fixed: 2 loads and
            // 2 stores per iteration.
            constexpr int P = RING;
            static_assert(NLOAD == 2 && P >= 2 && P <= 6, "the wait counts below assume two loads per wave and tile");
            // lane i of load j fills bytes [16 i, 16 i + 16) of KiB (wave * NLOAD + j) of the slot: vector
            // vl = (wave * NLOAD + j) * 4 + i / 16, position i % 16, which has to hold piece (i % 16) ^ (vl & 15)
            uint32_t src_off[NLOAD];
#pragma unroll
            for (int j = 0; j < NLOAD; ++j) {
                const uint32_t vl = (wave * NLOAD + j) * VEC_PER_LOAD + ld_vec;
                src_off[j] = vl * (uint32_t)job.token_stride + ((ld_piece ^ (vl & 15u)) << 4);
            }
            const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(
                (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)&lds_stage[0][0] + wave * (NLOAD * 1024u));

            // ---- the block's sequence of tiles.  q[i] = the tile of iteration j - 1 + i while iteration j runs: q[0] is
            // searched and stored, q[1] rotated, q[P] loaded.  All of it lives in scalar registers.  A value >= n_full
            // marks the end (the sequence of a block only grows); loads past the end re-read the job's last full tile.
            const uint32_t per_ticket = 1u << tshift;
            const uint32_t drawn_origin = blk.grid << tshift;
            uint32_t q[P + 1];
            uint32_t left = per_ticket - 1u;    // tiles of the head's ticket beyond the head
            uint32_t kt = 0;                    // tickets the head has entered beyond the first
            uint32_t drawn = 0;                 // thread 0: what the atomic of this iteration's draw returned, not yet looked at
            bool have_drawn = false;
            auto draw = [&]() {                 // counter mode; the value is taken by thread 0 alone
                // (the returned value stays untouched until publish(): arithmetic on it here would put a wait for all of
                // the wave's memory operations right behind the atomic)
                if (tid == 0) drawn = atomicAdd(counter, per_ticket);
                have_drawn = true;
            };
            auto publish = [&]() {              // at the end of an iteration: the draw's latency hides behind the tile's work
                if (have_drawn) {
                    if (tid == 0) tk[(kt + 1u) & 3u] = drawn_origin + drawn;
                    have_drawn = false;
                }
            };
            auto advance = [&](uint32_t head) -> uint32_t {    // the tile after `head` in this block's sequence
                if (left) {
                    --left;
                    return head + 1u;
                }
                left = per_ticket - 1u;
                ++kt;
                if (counter) {
                    // ticket kt was drawn when the head entered ticket kt - 1, at least four iterations (one barrier) ago
                    const uint32_t base = (uint32_t)__builtin_amdgcn_readfirstlane(tk[kt & 3u]);
                    draw();
                    return base;
                }
                return (blk.x + kt * blk.grid) << tshift;
            };
            q[0] = 0xffffffffu;
            q[1] = tile;
#pragma unroll
            for (int i = 2; i <= P; ++i) q[i] = advance(q[i - 1]);     // (counter mode: tickets hold more than P tiles, no draw here)
            if (counter) draw();                // ticket 1: in LDS at the end of the first iteration, read per_ticket - P iterations later
            // Row and token of a tile's first vector v, on the scalar unit: with inv_tokens = floor(2^32 / tokens) + 1 the high
            // half of v * inv_tokens is v / tokens or one more (v < 2^31); one row: inv_tokens = 0 and the row is 0.
            const uint32_t inv_tokens = one_row ? 0u : 0xffffffffu / job.tokens + 1u;
            auto row_of = [&](uint32_t v) -> uint32_t {
                const uint32_t r = (uint32_t)(((uint64_t)v * inv_tokens) >> 32);
                return r * job.tokens > v ? r - 1u : r;
            };
            auto issue = [&](uint32_t slot, uint32_t tl) {
                tl = tl < n_full ? tl : n_full - 1u;
                const uint32_t row = row_of(tl * 32u);
                const uint64_t a = (uint64_t)(uintptr_t)job.states + (uint64_t)tl * (uint64_t)(32 * job.token_stride) + (uint64_t)row * (uint64_t)row_skip;
                // (the builtin returns int: widen through uint32_t, or the low half is sign-extended into the high one)
                const uint32_t a_hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
                const uint32_t a_lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
                const uint64_t base = ((uint64_t)a_hi << 32) | (uint64_t)a_lo;
                // vectors of the tile that belong to its first row (all of them, unless a row ends inside the tile)
                const uint32_t mine = one_row ? 32u : (row + 1u) * job.tokens - tl * 32u;
                uint32_t off[NLOAD];
#pragma unroll
                for (int j = 0; j < NLOAD; ++j) off[j] = src_off[j];
                if (mine < 32u) {       // uniform
                    asm volatile("");   // stays a branch (as selects in every tile: 24 tensors of 8 x 4099 tokens, 4-bit, 63.0 us, this way 62.2)
#pragma unroll
                    for (int j = 0; j < NLOAD; ++j)
                        if ((wave * NLOAD + j) * VEC_PER_LOAD + ld_vec >= mine) off[j] += (uint32_t)row_skip;
                }
#pragma unroll
                for (int j = 0; j < NLOAD; ++j) {
                    const uint32_t dst = lds_wave + slot * (uint32_t)STAGE + j * 1024u;
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                                 :: "s"(dst), "v"(off[j]), "s"(base) : "memory", "m0");
                }
            };
            // operand addresses inside a slot, in this wave's step order
            uint32_t op_off[TQ_STEPS];
#pragma unroll
            for (int i = 0; i < TQ_STEPS; ++i) {
                const uint32_t piece = 2u * ((i + step0) & 7u) + hk;
                op_off[i] = n * VEC_BYTES + ((piece ^ (n & 15u)) << 4);
            }
            const uint32_t bperm_other_half = (lane ^ 32u) << 2;

            // output addresses: a base per tile that is the same in every lane, plus a per-lane constant
            const uint32_t cd_lane = n * (8 * NB) + lane_slot, nd_lane = n;
            const uint32_t slot_skip = job.packed_row_stride - job.tokens;     // packed slots between the rows (one row: not looked at)
            auto store_tile = [&](uint32_t tl, const uint32_t (&w)[NW], float nrm_of_tile) {
                if (one_row) {
                    store(job.idx_bytes + (size_t)tl * (32u * (8 * NB)) + cd_lane, job.vec_norms + norm_slot((size_t)tl * 32u + nd_lane), w, nrm_of_tile);
                } else {
                    const uint32_t row = row_of(tl * 32u), v = tl * 32u + n;
                    const uint32_t slot = v + (row + (v >= (row + 1u) * job.tokens ? 1u : 0u)) * slot_skip;
                    store(job.idx_bytes + (size_t)slot * (8 * NB) + lane_slot, job.vec_norms + norm_slot(slot), w, nrm_of_tile);
                }
            };

            auto scale_from_shares = [&](uint32_t par) {
                const float4 q = *reinterpret_cast<const float4 *>(&lds_part[par][n][0]);
                const float lo_half = q.x + q.y, hi_half = q.z + q.w;
                return scale_from_ss(paired ? (half ? hi_half : lo_half) : lo_half + hi_half);
            };
            // iteration j: slot = j % P; `acc_new` receives t_j, `acc_old` holds t_{j-1}
            auto iteration = [&](auto with_search, auto slot_tag, bool warm, uint32_t par, tq_f16v &acc_new, const tq_f16v &acc_old) {
                constexpr bool SEARCH = decltype(with_search)::value;
                constexpr uint32_t SLOT = decltype(slot_tag)::value;
                // younger than the loads of t_j: the loads of P-2 tiles and, once the pipeline is full, the stores of P-1
                if (warm) wait_vmcnt<2 * (P - 2) + 2 * (P - 1)>(); else wait_vmcnt<2 * (P - 2)>();
                __syncthreads();
                issue((SLOT + P - 1u) % P, q[P]);
                const uint32_t head_next = advance(q[P]);
                const uint8_t *stage = lds_stage[SLOT];
                auto operand = [&](int i) { return *reinterpret_cast<const tq_u4 *>(stage + op_off[i]); };
                auto mfma = [&](int term, int i, tq_u4 bop) {
#if TQ_SKEL_NO_MFMA
                    if (term == 0) acc_new[i] = __uint_as_float(bop[0] ^ bop[1] ^ bop[2] ^ bop[3]);     // the operand read stays alive
#else
                    acc_new = (DTYPE == TQ_F16) ? mfma_f16(areg[term][i], bop, acc_new) : mfma_bf16(areg[term][i], bop, acc_new);
#endif
                };
                acc_new = tq_zero16();
                Search z;
                search_begin(z);
                Scale sc_old{};
                float share = 0.f;
                // Order of the instruction stream: the first step's MFMAs come before anything that depends on the
                // scale of t_{j-1} (an LDS read, a reciprocal square root); the search runs one step behind:
                // coordinates 2i-2, 2i-1 are looked up in step i-1 and applied in step i.
                tq_u4 bop = operand(0);
                tq_u2 c0 = {0u, 0u}, c1 = {0u, 0u};
#pragma unroll
                for (int i = 0; i < TQ_STEPS; ++i) {
                    tq_u4 bop_next = bop;
                    tq_u2 n0 = c0, n1 = c1;
                    if (i + 1 < TQ_STEPS) bop_next = operand(i + 1);
                    if constexpr (SEARCH && !TQ_SKEL_NO_SEARCH) {
                        if (i >= 1) { n0 = search_lookup(2 * i - 2, acc_old, sc_old); n1 = search_lookup(2 * i - 1, acc_old, sc_old); }
                    }
                    mfma(0, i, bop);
                    if (i < 2) share = sumsq8<DTYPE>(bop, share);
                    if constexpr (SEARCH) {
                        if (i == 0) sc_old = scale_from_shares(par ^ 1u);
                        if (i >= 2 && !TQ_SKEL_NO_SEARCH) search_apply(z, 2 * i - 4, acc_old, sc_old, c0);
                    }
                    mfma(1, i, bop);
                    if constexpr (SEARCH && !TQ_SKEL_NO_SEARCH) {
                        if (i >= 2) search_apply(z, 2 * i - 3, acc_old, sc_old, c1);
                    }
                    if (i == 1) {
                        share += __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((int)bperm_other_half, __builtin_bit_cast(int, share)));
                        lds_part[par][n][wave] = share;
                    }
#if TQ_PIN_SCHEDULE && !TQ_SKELETON
                    if constexpr (SEARCH) {
                        // pin the order: address arithmetic, the step's LDS reads, then each MFMA followed by the
                        // VALU work that fills its shadow
                        if (i == 0) {
                            __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);   // DS read: next operand, shares
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                            __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);  // VALU: squares, scale
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);
                        } else if (i == 1) {
                            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        } else {
                            __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);   // VALU
                            __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // DS read
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // MFMA
                            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);
                        }
                    }
#endif
                    bop = bop_next; c0 = n0; c1 = n1;
                }
                if constexpr (SEARCH) {
#if TQ_SKEL_NO_SEARCH
#pragma unroll
                    for (int w = 0; w < NW; ++w) words[w] = __float_as_uint(acc_old[w] * sc_old.inv);
#else
                    search_apply(z, 12, acc_old, sc_old, c0);
                    search_apply(z, 13, acc_old, sc_old, c1);
                    search_coord(z, 14, acc_old, sc_old);
                    search_coord(z, 15, acc_old, sc_old);
                    search_end(z, words);
#endif
                    store_tile(q[0], words, sc_old.nrm);
                }
                publish();
#pragma unroll
                for (int i = 0; i < P; ++i) q[i] = q[i + 1];
                q[P] = head_next;
            };
            auto drain = [&](uint32_t par, const tq_f16v &acc_old) {    // par: parity of the iteration that would come next
                __syncthreads();    // the last tile's shares of the sum of squares are complete
                const Scale sc_old = scale_from_shares(par ^ 1u);
                Search z;
                search_begin(z);
#pragma unroll
                for (int q = 0; q < 16; ++q) search_coord(z, q, acc_old, sc_old);
                search_end(z, words);
                store_tile(q[0], words, sc_old.nrm);
            };

#pragma unroll
            for (int p = 0; p < P - 1; ++p) issue((uint32_t)p, q[1 + p]);
            load_tables();      // (the waits for these loads also cover the older tile loads: harmless, once per block)
            tq_f16v acc_a, acc_b;
            uint32_t done = 0;     // iterations finished
            iteration(std::false_type{}, std::integral_constant<uint32_t, 0>{}, false, 0u, acc_a, acc_a);
            ++done;
            // unrolled by U = lcm(2 accumulator sets, P slots); iteration j runs variant j % U
            constexpr uint32_t U = (P % 2 == 0) ? P : 2 * P;
            // The blocks that share a compute unit do not advance at the same pace: the instruction arbiter prefers the
            // oldest wave, so the block dispatched first finishes its tiles well before the one dispatched last, and the
            // unit then runs under-occupied until that one is done.  Every block therefore walks through the issue
            // priorities 0 .. RES-1, a few iterations each, starting from its place in the dispatch order: over time each
            // of the co-resident blocks is preferred equally often, and they finish together.
            constexpr uint32_t RES = T::MIN_WAVES;
            const uint32_t age = ((blockIdx.y * gridDim.x + blockIdx.x) * RES) / (gridDim.x * gridDim.y);
            auto step = [&](auto k_tag) -> bool {    // true = all tiles rotated
                constexpr uint32_t K = decltype(k_tag)::value;
                if (q[1] >= n_full) return true;
                if constexpr (K == 0 && TQ_PRIO_SHIFT > 0) {
                    if ((done & ((1u << TQ_PRIO_SHIFT) - 1u)) == 0u) {
                        const uint32_t prio = (age + (done >> TQ_PRIO_SHIFT)) % RES;
                        if (prio == 0u) __builtin_amdgcn_s_setprio(0);
                        else if (prio == 1u) __builtin_amdgcn_s_setprio(1);
                        else __builtin_amdgcn_s_setprio(2);
                    }
                }
                if constexpr (K & 1u) iteration(std::true_type{}, std::integral_constant<uint32_t, K % P>{}, done >= (uint32_t)P, 1u, acc_b, acc_a);
                else iteration(std::true_type{}, std::integral_constant<uint32_t, K % P>{}, done >= (uint32_t)P, 0u, acc_a, acc_b);
                ++done;
                return false;
            };
            bool fin = run_tail<1, U>(step);         // the first trip starts at iteration 1
            while (!fin) fin = run_tail<0, U>(step);
            // the accumulator set filled last belongs to iteration done - 1
            if (done & 1u) drain(1u, acc_a); else drain(0u, acc_b);
            wait_vmcnt<0>();       // re-reads past the last tile may still be on their way into the ring
            __syncthreads();
            tile = q[1];           // where the sequence left the full tiles: n_full itself in the one block whose turn the partial tile is
            buf = 0u;
        }
    } else if (!ticket_job && tile < n_full) {
        if constexpr (ELEM == 2) {
            // General case (rows of fewer than 32 tokens or too far apart).  Iteration k: start the
            // loads of tile k+1, barrier (publishes buffer k, and everyone has finished reading buffer
            // k-1), compute and store tile k, then park tile k+1 into the other buffer.  Loads, stores
            // and the wait for the loads sit in one straight line, unpredicated: s_waitcnt vmcnt(#stores).
            issue_loads(std::true_type{}, tile);
            park(0u, 0u, pre);
            while (tile < n_full) {
                const uint32_t next = tile + tile_stride;
                issue_loads(std::true_type{}, next < n_full ? next : tile);
                __syncthreads();
                compute(buf, words, nrm);
                const uint32_t slot = tq_packed_slot(job, tile * 32u + n);
                store(job.idx_bytes + (size_t)slot * (8 * NB) + lane_slot, job.vec_norms + norm_slot(slot), words, nrm);
                buf ^= 1u;
                park(buf, buf, pre);
                tile = next;
            }
        } else {
            // fp32 elements, any rows: the same with the search of tile k-1 between the matrix instructions of tile k, from the other
            // accumulator set (sums of squares wait in three slots).  Six bf16 products a step keep the matrix pipe busy for a third of the
            // time, set-up and the first tile take another 4 us; the rest are waits of two waves a SIMD, the rotation's three terms leave no
            // registers for a third (nor for loads two tiles ahead: 32.5 us, spilled).  131168 vectors, 4-bit: 34.6 us while every wave
            // split the whole tile into its terms, now 31.5.
            const uint32_t m = (n_full - tile + tile_stride - 1u) / tile_stride;      // this block's full tiles
            auto only_one = [&]() __attribute__((always_inline)) {          // a small job: nothing to overlap
                issue_loads(std::true_type{}, tile);
                load_tables();
                park(0u, 0u, pre);
                __syncthreads();
                compute(0u, words, nrm);
                const uint32_t slot = tq_packed_slot(job, tile * 32u + n);
                store(job.idx_bytes + (size_t)slot * (8 * NB) + lane_slot, job.vec_norms + norm_slot(slot), words, nrm);
            };
            auto several = [&]() __attribute__((always_inline)) {
                TqTileWalk ahead(job, tile, tile_stride), done = ahead;
                const uint32_t first = wave * 8u + ld_vec;
                const long long own = (long long)first * job.token_stride + ld_piece * 16u;
                auto issue = [&]() { load_vector(job.states + ahead.offset(job, first, own)); };
                auto trip = [&](auto rot_tag, auto search_tag, uint32_t j, tq_f16v &acc_new, const tq_f16v &acc_old) {
                    constexpr bool ROT = decltype(rot_tag)::value, SEARCH = decltype(search_tag)::value;
                    const bool more = ROT && j + 1u < m;
                    if (more) {
                        ahead.next(job);
                        issue();
                    }
                    __syncthreads();        // tile j and its sums are parked, and nobody reads buffer (j + 1) & 1 any more
                    const uint8_t *stage = lds_stage[j & 1u];
                    Scale sc{};
                    if constexpr (SEARCH) sc = scale_of((j + 2u) % 3u);       // tile j-1 sits in slot (j-1) % 3
                    if constexpr (ROT) acc_new = tq_zero16();
                    Search z;
                    search_begin(z);
#pragma unroll
                    for (int s = 0; s < TQ_STEPS; ++s) {
                        if constexpr (ROT) rotate_step(stage, s, acc_new);
                        if constexpr (SEARCH) {
                            search_coord(z, 2 * s, acc_old, sc);
                            search_coord(z, 2 * s + 1, acc_old, sc);
                        }
                    }
                    if constexpr (SEARCH) {
                        search_end(z, words);
                        const uint32_t slot = done.slot(job, n);
                        store(job.idx_bytes + (size_t)slot * (8 * NB) + lane_slot, job.vec_norms + norm_slot(slot), words, sc.nrm);
                        done.next(job);
                    }
                    if (more) park((j + 1u) & 1u, (j + 1u) % 3u, pre);
                };
                using Y = std::true_type;
                using N = std::false_type;
                tq_f16v acc_a, acc_b;       // tiles with an even index rotate into acc_a, the others into acc_b
                issue();
                load_tables();
                park(0u, 0u, pre);
                trip(Y{}, N{}, 0u, acc_a, acc_a);
                uint32_t j = 1;
                for (; j + 1u < m; j += 2u) {
                    trip(Y{}, Y{}, j, acc_b, acc_a);
                    trip(Y{}, Y{}, j + 1u, acc_a, acc_b);
                }
                if (j < m) {
                    trip(Y{}, Y{}, j, acc_b, acc_a);
                    ++j;
                }
                if (m & 1u) trip(N{}, Y{}, m, acc_b, acc_a);        // the last tile's codes
                else trip(N{}, Y{}, m, acc_a, acc_b);
            };
            if (m == 1u) only_one(); else several();
            tile += m * tile_stride;
            __syncthreads();
        }
    }
    // the partial last tile of the job, if this block is the one whose turn it is
    if (tile == n_full && n_full < n_tiles) {
        issue_loads(std::false_type{}, tile);
        park(buf, buf, pre);
        __syncthreads();
        compute(buf, words, nrm);
        const uint32_t v = tile * 32u + n;
        if (v < job.n_vec) {
            const uint32_t slot = tq_packed_slot(job, v);
            store(job.idx_bytes + (size_t)slot * (8 * NB) + lane_slot, job.vec_norms + norm_slot(slot), words, nrm);
        }
    }
    report_done();
}

template <int DTYPE, int BITS>
__global__ __launch_bounds__(CTHREADS, InTraits<DTYPE>::MIN_WAVES) void tq_compress_kernel(TqDevJob job0, const tq_job *jobs, uint32_t *workspace,
                                                                                          uint32_t tshift, uint32_t paired) {
    const TqDevJob job = tq_uniform_job(tq_pair_job(tq_load_job(job0, jobs, blockIdx.y, InTraits<DTYPE>::ELEM), paired != 0u));
    compress_job<DTYPE, BITS>(job, TqBlock{blockIdx.x, gridDim.x}, workspace ? workspace + blockIdx.y * (TQ_WORKSPACE_BYTES_PER_JOB / 4) : nullptr,
                              tshift, paired);
}

// keys and values of a layer; their counters share one job's record of the workspace
template <int DTYPE>
__global__ __launch_bounds__(CTHREADS, InTraits<DTYPE>::MIN_WAVES) void tq_compress_layer_kernel(TqLayer l, uint32_t *workspace, uint32_t tshift, uint32_t paired) {
    const uint32_t which = tq_layer_job(l);
    const TqDevJob job = tq_uniform_job(tq_pair_job(which ? l.job[1] : l.job[0], paired != 0u));
    const TqBlock blk = tq_layer_block(l, which);
    uint32_t *counters = workspace ? workspace + which * (TQ_WORKSPACE_BYTES_PER_JOB / 8) : nullptr;
    switch (which ? l.bits[1] : l.bits[0]) {
        case 1: compress_job<DTYPE, 1>(job, blk, counters, tshift, paired); break;
        case 2: compress_job<DTYPE, 2>(job, blk, counters, tshift, paired); break;
        case 3: compress_job<DTYPE, 3>(job, blk, counters, tshift, paired); break;
        case 4: compress_job<DTYPE, 4>(job, blk, counters, tshift, paired); break;
        default: compress_job<DTYPE, 8>(job, blk, counters, tshift, paired); break;
    }
}

// ---- host side --------------------------------------------------------------------------

constexpr int MAX_DEVICES = 64;
std::mutex host_state_mutex;   // guards the per-device tables below (filled once per device, read often)

struct DeviceInfo {
    int dev = 0;
    int cus = 0;
    int lds_optin = 0;
};
int query_device(DeviceInfo &info) {
    static DeviceInfo cache[MAX_DEVICES];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= MAX_DEVICES) return TQ_ERR_NO_DEVICE;
    std::lock_guard<std::mutex> lock(host_state_mutex);
    if (cache[dev].cus == 0) {
        int cus = 0, lds = 0;
        e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e != hipSuccess) return (int)e;
        e = hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
        if (e != hipSuccess) return (int)e;
        cache[dev].dev = dev;
        cache[dev].lds_optin = lds;
        cache[dev].cus = cus > 0 ? cus : 1;
    }
    info = cache[dev];
    return 0;
}

#ifndef TQ_COMPRESS_TICKET_SHIFT
#define TQ_COMPRESS_TICKET_SHIFT 3
#endif

// Blocks of a kernel that are resident per compute unit (registers and LDS decide): a grid is that many per unit, each walking its share
// of the tiles.  Asked once per device; `resident_on` is the kernel's own.
template <typename K>
int resident_blocks(K kernel, const DeviceInfo &info, int (&resident_on)[MAX_DEVICES], int &resident) {
    std::lock_guard<std::mutex> lock(host_state_mutex);
    if (resident_on[info.dev] == 0) {
        int nb = 0;
        hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, CTHREADS, 0);
        if (e != hipSuccess) return (int)e;
        resident_on[info.dev] = nb > 0 ? nb : 1;
    }
    resident = resident_on[info.dev];
    return 0;
}

template <int DTYPE, int BITS>
int launch_compress(const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_tiles, void *workspace, bool paired, hipStream_t stream) {
    DeviceInfo info;
    int rc = query_device(info);
    if (rc) return rc;
    static int resident_on[MAX_DEVICES] = {};
    int resident;
    rc = resident_blocks(tq_compress_kernel<DTYPE, BITS>, info, resident_on, resident);
    if (rc) return rc;
    // Tickets from a counter pay off once every block has several to draw; below that (and without a workspace) the
    // blocks walk single tiles b, b + grid, ..., which splits a small job most evenly.
    uint32_t bx = tq_blocks_per_job(max_tiles, info.cus * resident, n_jobs);
    uint32_t tshift = 0;
    uint32_t *counters = nullptr;
    if (workspace && InTraits<DTYPE>::ELEM == 2 && TQ_COMPRESS_TICKET_SHIFT > 0) {
        const uint32_t tickets = (max_tiles + (1u << TQ_COMPRESS_TICKET_SHIFT) - 1u) >> TQ_COMPRESS_TICKET_SHIFT;
        const uint32_t bt = tq_blocks_per_job(tickets, info.cus * resident, n_jobs);
        if (tickets >= 4u * bt) {
            bx = bt;
            tshift = TQ_COMPRESS_TICKET_SHIFT;
            counters = static_cast<uint32_t *>(workspace);
        }
    }
    dim3 grid(bx, (unsigned)n_jobs, 1), block(CTHREADS, 1, 1);
    hipLaunchKernelGGL((tq_compress_kernel<DTYPE, BITS>), grid, block, 0, stream, job, jobs_dev, counters, tshift, paired ? 1u : 0u);
    return (int)hipGetLastError();
}

template <int DTYPE>
int launch_layer(TqLayer &l, uint32_t tiles, void *workspace, bool paired, hipStream_t stream) {
    DeviceInfo info;
    int rc = query_device(info);
    if (rc) return rc;
    static int resident_on[MAX_DEVICES] = {};
    int resident;
    rc = resident_blocks(tq_compress_layer_kernel<DTYPE>, info, resident_on, resident);
    if (rc) return rc;
    const uint32_t slots = (uint32_t)(info.cus * resident);
    uint32_t blocks = tq_layer_blocks(l, tiles, slots), tshift = 0;
    uint32_t *counters = nullptr;
    if (workspace && InTraits<DTYPE>::ELEM == 2 && TQ_COMPRESS_TICKET_SHIFT > 0) {       // as in launch_compress
        const uint32_t tickets = (tiles + (1u << TQ_COMPRESS_TICKET_SHIFT) - 1u) >> TQ_COMPRESS_TICKET_SHIFT;
        if (2u * tickets >= 4u * slots) {
            blocks = tq_layer_blocks(l, tickets, slots);
            tshift = TQ_COMPRESS_TICKET_SHIFT;
            counters = static_cast<uint32_t *>(workspace);
        }
    }
    hipLaunchKernelGGL((tq_compress_layer_kernel<DTYPE>), dim3(blocks), dim3(CTHREADS), 0, stream, l, counters, tshift, paired ? 1u : 0u);
    return (int)hipGetLastError();
}

template <int DTYPE>
int dispatch_bits(int bits, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_tiles, void *ws, bool paired, hipStream_t s) {
    switch (bits) {
        case 1: return launch_compress<DTYPE, 1>(job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case 2: return launch_compress<DTYPE, 2>(job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case 3: return launch_compress<DTYPE, 3>(job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case 4: return launch_compress<DTYPE, 4>(job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case 5: case 6: case 7: case 8:  // one code per byte: identical packing
            return launch_compress<DTYPE, 8>(job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        default: return TQ_ERR_BITS;
    }
}

int dispatch(int dtype, int bits, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_tiles, void *ws, bool paired, hipStream_t s) {
    switch (dtype) {
        case TQ_F32: return dispatch_bits<TQ_F32>(bits, job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case TQ_F16: return dispatch_bits<TQ_F16>(bits, job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        case TQ_BF16: return dispatch_bits<TQ_BF16>(bits, job, jobs_dev, n_jobs, max_tiles, ws, paired, s);
        default: return TQ_ERR_DTYPE;
    }
}

int elem_bytes(int dtype) { return dtype == TQ_F32 ? 4 : (dtype == TQ_F16 || dtype == TQ_BF16) ? 2 : 0; }

// Shared argument checks of one job; fills n_vec.
int check_job(const void *states, int dtype, long long rows, long long tokens, long long row_stride,
              long long token_stride, const void *table, int head_dim, int bits, const void *idx_bytes,
              const void *vec_norms, long long packed_row_stride, long long *n_vec) {
    if (bits < 1 || bits > 8) return TQ_ERR_BITS;
    if (head_dim != TQ_HEAD_DIM && !tq_anydim_supported(head_dim)) return TQ_ERR_HEAD_DIM;
    const int eb = elem_bytes(dtype);
    if (!eb) return TQ_ERR_DTYPE;
    if (rows < 0 || tokens < 0) return TQ_ERR_SIZE;
    if (rows != 0 && tokens > (long long)0x7fffffff / rows) return TQ_ERR_SIZE;
    *n_vec = rows * tokens;
    if (*n_vec == 0) return TQ_OK;
    if (!states || !table || !idx_bytes || !vec_norms) return TQ_ERR_NULL;
    if (token_stride < head_dim && tokens > 1) return TQ_ERR_SIZE;
    if (rows > 1 && row_stride < 0) return TQ_ERR_SIZE;
    if (packed_row_stride != 0 && (packed_row_stride < tokens || packed_row_stride > (long long)0x7fffffff / rows)) return TQ_ERR_SIZE;
    const uintptr_t va = tq_vector_alignment(head_dim, eb) - 1u;
    if (((uintptr_t)states & va) || ((uintptr_t)table & 15u) || ((uintptr_t)idx_bytes & (tq_packed_alignment(head_dim, bits) - 1u)) || ((uintptr_t)vec_norms & 1u))
        return TQ_ERR_ALIGN;
    if (((uintptr_t)(token_stride * eb) & va) || (rows > 1 && ((uintptr_t)(row_stride * eb) & va))) return TQ_ERR_ALIGN;
    return TQ_OK;
}

}  // namespace

extern "C" int tq_compress(const void *states, int dtype, long long rows, long long tokens,
                           long long row_stride, long long token_stride, const void *table_dev,
                           int head_dim, int bits, uint8_t *idx_bytes, uint16_t *vec_norms,
                           long long packed_row_stride, void *workspace, void *stream) {
    long long n_vec = 0;
    const int rc = check_job(states, dtype, rows, tokens, row_stride, token_stride, table_dev, head_dim, bits,
                             idx_bytes, vec_norms, packed_row_stride, &n_vec);
    if (rc) return rc;
    if ((uintptr_t)workspace & 63u) return TQ_ERR_ALIGN;
    if (n_vec == 0) return TQ_OK;
    TqDevJob job;
    job.states = static_cast<const uint8_t *>(states);
    job.idx_bytes = idx_bytes;
    job.vec_norms = vec_norms;
    job.table = static_cast<const uint8_t *>(table_dev);
    job.n_vec = (uint32_t)n_vec;
    job.tokens = (uint32_t)tokens;
    job.packed_row_stride = (uint32_t)(packed_row_stride ? packed_row_stride : tokens);
    job.row_stride = row_stride * elem_bytes(dtype);
    job.token_stride = token_stride * elem_bytes(dtype);
    if (head_dim == TQ_HEAD_DIM / 2 && tq_pairable(rows, tokens, token_stride, packed_row_stride, head_dim, idx_bytes))
        return dispatch(dtype, bits, job, nullptr, 1, (uint32_t)((n_vec / 2 + 31) / 32), workspace, true, static_cast<hipStream_t>(stream));
    if (head_dim != TQ_HEAD_DIM)
        return tq_anydim_compress(dtype, bits, head_dim, job, nullptr, 1, (uint32_t)n_vec, static_cast<hipStream_t>(stream));
    return dispatch(dtype, bits, job, nullptr, 1, (uint32_t)((n_vec + 31) / 32), workspace, false, static_cast<hipStream_t>(stream));
}

extern "C" int tq_compress_layer(const void *keys, const void *values, int dtype, long long rows, long long tokens, long long row_stride, long long token_stride,
                                 const void *table_k, const void *table_v, int head_dim, int bits_k, int bits_v, uint8_t *k_idx, uint16_t *k_norms,
                                 uint8_t *v_idx, uint16_t *v_norms, void *workspace, void *stream) {
    long long n_vec = 0;
    int rc = check_job(keys, dtype, rows, tokens, row_stride, token_stride, table_k, head_dim, bits_k, k_idx, k_norms, 0, &n_vec);
    if (!rc) rc = check_job(values, dtype, rows, tokens, row_stride, token_stride, table_v, head_dim, bits_v, v_idx, v_norms, 0, &n_vec);
    if (rc) return rc;
    if ((uintptr_t)workspace & 63u) return TQ_ERR_ALIGN;
    if (n_vec == 0) return TQ_OK;
    const bool paired = tq_pairable(rows, tokens, token_stride, 0, head_dim, k_idx) && tq_pairable(rows, tokens, token_stride, 0, head_dim, v_idx);
    if (head_dim == TQ_HEAD_DIM || paired || tq_anydim_layer_supported(head_dim, dtype)) {
        const int eb = elem_bytes(dtype);
        TqLayer l{};
        for (int i = 0; i < 2; ++i) {
            TqDevJob &job = l.job[i];
            job.states = static_cast<const uint8_t *>(i ? values : keys);
            job.idx_bytes = i ? v_idx : k_idx;
            job.vec_norms = i ? v_norms : k_norms;
            job.table = static_cast<const uint8_t *>(i ? table_v : table_k);
            job.n_vec = (uint32_t)n_vec;
            job.tokens = job.packed_row_stride = (uint32_t)tokens;
            job.row_stride = row_stride * eb;
            job.token_stride = token_stride * eb;
            l.bits[i] = i ? bits_v : bits_k;
        }
        const hipStream_t s = static_cast<hipStream_t>(stream);
        if (head_dim != TQ_HEAD_DIM && !paired) return tq_anydim_compress_layer(dtype, head_dim, l, (uint32_t)n_vec, s);
        const uint32_t tiles = (uint32_t)(((paired ? n_vec / 2 : n_vec) + 31) / 32);
        switch (dtype) {
            case TQ_F32: return launch_layer<TQ_F32>(l, tiles, workspace, paired, s);
            case TQ_F16: return launch_layer<TQ_F16>(l, tiles, workspace, paired, s);
            default: return launch_layer<TQ_BF16>(l, tiles, workspace, paired, s);
        }
    }
    rc = tq_compress(keys, dtype, rows, tokens, row_stride, token_stride, table_k, head_dim, bits_k, k_idx, k_norms, 0, workspace, stream);
    if (rc) return rc;
    return tq_compress(values, dtype, rows, tokens, row_stride, token_stride, table_v, head_dim, bits_v, v_idx, v_norms, 0, workspace, stream);
}

extern "C" int tq_compress_batched(const tq_job *jobs_host, const tq_job *jobs_dev, int n_jobs,
                                   int head_dim, void *workspace, void *stream) {
    if (n_jobs == 0) return TQ_OK;
    if (!jobs_host || !jobs_dev) return TQ_ERR_NULL;
    if (n_jobs < 0 || n_jobs > TQ_MAX_JOBS) return TQ_ERR_SIZE;
    if ((uintptr_t)workspace & 63u) return TQ_ERR_ALIGN;
    long long max_vec = 0;
    bool paired = head_dim == TQ_HEAD_DIM / 2;     // 64-wide vectors in pairs, if every job of the launch allows it
    for (int i = 0; i < n_jobs; ++i) {
        const tq_job &j = jobs_host[i];
        if (j.bits != jobs_host[0].bits) return TQ_ERR_BITS;
        if (j.dtype != jobs_host[0].dtype) return TQ_ERR_DTYPE;
        long long n_vec = 0;
        const int rc = check_job(j.states, j.dtype, j.rows, j.tokens, j.row_stride, j.token_stride, j.table_dev,
                                 head_dim, j.bits, j.idx_bytes, j.vec_norms, j.packed_row_stride, &n_vec);
        if (rc) return rc;
        if (n_vec > max_vec) max_vec = n_vec;
        if (n_vec && !tq_pairable(j.rows, j.tokens, j.token_stride, j.packed_row_stride, head_dim, j.idx_bytes)) paired = false;
    }
    if (max_vec == 0) return TQ_OK;
    TqDevJob none{};
    if (paired)
        return dispatch(jobs_host[0].dtype, jobs_host[0].bits, none, jobs_dev, n_jobs, (uint32_t)((max_vec / 2 + 31) / 32),
                        workspace, true, static_cast<hipStream_t>(stream));
    if (head_dim != TQ_HEAD_DIM)
        return tq_anydim_compress(jobs_host[0].dtype, jobs_host[0].bits, head_dim, none, jobs_dev, n_jobs, (uint32_t)max_vec,
                                  static_cast<hipStream_t>(stream));
    return dispatch(jobs_host[0].dtype, jobs_host[0].bits, none, jobs_dev, n_jobs, (uint32_t)((max_vec + 31) / 32),
                    workspace, false, static_cast<hipStream_t>(stream));
}
