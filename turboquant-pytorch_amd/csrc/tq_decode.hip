// One decode step of a streaming cache layer in two launches, for head dimensions 64, 96, 128 and 256 and 16-bit elements:
//   tq_decode_append   the token that leaves the window is compressed into the next packed slot and the new token takes its
//                      window slot, keys and values, every row, in one launch;
//   tq_decode_attend   softmax(scale q K^T) V over the packed history and the uncompressed window, one launch: the queries are
//                      rotated, the window is attended to and the splits are merged inside the kernel that reads the codes.
// Few rows: a step is a chain of latencies (tables, query rotation, one or two runs per wave, merge), so launches are what
// counts; many rows: the main loop, which is bound by the vector and LDS work of the table lookups.
// Per layer and whole step, six launches / these two (MI355X): 8 rows x 32768 tokens, K4/V2, 4 heads a row 48.9 -> 22.5 us;
// 512 rows x 16384 tokens 226 -> 175 us, of which attention 170; head dimension 64, 32 rows x 6000 tokens, K6/V4 (before:
// de-quantised to float32 and multiplied by library products) 190 -> 18.7 us.
// What they compute is what tq_compress and the prepare / partials / merge trio of tq_attend.hip compute (upstream
// turboquant/generation_test_v2.py:96-135, score definition validate_v3.py:87); at 128 those remain for float32 caches, queries of
// another type than the cache's and more than 65535 rows.  A value whose norm is infinite in float16 makes its row's results NaN, as there.
#include <type_traits>

#include "tq_decode.h"

namespace {

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

// Block (32 rows, tensor, w): one wave, which produces the rotated coordinates [32 w, 32 w + 32) of 32 vectors, one per row, and their
// codes.  A step has one vector per row, so nothing is reused and the launch lasts as long as its chain of loads: everything a
// wave reads (vectors, operands, the quantiser's grid, its share of the new tokens) is asked for before anything is waited for, sections of the
// tables at the places every table has them, and the cells then come from LDS.  A wave each, since four waves of 30 loads share a compute
// unit's one load pipe, and a launch has few blocks anyway.  (Blocks of D / 32 waves that took the header, the new tokens, the vectors
// and the cells one after the other / this, append and attend of a layer, us: 8 rows x 32768 tokens at 128 24.7 / 22.5, 32 x 6000 at 64 20.8 / 18.7.)
// Products and sums run in the order of the kernels that compress
// whole tensors of this head dimension, so the bytes are theirs.
template <int D, bool BF>
__global__ __launch_bounds__(TQ_WAVE) void tq_decode_append_kernel(AppendArgs a) {
    constexpr int STEPS = D / 16;
    constexpr int CELL_LOADS = (D == 128 ? TQ_GRID_COPY_STRIDE(8) : TQ_GRID_LDS_BYTES) / 1024;      // 128: the grids fit two copies at least
    static_assert(CELL_LOADS * 1024 == (D == 128 ? TQ_GRID_COPY_STRIDE(8) : TQ_GRID_LDS_BYTES), "whole loads of a wave");
    __shared__ __align__(16) uint8_t lds_grid[CELL_LOADS * 1024];
    const uint32_t lane = threadIdx.x, which = blockIdx.y, wave = blockIdx.z;
    const uint32_t n = lane & 31u, hk = lane >> 5;
    const uint32_t row0 = blockIdx.x * 32u;
    uint8_t *win = a.win[which];
    // the new tokens, 64 bytes of each row to a wave: to another slot than the one read below
    tq_u4 fresh[2];
    uint32_t fresh_row[2];
    const uint32_t fresh_piece = 4u * wave + (lane & 3u);
    auto load_fresh = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            fresh_row[i] = row0 + 16u * i + (lane >> 2);
            fresh[i] = tq_gload16(a.fresh[which] + (size_t)min(fresh_row[i], a.rows - 1u) * a.new_stride[which] * 2u + fresh_piece * 16u);
        }
    };
    auto store_fresh = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            if (fresh_row[i] < a.rows) tq_gstore16(win + ((size_t)fresh_row[i] * a.win_stride + (size_t)a.put * D) * 2u + fresh_piece * 16u, fresh[i]);
    };
    if (!a.compress) {
        load_fresh();
        store_fresh();
        return;
    }
    const uint8_t *table = a.table[which];
    const TqTableHeader *hd = reinterpret_cast<const TqTableHeader *>(table);
    const uint32_t r = min(row0 + n, a.rows - 1u);
    const uint8_t *src = win + ((size_t)r * a.win_stride + (size_t)a.evict * D) * 2u + 16u * hk;
    const uint8_t *asrc = table + (BF ? TQ_OFF_A_BF16(D) : TQ_OFF_A_F16) + ((size_t)wave * STEPS * 64u + lane) * 16u;
    const uint32_t step0 = D == 128 ? 2u * wave : 0u;      // the 128-wide kernel starts the contraction at the wave's own quarter
    tq_u4 x[STEPS], p[2][STEPS], cells[CELL_LOADS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        const uint32_t sg = D == 128 ? (s + step0) & 7u : (uint32_t)s;
        x[s] = tq_gload16(src + 32u * sg);
#pragma unroll
        for (int t = 0; t < 2; ++t) p[t][s] = tq_gload16(asrc + t * TQ_OPERAND_BYTES_FOR(D) + (size_t)sg * 1024u);
    }
#pragma unroll
    for (int i = 0; i < CELL_LOADS; ++i) cells[i] = tq_gload16(table + TQ_OFF_GRID(D) + 1024u * i + 16u * lane);
    load_fresh();
    const float grid_scale = hd->grid_scale, grid_bias = hd->grid_bias;
    const uint32_t width = hd->bits;
    __builtin_amdgcn_sched_barrier(0);
    tq_f16v acc = tq_zero16();
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc = BF ? mfma_bf16(p[t][s], x[s], acc) : mfma_f16(p[t][s], x[s], acc);
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
        // share[q] is that of quarter q + w: the pairs (0, 1) and (2, 3) of the vector's quarters
        ss = wave & 1u ? (share[3] + share[0]) + (share[1] + share[2]) : (share[0] + share[1]) + (share[2] + share[3]);
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
    const float inv_cell = inv * grid_scale;
    // ---- code search: lane (n, hk) holds coordinates 32 w + 16 hk + r
#pragma unroll
    for (int i = 0; i < CELL_LOADS; ++i) *reinterpret_cast<tq_u4 *>(lds_grid + 1024u * i + 16u * lane) = cells[i];
    __syncthreads();      // (one wave: the order of its own LDS accesses)
    tq_u2 cell[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) cell[q] = *reinterpret_cast<const tq_u2 *>(lds_grid + (__float_as_uint(fmaf(acc[q], inv_cell, grid_bias)) & TQ_GRID_ADDR_MASK));
    uint32_t code[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) code[q] = cell[q][1] + (~__float_as_uint(fmaf(acc[q], inv, -__uint_as_float(cell[q][0]))) >> 31);
    store_fresh();
    if (row0 + n >= a.rows) return;
    const int ipb = a.ipb[which];
    const size_t slot = (size_t)r * a.packed_row_stride;
    uint8_t *dst = a.idx[which] + slot * (uint32_t)(D / ipb) + (2u * wave + hk) * (uint32_t)(16 / ipb);
    auto pack = [&](auto ipb_tag) __attribute__((always_inline)) {       // most significant code of a byte first
        constexpr int I = decltype(ipb_tag)::value, BITS = 8 / I, NB = 16 / I, NW = NB < 4 ? 1 : NB / 4;
        uint32_t w[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) w[k] = 0u;
        // 3-bit codes sit two to a byte, three bits apart
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

template <int D>
void launch_append(dim3 grid, hipStream_t s, const AppendArgs &a) {
    const dim3 block(TQ_WAVE);
    if (a.bf16) hipLaunchKernelGGL((tq_decode_append_kernel<D, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((tq_decode_append_kernel<D, false>), grid, block, 0, s, a);
}

// Packed histories are read with the non-temporal hint (see launch_decode) where the cache cannot stay in the last-level cache, 256 MiB, from one step
// to the next: from 224 MiB on that a step reads, packed store and windows of all layers.  us of plain loads / with the hint, a step with
// its appends, 128 wide and 8 rows unless stated: 16 layers of K4/V2 at 158 MiB 252 / 258, 200 273 / 278, 232 281 / 279, 360 300 / 295; 32 layers at
// 144 473 / 492, 208 486 / 491, 240 514 / 511, 528 593 / 556; 16 of 6289 tokens, K6/V4, at 158 267 / 275; 32 x 3932 tokens at 64, K6/V4,
// 16 layers at 208 233 / 236, 32 x 5242 at 272 248 / 242; 256 wide, 16 layers at 192 504 / 509, 32 layers at 256 1035 / 987; 128 rows x 655 tokens, half
// of it windows, 16 layers at 256 291 / 281.  Of 291 sizes drawn 4 lose more than 1 % by this line, of 224 MiB of packed store alone 28, of 8 MiB
// a layer 53.  A caller that names no cache is taken to have sixteen layers like this one.
constexpr long long CACHE_STREAMED = 224ll << 20, LAYER_STREAMED = CACHE_STREAMED / 16;

// splits of the token range per row
int decode_splits(long long rows, long long tokens) {
    if (rows <= 0 || tokens <= 0) return 1;
    int cus = 0;
    if (tq_device_cus(cus)) cus = 256;
    // One block is resident per compute unit.  A launch takes as many rounds of blocks as rows * splits fill the chip, each as
    // long as a block's tokens plus about what 2000 tokens take for tables, query rotation and result, and 400 more where the splits
    // of a row have to be merged; every record to merge counts like 12 tokens.  Blocks of less than 192 tokens gain nothing.
    // (Best of a sweep / what this rule takes, us a layer with its append, K4/V2: 8 x 32768 tokens 19.1 / 19.1 with 32 splits, 21.1 with 16 and 26.2
    // with 48; 2 x 8738 14.0 / 14.0; 32 x 6000 at 64, K6/V4, 15.8 / 15.8 with 8, 18.0 with 4; 128 x 4182, K3/V2, 24.6 with 2, 29.3 with 1, 33.1
    // with 4; off the best 8 x 6289, K6/V4, 16.0 with 32 / 17.0 with 22 and 2 x 8574 at 96, K6/V4, 13.6 with 39 / 14.3 with 26.  A launch alone, when it was
    // some 2 us longer: 8 x 1024 12.0 / 12.4, 14.9 in one split; 160 x 6000 34.6 / 34.6 in one split, 40.4 with 3.)
    long long most = (tokens + 191) / 192;
    if (most > MAX_SPLITS) most = MAX_SPLITS;
    long long best = 1, best_cost = 0;
    for (long long s = 1; s <= most; ++s) {
        const long long rounds = (rows * s + cus - 1) / cus;
        const long long cost = rounds * ((tokens + s - 1) / s + 2000 + (s > 1 ? 400 : 0)) + 12 * s;
        if (s == 1 || cost < best_cost) { best = s; best_cost = cost; }
        if (rounds > 16 && s > 1) break;
    }
    return (int)best;
}

// Whether the packed history is read with the non-temporal hint (what it does: see launch_decode).
bool streams(const tq_decode_layer *l, long long tokens, long long n_win, long long cache_bytes) {
    const long long slot = l->head_dim / (8 / l->bits_k) + l->head_dim / (8 / l->bits_v) + 4, layer = l->rows * (tokens * slot + n_win * l->head_dim * 4);
    return cache_bytes > 0 ? cache_bytes >= CACHE_STREAMED : layer >= LAYER_STREAMED;
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
    return scratch_floats(rows, group, head_dim, decode_splits(rows, tokens), n_win) + 1;      // (see tq_decode_attend)
}

extern "C" int tq_decode_streams(const tq_decode_layer *layer, long long tokens, long long n_win, long long cache_bytes) {
    const int rc = check_layer(layer);
    if (rc) return rc;
    if (tokens < 0 || tokens > 0x7fffffff || n_win < 0 || n_win > MAX_WINDOW) return TQ_ERR_SIZE;
    return streams(layer, tokens, n_win, cache_bytes) ? 1 : 0;
}

extern "C" int tq_decode_attend_cached(const tq_decode_layer *layer, const void *queries, int group, float scale, long long win_first, long long n_win,
                                       long long tokens, float *scratch, long long scratch_size, uint32_t *arrived, long long n_arrived,
                                       long long cache_bytes, void *out, void *stream) {
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
    // records are stored and exchanged between blocks in pairs of floats, 8 bytes at a time
    if ((uintptr_t)scratch & 4u) { ++scratch; --scratch_size; }
    if (scratch_size < scratch_floats(rows, group, D, splits, n_win) || n_arrived < rows) return TQ_ERR_CAPACITY;
    TqDecodeArgs a;
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
    // A counter of its own to every line of 128 bytes where there are enough of them (closer together where there are fewer): the blocks
    // that finish together would otherwise queue at one line, an atomic about every 14 ns.
    a.arrived_stride = 32u;
    while (a.arrived_stride > 1u && (long long)a.arrived_stride * rows > n_arrived) a.arrived_stride >>= 1;
    a.out = static_cast<uint8_t *>(out);
    a.win_stride = layer->win_stride;
    a.scale = scale;
    a.tokens = (uint32_t)tokens;
    a.packed_row_stride = (uint32_t)layer->packed_row_stride;
    a.group = (uint32_t)group;
    a.chunk = (uint32_t)(((tokens + splits - 1) / splits + 15) / 16 * 16);
    a.n_win = (uint32_t)n_win;
    a.bf16 = layer->dtype == TQ_BF16 ? 1u : 0u;
    a.stream = streams(layer, tokens, n_win, cache_bytes) ? 1u : 0u;
    if (!tokens) {       // no history: the loads that every wave starts with find the tables instead, and nothing is done with them
        a.k_idx = a.table_k; a.v_idx = a.table_v;
        a.k_norms = reinterpret_cast<const uint16_t *>(a.table_k); a.v_norms = reinterpret_cast<const uint16_t *>(a.table_v);
        a.packed_row_stride = 0;
    }
    const dim3 grid((unsigned)splits, (unsigned)rows, 1);
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const int ik = 8 / layer->bits_k, iv = 8 / layer->bits_v;
    switch (D) {
        case 64: return tq_decode_launch_d64(ik, iv, grid, s, a);
        case 96: return tq_decode_launch_d96(ik, iv, grid, s, a);
        case 128: return ik >= 4 ? tq_decode_launch_d128_narrow(ik, iv, grid, s, a) : tq_decode_launch_d128_wide(ik, iv, grid, s, a);
        default: return tq_decode_launch_d256(ik, iv, grid, s, a);
    }
}

extern "C" int tq_decode_attend_spread(const tq_decode_layer *layer, const void *queries, int group, float scale, long long win_first, long long n_win,
                                       long long tokens, float *scratch, long long scratch_size, uint32_t *arrived, long long n_arrived, void *out,
                                       void *stream) {
    return tq_decode_attend_cached(layer, queries, group, scale, win_first, n_win, tokens, scratch, scratch_size, arrived, n_arrived, 0, out, stream);
}

extern "C" int tq_decode_attend(const tq_decode_layer *layer, const void *queries, int group, float scale, long long win_first, long long n_win,
                                long long tokens, float *scratch, long long scratch_size, uint32_t *arrived, void *out, void *stream) {
    return tq_decode_attend_cached(layer, queries, group, scale, win_first, n_win, tokens, scratch, scratch_size, arrived, layer ? layer->rows : 0, 0, out, stream);
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
    const dim3 grid((unsigned)((rows + 31) / 32), 2, (unsigned)(D / 32));
    const hipStream_t s = static_cast<hipStream_t>(stream);
    switch (D) {
        case 64: launch_append<64>(grid, s, a); break;
        case 96: launch_append<96>(grid, s, a); break;
        case 128: launch_append<128>(grid, s, a); break;
        default: launch_append<256>(grid, s, a); break;
    }
    return (int)hipGetLastError();
}
