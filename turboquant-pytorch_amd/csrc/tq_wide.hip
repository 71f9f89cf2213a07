// Which source of the kernels in tq_wide_kernel.h a head dimension goes to: 65 to 96, 129 to 224, 16-bit elements.
#include "tq_wide.h"

bool tq_wide_supported(int head_dim, int dtype) {
    const int padded = TQ_PADDED_DIM(head_dim);      // 65 ... 96, 129 ... 224
    return (dtype == TQ_F16 || dtype == TQ_BF16) && head_dim >= 8 && (padded == 96 || padded == 160 || padded == 192 || padded == 224);
}

int tq_wide_compress(int dtype, int bits, int head_dim, const TqDevJob &single, const tq_job *jobs_dev, int n_jobs,
                     uint32_t max_vec, hipStream_t stream) {
    if (!tq_wide_supported(head_dim, dtype)) return TQ_ERR_HEAD_DIM;
    if (bits < 1 || bits > 8) return TQ_ERR_BITS;
    const uint32_t dl = (uint32_t)head_dim;
    switch (TQ_PADDED_DIM(head_dim)) {
        case 96: return tq_wide_compress_d96(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        case 160: return tq_wide_compress_d160(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        case 192: return tq_wide_compress_d192(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        default: return tq_wide_compress_d224(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
    }
}

int tq_wide_decompress(int dtype, int bits, int head_dim, const TqDevJob &single, const tq_job *jobs_dev, int n_jobs,
                       uint32_t max_vec, hipStream_t stream) {
    if (!tq_wide_supported(head_dim, dtype)) return TQ_ERR_HEAD_DIM;
    if (bits < 1 || bits > 8) return TQ_ERR_BITS;
    const uint32_t dl = (uint32_t)head_dim;
    switch (TQ_PADDED_DIM(head_dim)) {
        case 96: return tq_wide_decompress_d96(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        case 160: return tq_wide_decompress_d160(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        case 192: return tq_wide_decompress_d192(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
        default: return tq_wide_decompress_d224(dtype, bits, dl, single, jobs_dev, n_jobs, max_vec, stream);
    }
}

int tq_wide_compress_layer(int dtype, int head_dim, TqLayer &l, uint32_t n_vec, hipStream_t stream) {
    if (!tq_wide_supported(head_dim, dtype)) return TQ_ERR_HEAD_DIM;
    const uint32_t dl = (uint32_t)head_dim;
    switch (TQ_PADDED_DIM(head_dim)) {
        case 96: return tq_wide_compress_layer_d96(dtype, dl, l, n_vec, stream);
        case 160: return tq_wide_compress_layer_d160(dtype, dl, l, n_vec, stream);
        case 192: return tq_wide_compress_layer_d192(dtype, dl, l, n_vec, stream);
        default: return tq_wide_compress_layer_d224(dtype, dl, l, n_vec, stream);
    }
}

int tq_wide_restore_layer(int dtype, int head_dim, TqLayer &l, const TqWindowCopy &w, uint32_t n_vec, hipStream_t stream) {
    if (!tq_wide_supported(head_dim, dtype)) return TQ_ERR_HEAD_DIM;
    const uint32_t dl = (uint32_t)head_dim;
    switch (TQ_PADDED_DIM(head_dim)) {
        case 96: return tq_wide_restore_layer_d96(dtype, dl, l, w, n_vec, stream);
        case 160: return tq_wide_restore_layer_d160(dtype, dl, l, w, n_vec, stream);
        case 192: return tq_wide_restore_layer_d192(dtype, dl, l, w, n_vec, stream);
        default: return tq_wide_restore_layer_d224(dtype, dl, l, w, n_vec, stream);
    }
}
