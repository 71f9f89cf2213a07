// Entry points of the codec kernels for the head dimensions 96, 160, 192 and 224 with 16-bit elements
// (tq_wide.hip, kernels in tq_wide_kernel.h), called by the dispatchers of tq_anydim.hip.  Arguments as there: `single` describes the one job of a
// plain call (jobs_dev NULL), `jobs_dev` the device copy of a batch.
#pragma once
#include "tq_device.h"

bool tq_wide_supported(int head_dim, int dtype);
int tq_wide_compress(int dtype, int bits, int head_dim, const TqDevJob &single, const tq_job *jobs_dev, int n_jobs,
                     uint32_t max_vec, hipStream_t stream);
int tq_wide_decompress(int dtype, int bits, int head_dim, const TqDevJob &single, const tq_job *jobs_dev, int n_jobs,
                       uint32_t max_vec, hipStream_t stream);
// keys and values of a layer in one launch (TqLayer: everything but `split` filled in)
int tq_wide_compress_layer(int dtype, int head_dim, TqLayer &l, uint32_t n_vec, hipStream_t stream);
int tq_wide_restore_layer(int dtype, int head_dim, TqLayer &l, const TqWindowCopy &w, uint32_t n_vec, hipStream_t stream);

// The same for one padded dimension each (tq_wide_d96.hip ... tq_wide_d224.hip), `dl` of whose coordinates a vector has; arguments checked above.
#define TQ_WIDE_DECLARE(D)                                                                                                                       \
    int tq_wide_compress_d##D(int dtype, int bits, uint32_t dl, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec,       \
                              hipStream_t s);                                                                                                   \
    int tq_wide_decompress_d##D(int dtype, int bits, uint32_t dl, const TqDevJob &job, const tq_job *jobs_dev, int n_jobs, uint32_t max_vec,     \
                                hipStream_t s);                                                                                                 \
    int tq_wide_compress_layer_d##D(int dtype, uint32_t dl, TqLayer &l, uint32_t n_vec, hipStream_t s);        \
    int tq_wide_restore_layer_d##D(int dtype, uint32_t dl, TqLayer &l, const TqWindowCopy &w, uint32_t n_vec,  \
                                   hipStream_t s);
TQ_WIDE_DECLARE(96)
TQ_WIDE_DECLARE(160)
TQ_WIDE_DECLARE(192)
TQ_WIDE_DECLARE(224)
#undef TQ_WIDE_DECLARE
