// Launches shared between the library's translation units (host side): the
// write path as one call (lq_encode_chunks) is made of them.
#pragma once

#include "latticequant_amd.h"

namespace lq {

// Words cleared on the side by the first launch of a write: the histograms,
// the chunks' status words and one counter.
struct Clear {
    uint32_t* hist = nullptr;
    int64_t n_hist = 0;
    int32_t* status = nullptr;
    int64_t n_status = 0;
    uint32_t* counter = nullptr;
};

// lq_head_scales (signs null) or lq_head_scales_rht
int head_scales_launch(const void* x, int dtype, int64_t n_chunks, int64_t n_heads, int64_t bph, int head_dim,
                       const float* signs, const int32_t* bits, double* work, float* sigma2, float* scale32,
                       uint16_t* scale16, int32_t* fastdiv, const Clear& clear, hipStream_t s);

// lq_scale_fastdiv, and the fp16 copies of the scales (scale16 nullable)
int scale_fastdiv_launch(const float* scale32, int64_t n, int dtype, int32_t* fastdiv, uint16_t* scale16,
                         const Clear& clear, hipStream_t s);

}  // namespace lq
