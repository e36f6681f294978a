// The matrix-core launches for the layer driver, which knows more than their entry points take: of the segments, whose table it
// made, and of what runs beside a launch. Arguments and results as the dgpp_launch_moe_grouped_mma_* and _w4a4_* entry points.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "../../include/dgpp_amd.h"

namespace dgpp_amd {

struct SegmentRows {
  int max_rows;            // no segment has more
  int64_t total_rows = 0;  // of all segments, 0: not known
  int long_segs = 0;       // so many segments at the table's end have exactly max_rows (a shared expert's)
};

// fp4_group: 0 block FP8, 16 NVFP4, 32 MXFP4. gate_up_limit: null, or gate + up + SwiGLU (`which` 0).
int grouped_mma(int fp4_group, const uint16_t* act, size_t act_stride, const DgppMoeSegment* segs, int n_segs,
                const SegmentRows& rows, const DgppMoeExpertView* views, int which, void* out, int out_f32, size_t out_stride,
                int n, int k, void* stream, const int32_t* act_rows, const float* gate_up_limit);
int grouped_w4a4(const uint8_t* codes, const uint8_t* scales, const float* gs, const int32_t* act_rows,
                 const DgppMoeSegment* segs, int n_segs, const SegmentRows& rows, const DgppMoeExpertView* views, int which,
                 void* out, int out_f32, size_t out_stride, int n, int k, void* stream);

// A projection with MXFP8 weights (one scale byte per 32 values). beside: other work fills the chip meanwhile.
int scale_gemm_mxfp8(const uint16_t* act, size_t act_stride, const uint8_t* payload, const uint8_t* scales, void* out, int out_f32,
                     int m, int n, int k, void* stream, void* ws, size_t ws_bytes, bool beside);

}  // namespace dgpp_amd
