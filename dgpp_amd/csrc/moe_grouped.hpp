// Launches for the layer driver, which knows more than their entry points take: of the segments, whose table it made, and of what
// runs beside a launch. Arguments and results as the dgpp_launch_moe_grouped_mma_* and _w4a4_* entry points.
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

// The routed experts and a block-FP8 shared expert of a small decode batch, a launch per pass: gate + up + SwiGLU (with scores, the
// selection of a one-token step too), then down and the tokens' accumulation. Bit for bit the launches they stand for. DGPP_OK and
// taken false: the call is not of that form or would be refused, and nothing was launched. ask: only whether it is of that form.
struct SharedExpert {
  const uint8_t* payload[3];
  const float* scales[3];
  int inter, rs, cs;
};
struct RouterScores {
  const float* scores;
  const float* biased;
  int32_t* ids;
  float* weights;
  const DgppMoeConfig* cfg;
};
int gate_up_with_shared(int fp4_group, const RouterScores* select, const uint16_t* x, size_t x_stride, const int32_t* ids,
                        const DgppMoeExpertView* views, int inter, int hidden, const SharedExpert& shared, uint16_t* act, int act_stride,
                        int tokens, int top_k, float limit, void* stream, bool& taken);
int down_accum_with_shared(int fp4_group, const uint16_t* act, size_t act_stride, const int32_t* ids, const DgppMoeExpertView* views,
                           int hidden, int inter, const SharedExpert& shared, int tokens, int top_k, const float* weights,
                           uint16_t* out_bf16, bool ask, void* stream, bool& taken);

}  // namespace dgpp_amd
