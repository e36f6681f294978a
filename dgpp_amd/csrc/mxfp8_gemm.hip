// Activation-quantized MXFP8 form: per-row dynamic MXFP8 quantizers (plain, and fused behind the
// clamped SwiGLU of the MiniMax shared expert) and the block-scaled E4M3 x E4M3 GEMM on the
// scaled matrix-core instruction V_MFMA_SCALE_F32_16X16X128_F8F6F4, which takes both payloads as
// stored and one e8m0 scale per 32 values of either operand: no weight decode on the VALU at all.
//
// Reference counterparts: src/kernels/mxfp8_gemm.hpp:8-31 (interface), src/kernels/mxfp8_gemm.cu:24-79
// (quantizer), :106-203 (GEMM), :217-243 (argument rules), :246-275 (launchers).
#include <hip/hip_runtime.h>

#include <string>
#include <type_traits>

#include "../../include/dgpp_amd.h"
#include "../../include/dgpp_amd_bench.h"
#include "capi_errors.hpp"
#include "gemv_core.hpp"
#include "numerics.hpp"

namespace dgpp_amd {
namespace {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kQuantThreads = 256;

// ---- quantizers ----------------------------------------------------------------------------------

// The e8m0 exponent of a 32-group whose largest magnitude is `maximum`: ceil(log2(maximum / 448)), at
// least -127, read off the float's own fields (448 = 1.75 * 2^8, so the ceiling steps where the
// significand passes 1.75). src/kernels/mxfp8_gemm.cu:61-66.
__device__ __forceinline__ int group_exponent(float maximum) {
  const int biased = static_cast<int>((f32_bits(maximum) >> 23) & 255u);
  const float threshold = bits_f32((static_cast<uint32_t>(biased) << 23) | 0x600000u);
  const int e = biased - 135 + (maximum > threshold ? 1 : 0);
  return e < -127 ? -127 : e;
}

// Four E4M3 codes (round to nearest even; the scaled group never exceeds 448, the clamp only keeps an
// out-of-contract input finite) in one word, lowest address first.
__device__ __forceinline__ uint32_t pack_e4m3x4(float v0, float v1, float v2, float v3) {
  v0 = __builtin_amdgcn_fmed3f(v0, -448.f, 448.f);
  v1 = __builtin_amdgcn_fmed3f(v1, -448.f, 448.f);
  v2 = __builtin_amdgcn_fmed3f(v2, -448.f, 448.f);
  v3 = __builtin_amdgcn_fmed3f(v3, -448.f, 448.f);
  int word = 0;
  word = __builtin_amdgcn_cvt_pk_fp8_f32(v0, v1, word, false);
  word = __builtin_amdgcn_cvt_pk_fp8_f32(v2, v3, word, true);
  return static_cast<uint32_t>(word);
}

__device__ __forceinline__ void unpack_bf16x4(const uint2& q, float (&v)[4]) {
  v[0] = bits_f32(q.x << 16);
  v[1] = bits_f32(q.x & 0xffff0000u);
  v[2] = bits_f32(q.y << 16);
  v[3] = bits_f32(q.y & 0xffff0000u);
}

// One lane holds four adjacent values, eight lanes one 32-group (rows may start on any multiple of four
// elements, as in the reference). A row is k / 4 lanes; blockIdx.y is the row. With SWIGLU the values
// are first bf16(min(g, limit) * sigmoid(alpha * min(g, limit)) * (clamp(u, +-limit) + 1)), the sigmoid
// through the hardware's base-2 exponential and reciprocal where the reference goes through its
// approximate ones (src/kernels/mxfp8_gemm.cu:37-56).
template <bool SWIGLU>
__global__ __launch_bounds__(kQuantThreads) void mxfp8_quantize_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ up, size_t stride, int k, float alpha, float limit,
    uint8_t* __restrict__ codes, uint8_t* __restrict__ scales) {
  const int row = blockIdx.y;
  const int piece = blockIdx.x * kQuantThreads + threadIdx.x;
  const int column = piece * 4;
  // k is a multiple of 32, so the eight lanes of a group leave together.
  if (column >= k) return;
  float v[4];
  unpack_bf16x4(*reinterpret_cast<const uint2*>(x + static_cast<size_t>(row) * stride + column), v);
  if constexpr (SWIGLU) {
    float u[4];
    unpack_bf16x4(*reinterpret_cast<const uint2*>(up + static_cast<size_t>(row) * stride + column), u);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float g = fminf(v[i], limit);
      const float uc = fminf(fmaxf(u[i], -limit), limit);
      const float e = __builtin_amdgcn_exp2f((g * -alpha) * 1.4426950216293335f);
      const float sigmoid = __builtin_amdgcn_rcpf(1.f + e);
      v[i] = bf16_to_f32(f32_to_bf16((g * sigmoid) * (uc + 1.f)));
    }
  }
  float maximum = fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3])));
  maximum = fmaxf(maximum, __shfl_xor(maximum, 1));
  maximum = fmaxf(maximum, __shfl_xor(maximum, 2));
  maximum = fmaxf(maximum, __shfl_xor(maximum, 4));
  const int exponent = group_exponent(maximum);
  const float inverse = bits_f32(static_cast<uint32_t>(127 - exponent) << 23);
  *reinterpret_cast<uint32_t*>(codes + static_cast<size_t>(row) * k + column) =
      pack_e4m3x4(v[0] * inverse, v[1] * inverse, v[2] * inverse, v[3] * inverse);
  if ((piece & 7) == 0) scales[static_cast<size_t>(row) * (k >> 5) + (column >> 5)] = static_cast<uint8_t>(exponent + 127);
}

// ---- GEMM ----------------------------------------------------------------------------------------

__device__ __forceinline__ v8i as_operand(const u32x4& lo, const u32x4& hi) {
  v8i r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[i] = static_cast<int>(lo[i]);
    r[4 + i] = static_cast<int>(hi[i]);
  }
  return r;
}

template <typename Out>
__device__ __forceinline__ void put(Out* p, float v);
template <>
__device__ __forceinline__ void put<float>(float* p, float v) { *p = v; }
template <>
__device__ __forceinline__ void put<uint16_t>(uint16_t* p, float v) { *p = f32_to_bf16(v); }

// out[m, n] = A[m, k] * W[n, k]^T. A block owns 16 rows of W over all of k and MT * 16 rows of A.
//
// One matrix-core step covers 128 of k. Its operand layout: lane (r, g) = (lane % 16, lane / 16) holds,
// for row r of its 16, the 16 bytes at k = 16 g of the step in registers 0-3 and the 16 bytes at
// k = 64 + 16 g in registers 4-7, and supplies the scale byte of the row's k-block g of the step, which
// the hardware applies to that block wherever its bytes sit. W is the first operand, a 16-row tile of A
// the second; the lane receives out[a row r][w rows 4 g .. 4 g + 3].
//
// Loading in that layout would ask the memory pipe for 64 bytes of 16 different rows per instruction,
// which it serves at about half its streaming rate. A step's 16 x 128 bytes of either operand are
// therefore loaded row-major (two instructions of 8 rows x 128 contiguous bytes), parked in a
// wavefront-private LDS region and read back in operand layout; the region is XOR-swizzled so that the
// writes and the reads both touch every bank once.
//
// The block's WAVES waves split k: wave w takes the steps w, w + WAVES, ..., and the partial sums are
// added in wave order (tile t by wave t). The chain of every output element is therefore fixed by k alone
// (WAVES is chosen from k), whatever m, n and the rows that share a launch
// (src/kernels/mxfp8_gemm.hpp:23 asks the same of the reference's row geometries).
// Rows past n or m are clamped to the last one and never stored; bytes past k contribute zeros.
constexpr int kStepUnits = 128;   // 16-byte units of one step of one operand tile: 16 rows x 128 bytes

// The swizzled place of 16-byte piece `piece` (0-7) of row `row` (0-15) in a region.
__device__ __forceinline__ int region_unit(int row, int piece) { return row * 8 + (piece ^ ((row >> 1) & 7)); }

// This lane's two row-major loads of a step: rows (lane / 8) and 8 + (lane / 8) of the 16 that start at
// row0 (clamped to the last row), piece lane % 8 of the step's 128 bytes; zeros past k.
template <bool NT>
__device__ __forceinline__ void issue_step(const uint8_t* __restrict__ base, int row0, int rows, int k, int step,
                                           u32x4 (&t)[2]) {
  const int lane = threadIdx.x & 63;
  const int at = step * 128 + (lane & 7) * 16;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = min(row0 + 8 * i + (lane >> 3), rows - 1);
    const u32x4* src = reinterpret_cast<const u32x4*>(base + static_cast<size_t>(row) * k + (at < k ? at : 0));
    const u32x4 v = NT ? __builtin_nontemporal_load(src) : *src;
    t[i] = at < k ? v : u32x4{0u, 0u, 0u, 0u};
  }
}
__device__ __forceinline__ void commit_step(u32x4* __restrict__ region, const u32x4 (&t)[2]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < 2; ++i) region[region_unit(8 * i + (lane >> 3), lane & 7)] = t[i];
}
__device__ __forceinline__ v8i step_operand(const u32x4* __restrict__ region) {
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, g = lane >> 4;
  return as_operand(region[region_unit(r, g)], region[region_unit(r, 4 + g)]);
}

template <typename Out, int MT, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void mxfp8_gemm_kernel(
    const uint8_t* __restrict__ a, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ w,
    const uint8_t* __restrict__ w_scales, Out* __restrict__ out, int m, int n, int k, size_t out_stride) {
  static_assert(WAVES >= MT, "one folding wave per tile");
  // Two regions per wave while the steps run, the partial sums of every wave afterwards.
  constexpr int kStageUnits = WAVES * 2 * kStepUnits, kFoldUnits = WAVES * MT * 64;
  __shared__ u32x4 lds[kStageUnits > kFoldUnits ? kStageUnits : kFoldUnits];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * (16 * MT);
  const int kblocks = k >> 5;
  const int steps = (kblocks + 3) >> 2;
  u32x4* region = lds + wave * 2 * kStepUnits;

  const uint8_t* wsp = w_scales + static_cast<size_t>(min(n0 + r, n - 1)) * kblocks;
  const uint8_t* asp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) asp[t] = a_scales + static_cast<size_t>(min(m0 + t * 16 + r, m - 1)) * kblocks;

  v4f acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = v4f{0.f, 0.f, 0.f, 0.f};

  // Steps interleave over the waves, so that at any time the block reads a few KB of each row in one piece.
  // DEPTH steps of a wave are in flight together: every load of them is issued before the first use.
  constexpr int DEPTH = MT == 1 ? 4 : MT == 2 ? 2 : 1;
  for (int s0 = wave; s0 < steps; s0 += WAVES * DEPTH) {
    u32x4 wq[DEPTH][2], aq[DEPTH][MT][2];
    int ws[DEPTH], as[DEPTH][MT];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      const int s = s0 + d * WAVES;
      if (s >= steps) break;   // the same for the whole wave
      issue_step<true>(w, n0, n, k, s, wq[d]);
#pragma unroll
      for (int t = 0; t < MT; ++t) issue_step<false>(a, m0 + t * 16, m, k, s, aq[d][t]);
      const int kb = s * 4 + g;
      const int kc = kb < kblocks ? kb : kblocks - 1;   // a block past k holds zeros: any scale does
      ws[d] = wsp[kc];
#pragma unroll
      for (int t = 0; t < MT; ++t) as[d][t] = asp[t][kc];
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      if (s0 + d * WAVES >= steps) break;
      // The LDS serves a wavefront's accesses in order: a region is rewritten as soon as the read of its
      // previous content has been issued. The barriers only keep the compiler from moving accesses across.
      commit_step(region, wq[d]);
      __builtin_amdgcn_wave_barrier();
      const v8i wv = step_operand(region);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        u32x4* mine = region + ((t + 1) & 1) * kStepUnits;   // the other region than the tile before
        commit_step(mine, aq[d][t]);
        __builtin_amdgcn_wave_barrier();
        acc[t] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv, step_operand(mine), acc[t], 0, 0, 0, ws[d], 0, as[d][t]);
      }
    }
  }

  __syncthreads();   // every wave is done with its regions
  float4* fold = reinterpret_cast<float4*>(lds);
#pragma unroll
  for (int t = 0; t < MT; ++t) fold[(wave * MT + t) * 64 + lane] = float4{acc[t][0], acc[t][1], acc[t][2], acc[t][3]};
  __syncthreads();
  if (wave >= MT) return;
  const int t = wave;
  float4 sum = fold[t * 64 + lane];
#pragma unroll
  for (int p = 1; p < WAVES; ++p) {
    const float4 part = fold[(p * MT + t) * 64 + lane];
    sum.x += part.x;
    sum.y += part.y;
    sum.z += part.z;
    sum.w += part.w;
  }
  const int a_row = m0 + t * 16 + r;
  if (a_row >= m) return;
  Out* dst = out + static_cast<size_t>(a_row) * out_stride + n0 + g * 4;
  const float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n0 + g * 4 + i < n) put<Out>(dst + i, v[i]);
}

template <typename Out, int MT, int WAVES>
hipError_t launch_gemm_mt(const uint8_t* a, const uint8_t* as, const uint8_t* w, const uint8_t* ws, Out* out, int m, int n,
                          int k, size_t stride, hipStream_t stream) {
  const dim3 grid(static_cast<unsigned>((n + 15) / 16), static_cast<unsigned>((m + 16 * MT - 1) / (16 * MT)));
  hipLaunchKernelGGL((mxfp8_gemm_kernel<Out, MT, WAVES>), grid, dim3(WAVES * 64), 0, stream, a, as, w, ws, out, m, n, k, stride);
  return hipGetLastError();
}

template <typename Out, int WAVES>
hipError_t launch_gemm_waves(const uint8_t* a, const uint8_t* as, const uint8_t* w, const uint8_t* ws, Out* out, int m, int n,
                             int k, size_t stride, hipStream_t s) {
  if (m <= 16) return launch_gemm_mt<Out, 1, WAVES>(a, as, w, ws, out, m, n, k, stride, s);
  if (m <= 32) return launch_gemm_mt<Out, 2, WAVES>(a, as, w, ws, out, m, n, k, stride, s);
  if (m <= 48) return launch_gemm_mt<Out, 3, WAVES>(a, as, w, ws, out, m, n, k, stride, s);
  return launch_gemm_mt<Out, 4, WAVES>(a, as, w, ws, out, m, n, k, stride, s);
}

// ---- GEMM, many activation rows --------------------------------------------------------------------
//
// A block of 2 x 2 wavefronts owns TN = 32 WN rows of W and TM = 32 WM rows of A, a wavefront WN x WM 16 x 16 tiles of
// them. The form above has every 16 rows of W pull all of A's k range through the L2 (m * k * n / 16 bytes); here an
// operand byte in LDS serves TN or TM rows. A step's (TN + TM) x 128 bytes go through registers, DEPTH steps ahead of their
// use, into one of two LDS stages in the layout above, the rows' four scale bytes beside them; one barrier per step.
//
// The chain of an output element is the other form's bit for bit: the steps s = c, c + CHAINS, ... accumulate one after
// the other, and the CHAINS sums are added in order of c - the steps are only visited in that order here.
template <int WN, int WM>
struct TileStage {
  static constexpr int kTN = 32 * WN, kTM = 32 * WM, kRows = kTN + kTM;
  u32x4 unit[kRows * 8];
  uint32_t scale[kRows];
};

template <typename Out, int WN, int WM, int DEPTH, int CHAINS>
__global__ __launch_bounds__(256, 2) void mxfp8_gemm_tiled_kernel(
    const uint8_t* __restrict__ a, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ w,
    const uint8_t* __restrict__ w_scales, Out* __restrict__ out, int m, int n, int k, size_t out_stride, int row_tiles,
    int passes) {
  using Stage = TileStage<WN, WM>;
  constexpr int kTN = Stage::kTN, kTM = Stage::kTM, kLoads = Stage::kRows / 32;
  __shared__ Stage stages[2];
  // Consecutive workgroups go to the eight XCDs in turn: an XCD keeps the column passes of a row tile to itself, so
  // that its L2 reads the tile's weights once.
  const int lin = static_cast<int>(blockIdx.x), idx = lin / 8;
  const int row_tile = idx / passes * 8 + lin % 8;
  if (row_tile >= row_tiles) return;
  const int n0 = row_tile * kTN, m0 = idx % passes * kTM;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int wn = (wave & 1) * WN * 16, wm = kTN + (wave >> 1) * WM * 16;   // first rows of the stage that the wave reads
  const int kblocks = k >> 5, steps = (kblocks + 3) >> 2;
  const int piece = threadIdx.x & 7;
  const uint8_t* src[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = i * 32 + static_cast<int>(threadIdx.x >> 3);
    src[i] = i * 32 < kTN ? w + static_cast<size_t>(min(n0 + row, n - 1)) * k
                          : a + static_cast<size_t>(min(m0 + row - kTN, m - 1)) * k;
  }
  static_assert(Stage::kRows <= 256, "a thread carries the scales of one row");
  const int srow = min(static_cast<int>(threadIdx.x), Stage::kRows - 1);   // the threads past it write the last row's again
  const uint8_t* ssrc = srow < kTN ? w_scales + static_cast<size_t>(min(n0 + srow, n - 1)) * kblocks
                                   : a_scales + static_cast<size_t>(min(m0 + srow - kTN, m - 1)) * kblocks;

  // No branch around a load: only then does the compiler count the loads in flight and wait for the oldest step alone.
  // Past k a lane reads the start of its row (W's become zeros in commit(), which is enough: A's and the scales that
  // meet them are the row's own, NaN only where the sums are). A row's four scale bytes are one unaligned word; where
  // the last step has two, it is the row's last word, turned so that they come first.
  struct __attribute__((packed, aligned(1))) Word { uint32_t v; };
  u32x4 t[DEPTH][kLoads];
  uint32_t sc[DEPTH];
  auto load = [&](int s, u32x4 (&to)[kLoads], uint32_t& scale) {
    const int at = s * 128 + piece * 16, from = at < k ? at : 0;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) to[i] = *reinterpret_cast<const u32x4*>(src[i] + from);
    scale = reinterpret_cast<const Word*>(ssrc + min(s * 4, kblocks - 4))->v;
  };
  auto commit = [&](int s, Stage& st, const u32x4 (&from)[kLoads], uint32_t scale) {
    const bool inside = s * 128 + piece * 16 < k;
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      u32x4 v = from[i];
      if (i * 32 < kTN) v = inside ? v : u32x4{0u, 0u, 0u, 0u};
      st.unit[region_unit(i * 32 + static_cast<int>(threadIdx.x >> 3), piece)] = v;
    }
    st.scale[srow] = __builtin_amdgcn_alignbit(scale, scale, s * 4 + 4 > kblocks ? 16 : 0);
  };

  v4f acc[WN][WM], sum[WN][WM];
#pragma unroll
  for (int i = 0; i < WN; ++i)
#pragma unroll
    for (int j = 0; j < WM; ++j) acc[i][j] = sum[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  // The order of the steps: s, s + CHAINS, ... of chain c, then chain c + 1 (c < CHAINS: every step once). `ahead` is
  // DEPTH steps before `at`.
  struct Walk {
    int s, c;
    __device__ __forceinline__ bool last_of_chain(int steps) const { return s + CHAINS >= steps; }
    __device__ __forceinline__ void next(int steps) { s = last_of_chain(steps) ? ++c : s + CHAINS; }
  };
  const int chains = min(CHAINS, steps);
  Walk at = {0, 0}, ahead = {0, 0};
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    load(min(ahead.s, steps - 1), t[d], sc[d]);   // past the last step: that step again, unused
    ahead.next(steps);
  }
  int buf = 0;
  for (;;) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      Stage& st = stages[buf];
      buf ^= 1;
      commit(at.s, st, t[d], sc[d]);
      load(min(ahead.s, steps - 1), t[d], sc[d]);
      ahead.next(steps);
      __syncthreads();   // the stage is whole; its readers of two steps before passed the barrier of the step between
      const uint8_t* sb = reinterpret_cast<const uint8_t*>(st.scale);
      v8i wv[WN];
      int ws[WN];
#pragma unroll
      for (int i = 0; i < WN; ++i) {
        const int row = wn + i * 16 + r;
        wv[i] = as_operand(st.unit[region_unit(row, g)], st.unit[region_unit(row, 4 + g)]);
        ws[i] = sb[row * 4 + g];
      }
#pragma unroll
      for (int j = 0; j < WM; ++j) {
        const int row = wm + j * 16 + r;
        const v8i av = as_operand(st.unit[region_unit(row, g)], st.unit[region_unit(row, 4 + g)]);
        const int as = sb[row * 4 + g];
#pragma unroll
        for (int i = 0; i < WN; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv[i], av, acc[i][j], 0, 0, 0, ws[i], 0, as);
      }
      if (at.last_of_chain(steps)) {
#pragma unroll
        for (int i = 0; i < WN; ++i)
#pragma unroll
          for (int j = 0; j < WM; ++j) {
            sum[i][j] = at.c == 0 ? acc[i][j] : sum[i][j] + acc[i][j];
            acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
          }
      }
      at.next(steps);
      if (at.c >= chains) goto summed;   // not a break: a loop condition would join here with fewer loads in flight
    }
  }
summed:
  if (chains < CHAINS) {   // the other form's empty partial sums: -0 becomes +0
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int j = 0; j < WM; ++j) sum[i][j] = sum[i][j] + acc[i][j];
  }

#pragma unroll
  for (int j = 0; j < WM; ++j) {
    const int a_row = m0 + wm - kTN + j * 16 + r;
    if (a_row >= m) continue;
#pragma unroll
    for (int i = 0; i < WN; ++i) {
      const int col = n0 + wn + i * 16 + g * 4;
      Out* dst = out + static_cast<size_t>(a_row) * out_stride + col;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (col + e < n) put<Out>(dst + e, sum[i][j][e]);
    }
  }
}

// ---- GEMM, a ring of stages --------------------------------------------------------------------------
//
// The tiles above have DEPTH steps on their way in registers. Here the operands go from memory to a ring of STAGES LDS stages without
// passing registers, and the e8m0 scales of all of a block's rows come once, to a panel whose words hold the scales of a k-block of
// four steps: the instruction takes the byte. WGN x WGM wavefronts, each WT 16-row tiles of W times MT of A. The chain of an output
// element is the other forms' (see above); SIDE of them run side by side, so that with four a row is read 512 bytes at a time
// and sums meet once in four chains.
//
// What bounds it: a step's own way, barrier, operands out of LDS, products, about 0.25 us whatever the tile up to 64 x 64 (a CU fetches
// 50 to 60 of the 130 bytes a ns that its L2 gives), and for cold weights the latency of memory. Reading the operands a step ahead
// gained nothing, nor did eight stages. n = 4096, k = 6144, us, the tiles above -> here: 64 rows 17.5 -> 15.8, 160 31.5 -> 17.6, 300
// 41.9 -> 22.3, 1024 66 -> 38; n = 6144, k = 4096: 64 22.0 -> 11.9, 300 31.8 -> 18.9, 1024 76 -> 52.

// 1 KB of a wavefront, a lane's 16 bytes after the other's, from base + offset + at to LDS; zeros from `bytes` on.
__device__ __forceinline__ void ring_load(const uint8_t* base, int bytes, uint32_t offset, int at, u32x4* to) {
  const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, bytes, 0x00027000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (__attribute__((address_space(3))) void*)to, 16, offset, at, 0, 0);
}
template <int WGN, int WGM, int WT, int MT, int STAGES, int QUADS, int SIDE>
struct RingShape {
  static constexpr int kWaves = WGN * WGM, kThreads = kWaves * 64;
  static constexpr int kTN = 16 * WT * WGN, kTM = 16 * MT * WGM, kRows = kTN + kTM;
  static constexpr int kUnits = kRows * 8;                     // 16-byte units of a stage: 128 bytes of every row
  static constexpr int kLoads = kUnits / kThreads;             // of a wavefront and stage, eight rows x 128 bytes each
  static constexpr int kMaxK = (QUADS < 16 ? QUADS : 16) * 4 * 128;
  static_assert(kLoads * kThreads == kUnits && kTN % 8 == 0, "whole loads");
  static_assert(QUADS % 2 == 1 && QUADS <= 17, "sixteen rows of the panel meet no bank twice");
  static constexpr int kTurns = STAGES == 3 ? 12 : STAGES;     // until the stages and the steps of a quad are in the same places again
  static_assert((STAGES == 3 || STAGES == 4) && (STAGES - 2) * kLoads < 64, "four named stages; the waits count to 63");
  static_assert(SIDE == 1 || SIDE == 4, "the panel holds the scales of four steps to a word");
};

template <int N>
__device__ __forceinline__ void ring_barrier() {   // all but the newest N loads of the wavefront have arrived; then the block's barrier
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Launched with kThreads threads; the bound of 512 keeps the compiler to 256 registers, and the accumulators out of those
// that it would have to move sums in and out of.
template <typename Out, int WGN, int WGM, int WT, int MT, int STAGES, int QUADS, int SIDE, int CHAINS>
__global__ __launch_bounds__(512) void mxfp8_gemm_ring_kernel(
    const uint8_t* __restrict__ a, const uint8_t* __restrict__ a_scales, const uint8_t* __restrict__ w,
    const uint8_t* __restrict__ w_scales, Out* __restrict__ out, int m, int n, int k, size_t out_stride, int row_tiles,
    int passes) {
  using Shape = RingShape<WGN, WGM, WT, MT, STAGES, QUADS, SIDE>;
  constexpr int kRows = Shape::kRows, kTN = Shape::kTN, kLoads = Shape::kLoads, kWaves = Shape::kWaves;
  // By name: the compiler then tells a stage that is read from those that are on their way.
  constexpr int kUnits = Shape::kUnits;
  __shared__ u32x4 stage0[kUnits], stage1[kUnits], stage2[kUnits], stage3[STAGES == 4 ? kUnits : 1];
  auto stage = [&](auto turn) -> u32x4* {
    constexpr int kAt = decltype(turn)::value % STAGES;
    if constexpr (kAt == 0) return stage0;
    else if constexpr (kAt == 1) return stage1;
    else if constexpr (kAt == 2) return stage2;
    else return stage3;
  };
  __shared__ u32x4 panel[kRows * QUADS];
  // Consecutive workgroups go to the eight XCDs in turn: an XCD keeps the column passes of a row tile to itself.
  const int lin = static_cast<int>(blockIdx.x), idx = lin / 8;
  const int row_tile = idx / passes * 8 + lin % 8;
  if (row_tile >= row_tiles) return;
  const int n0 = row_tile * kTN, m0 = idx % passes * Shape::kTM;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int kblocks = k >> 5, steps = (kblocks + 3) >> 2;

  // The order of the units, SIDE steps each, which belong to chains SIDE c .. SIDE c + SIDE - 1: c, c + CHAINS / SIDE, ..., then c + 1.
  const int quads = (steps + 3) >> 2, units = SIDE == 4 ? quads : steps;
  struct Walk {
    int at, first;
    __device__ __forceinline__ bool next(int units) {   // whether that was the last of its chains
      const bool last = at + CHAINS / SIDE >= units;
      first += last ? 1 : 0;
      at = last ? first : at + CHAINS / SIDE;
      return last;
    }
  };

  // The panel: a quad of a row to a thread, words of a step turned into words of a k-block. Where the last step has two blocks, its word
  // is the row's last, turned so that they come first; past the last step, that one again, which nobody uses. All of a thread's words
  // are on their way together, and the first stages behind them.
  struct __attribute__((packed, aligned(1))) Word { uint32_t v; };
  constexpr int kEach = kRows * 16 / Shape::kThreads;
  const int quad_of = static_cast<int>(threadIdx.x) & 15, row_of = static_cast<int>(threadIdx.x) >> 4;
  uint32_t word[kEach][4];
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const int row = row_of + e * (Shape::kThreads / 16);
    const uint8_t* src = row < kTN ? w_scales + static_cast<size_t>(min(n0 + row, n - 1)) * kblocks
                                   : a_scales + static_cast<size_t>(min(m0 + row - kTN, m - 1)) * kblocks;
#pragma unroll
    for (int i = 0; i < 4; ++i) word[e][i] = reinterpret_cast<const Word*>(src + min(quad_of * 16 + i * 4, kblocks - 4))->v;
  }

  // Load i of the wavefront: eight rows x 128 bytes of a step, the lane's piece the one that belongs at the lane's place. Where k ends
  // inside the last step the next row's bytes come along, or zeros behind the last row; multiply() clears them.
  uint32_t off[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = (i * kWaves + wave) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    const int of = row < kTN ? min(n0 + row, n - 1) - n0 : min(m0 + row - kTN, m - 1) - m0;
    off[i] = static_cast<uint32_t>(of) * static_cast<uint32_t>(k) + piece * 16;
  }
  const uint8_t* wbase = w + static_cast<size_t>(n0) * k;
  const uint8_t* abase = a + static_cast<size_t>(m0) * k;
  const int wbytes = min(n - n0, kTN) * k, abytes = min(m - m0, Shape::kTM) * k;
  Walk ahead = {0, 0}, at = {0, 0};
  auto load = [&](auto turn) {   // what that turn multiplies
    constexpr int kStep = decltype(turn)::value % 4;
    u32x4* const to = stage(turn);
    const int byte = min(SIDE == 4 ? ahead.at * 4 + kStep : ahead.at, steps - 1) * 128;   // past the last step that one again: the waits count the loads
    if constexpr (SIDE == 1 || kStep == 3) ahead.next(units);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const bool is_w = kTN / 8 % kWaves == 0 ? i * kWaves < kTN / 8 : (i * kWaves + wave) * 8 < kTN;
      ring_load(is_w ? wbase : abase, is_w ? wbytes : abytes, off[i], byte, to + (i * kWaves + wave) * 64);
    }
  };
  load(std::integral_constant<int, 0>{});
  load(std::integral_constant<int, 1>{});
  if constexpr (STAGES == 4) load(std::integral_constant<int, 2>{});
  if (quad_of < quads) {
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      uint32_t v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_amdgcn_alignbit(word[e][i], word[e][i], (quad_of * 4 + i) * 4 + 4 > kblocks ? 16 : 0);
      const uint32_t lo01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400), hi01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602);
      const uint32_t lo23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400), hi23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602);
      panel[(row_of + e * (Shape::kThreads / 16)) * QUADS + quad_of] =
          u32x4{__builtin_amdgcn_perm(lo23, lo01, 0x05040100), __builtin_amdgcn_perm(lo23, lo01, 0x07060302),
                __builtin_amdgcn_perm(hi23, hi01, 0x05040100), __builtin_amdgcn_perm(hi23, hi01, 0x07060302)};
    }
  }

  const int wn = wave % WGN * WT * 16, wm = kTN + wave / WGN * MT * 16;   // first rows of the stage that the wavefront reads
  v4f acc[SIDE][WT][MT], sum[WT][MT];
#pragma unroll
  for (int i = 0; i < WT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) {
#pragma unroll
      for (int c = 0; c < SIDE; ++c) acc[c][i][j] = v4f{0.f, 0.f, 0.f, 0.f};
      sum[i][j] = v4f{-0.f, -0.f, -0.f, -0.f};   // whose sum with a number is the number
    }

  int ws[WT], as[MT];   // a quad's scales
  const int* panel_lane = reinterpret_cast<const int*>(panel) + r * (QUADS * 4) + g;
  auto read_scales = [&](int quad, int shift) {
#pragma unroll
    for (int i = 0; i < WT; ++i) ws[i] = panel_lane[(wn + i * 16) * (QUADS * 4) + quad * 4] >> shift;
#pragma unroll
    for (int j = 0; j < MT; ++j) as[j] = panel_lane[(wm + j * 16) * (QUADS * 4) + quad * 4] >> shift;
  };
  const int cut = (k & 64) != 0 ? steps - 1 : -1;   // the step that k ends inside of
  int left = SIDE == 4 ? quads * 4 : steps;
  // A stage is whole for every wavefront after the barrier, which the readers of the one that is filled next have passed.
  auto turn = [&](auto i) {
    constexpr int kStep = decltype(i)::value % 4, kByte = SIDE == 4 ? kStep : 0, kChain = SIDE == 4 ? kStep : 0;
    ring_barrier<(STAGES - 2) * kLoads>();
    load(std::integral_constant<int, decltype(i)::value + STAGES - 1>{});
    const u32x4* unit = stage(i);
    const int s = SIDE == 4 ? at.at * 4 + kStep : min(at.at, steps - 1);
    if constexpr (SIDE == 1) read_scales(s >> 2, (s & 3) * 8);
    v8i wv[WT], av[MT];
#pragma unroll
    for (int t = 0; t < WT; ++t) wv[t] = as_operand(unit[region_unit(wn + t * 16 + r, g)], unit[region_unit(wn + t * 16 + r, 4 + g)]);
#pragma unroll
    for (int t = 0; t < MT; ++t) av[t] = as_operand(unit[region_unit(wm + t * 16 + r, g)], unit[region_unit(wm + t * 16 + r, 4 + g)]);
    if (s == cut) {   // clears what came from behind k (asm: else every step selects)
      // A matrix instruction may read what a vector one wrote two wait states later. The compiler does not see into asm: they are in it.
#pragma unroll
      for (int e = 4; e < 8; ++e) {
#pragma unroll
        for (int t = 0; t < WT; ++t) asm volatile("v_mov_b32 %0, 0\n\ts_nop 1" : "=v"(wv[t][e]));
#pragma unroll
        for (int t = 0; t < MT; ++t) asm volatile("v_mov_b32 %0, 0\n\ts_nop 1" : "=v"(av[t][e]));
      }
    }
    if (SIDE == 4 ? s < steps : left > 0) {
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int t = 0; t < WT; ++t)
          acc[kChain][t][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wv[t], av[j], acc[kChain][t][j], 0, 0, kByte, ws[t], kByte, as[j]);
    }
    if constexpr (SIDE == 1 || kStep == 3) {
      const bool fold = at.next(units);
      if constexpr (SIDE == 4) read_scales(min(at.at, quads - 1), 0);
      if (fold && left > 0) {
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
          for (int j = 0; j < MT; ++j)
#pragma unroll
            for (int c = 0; c < SIDE; ++c) {
              sum[t][j] = sum[t][j] + acc[c][t][j];
              acc[c][t][j] = v4f{0.f, 0.f, 0.f, 0.f};
            }
      }
    }
    --left;
  };
  auto four = [&](auto first) {   // whether there are more
    constexpr int kFirst = decltype(first)::value * 4;
    turn(std::integral_constant<int, kFirst>{});
    turn(std::integral_constant<int, kFirst + 1>{});
    turn(std::integral_constant<int, kFirst + 2>{});
    turn(std::integral_constant<int, kFirst + 3>{});
    return left > 0;
  };
  if constexpr (SIDE == 4) {   // the panel is whole
    __syncthreads();
    read_scales(0, 0);
  }
  for (;;) {
    if (!four(std::integral_constant<int, 0>{})) break;
    if constexpr (Shape::kTurns > 4) { if (!four(std::integral_constant<int, 1>{})) break; }
    if constexpr (Shape::kTurns > 8) { if (!four(std::integral_constant<int, 2>{})) break; }
  }
  if (SIDE == 1 && steps < CHAINS) {   // the other forms' empty partial sums: -0 becomes +0
#pragma unroll
    for (int t = 0; t < WT; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) sum[t][j] = sum[t][j] + acc[0][t][j];
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // nothing is on its way to the LDS when the block ends

  const bool vec = (reinterpret_cast<uintptr_t>(out) & 15u) == 0 && out_stride % 4 == 0;
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int a_row = m0 + wm - kTN + j * 16 + r;
    if (a_row >= m) continue;
#pragma unroll
    for (int i = 0; i < WT; ++i) {
      const int col = n0 + wn + i * 16 + g * 4;
      Out* dst = out + static_cast<size_t>(a_row) * out_stride + col;
      if (vec && col + 4 <= n) {
        struct alignas(4 * sizeof(Out)) Four { Out v[4]; } four;
#pragma unroll
        for (int e = 0; e < 4; ++e) put<Out>(&four.v[e], sum[i][j][e]);
        *reinterpret_cast<Four*>(dst) = four;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (col + e < n) put<Out>(dst + e, sum[i][j][e]);
      }
    }
  }
}

template <typename Out, int WGN, int WGM, int WT, int MT, int STAGES, int QUADS, int SIDE>
hipError_t launch_gemm_ring(const uint8_t* a, const uint8_t* as, const uint8_t* w, const uint8_t* ws, Out* out, int m, int n,
                            int k, size_t stride, hipStream_t stream) {
  using Shape = RingShape<WGN, WGM, WT, MT, STAGES, QUADS, SIDE>;
  if (k > Shape::kMaxK) return hipErrorInvalidValue;   // tiles_for() asks for no such
  note_launch(kFormTiles);
  const int row_tiles = (n + Shape::kTN - 1) / Shape::kTN, passes = (m + Shape::kTM - 1) / Shape::kTM;
  const dim3 grid(static_cast<unsigned>((row_tiles + 7) / 8 * 8) * static_cast<unsigned>(passes));
  if (k >= 16 * 128)
    hipLaunchKernelGGL((mxfp8_gemm_ring_kernel<Out, WGN, WGM, WT, MT, STAGES, QUADS, SIDE, 16>), grid, dim3(Shape::kThreads), 0, stream, a, as, w, ws, out, m, n, k, stride, row_tiles, passes);
  else
    hipLaunchKernelGGL((mxfp8_gemm_ring_kernel<Out, WGN, WGM, WT, MT, STAGES, QUADS, SIDE, 4>), grid, dim3(Shape::kThreads), 0, stream, a, as, w, ws, out, m, n, k, stride, row_tiles, passes);
  return hipGetLastError();
}

template <typename Out, int WN, int WM, int DEPTH>
hipError_t launch_gemm_tiled(const uint8_t* a, const uint8_t* as, const uint8_t* w, const uint8_t* ws, Out* out, int m, int n,
                             int k, size_t stride, hipStream_t stream) {
  note_launch(kFormTiles);
  constexpr int tn = 32 * WN, tm = 32 * WM;
  const int row_tiles = (n + tn - 1) / tn, passes = (m + tm - 1) / tm;
  const dim3 grid(static_cast<unsigned>((row_tiles + 7) / 8 * 8) * static_cast<unsigned>(passes));
  if (k >= 16 * 128)
    hipLaunchKernelGGL((mxfp8_gemm_tiled_kernel<Out, WN, WM, DEPTH, 16>), grid, dim3(256), 0, stream, a, as, w, ws, out, m, n, k, stride, row_tiles, passes);
  else
    hipLaunchKernelGGL((mxfp8_gemm_tiled_kernel<Out, WN, WM, DEPTH, 4>), grid, dim3(256), 0, stream, a, as, w, ws, out, m, n, k, stride, row_tiles, passes);
  return hipGetLastError();
}

// Which form takes an m x n x k product: 0 the 16-row one, 1 - 3 tiles of 32 x 64, 64 x 64 and 64 x 128 (W x A rows) through registers,
// 4 - 8 the ring's, of 32 x 64, 64 x 64, 64 x 128, 128 x 64 and 128 x 128.
//
// The 16-row form stays where its blocks, 16 rows of W each, are one round of the CUs and up to 48 rows of A (us, 16-row form /
// ring: n = 4096, k = 6144: 17 rows 10.1 / 15.2, 48 13.5 / 15.3, 64 16.6 / 15.8; n = 2048, k = 5184: 32 9.9 / 11.1, 48 12.0 / 11.2), two
// rounds and up to 16 rows (n = 6144, k = 6144: 1 row 12.7 / 15.5, 16 14.9 / 15.5; three rounds, n = 12288, k = 4096: 16.2 / 13.3 and
// 18.0 / 13.4; one row of n = 32768, k = 4096 35 / 24, of 65536 68 / 56), up to three quarters of a round below k = 3072 (56 shapes 0.76 to 1.3 times the ring's time, on average 0.97:
// 147 rows of n = 630, k = 2176 5.9 / 7.7; from 3072 on 0.79 to 1.6, 1.2), and where k is less than sixteen steps and its passes of 16 x 16 are few (n = 1024, k = 1088: 300 rows 5.5 /
// 6.0, 1024 12.3 / 6.9). Past one round it loses from 17 rows on (n = 6144, k = 4096: 17 rows 12.4 / 11.5, 64 21.4 / 11.9; n = 12288: 20.2 / 13.6).
//
// Among the ring's tiles the one whose rounds of 256 blocks cost least, counted on the fullest XCD (a row of tiles stays on one: 10688 rows of W in
// tiles of 128 by three passes are 33 blocks on three XCDs, two rounds). A round's cost by tile is what it took at k = 6144: 32 x 64
// 15 us, each further round 9 (two blocks fit a CU); 64 x 64 17; 64 x 128 23; 128 x 64 26; 128 x 128 35. n = 12288, k = 4096: 100
// rows 64 x 128 18.5 (32 x 64 24, 128 x 128 26), 160 128 x 128 26 (64 x 128 31), 300 128 x 64 36 (128 x 128 50, 64 x 64 46).
//
// The panel and the first stages of a block are paid by its walk, and the tiles through registers start sooner. 283 shapes of k = 128 to 1023, up to
// 131072 rows of W: the ring on average 1.08 times as long, up to 1.9 (20 rows of n = 37178, k = 192 8.0 / 13.2; 163 of 28995, k = 576 20.6
// / 28.8). From 1024 to 2047, 267 shapes: in one round 0.54 to 1.03, on average 0.83 (the largest tile from 1536 on; 1538 rows of n = 2164, k = 1024
// 17.9 / 21.6), in more 0.69 to 1.29, 0.99; against the 16-row form
// up to 16 rows of A 0.95 to 1.5, from 17 to 32 0.78 to 0.93 (32 rows of n = 22515, k = 1152 13.0 / 10.5). Past 2048, 450 shapes, on average 0.82.
//
// A panel holds the scales of 8192 of k, 6656 beside the largest tile. Without the ring, tiles through registers: the smallest while
// they are no more than the CUs, the largest once there are two for every CU; the 16-row form up to 32 rows and where its passes are few.
int tiles_for(int m, int n, int k) {
  if (k < 128) return 0;   // the tiles read whole words of scales
  const int knob = tune_get(kTuneTiled);   // bench / test switch: 1 never tiled, 2 - 9 the tiles
  if (knob >= 1 && knob <= (k <= 6656 ? 9 : k <= 8192 ? 8 : 4)) return knob - 1;
  constexpr int64_t kCus = 256;
  auto blocks = [&](int tn, int tm) { return static_cast<int64_t>((n + tn - 1) / tn) * ((m + tm - 1) / tm); };
  if (k >= 1024 && k <= 8192) {
    if (m <= 16 && blocks(16, 64) <= 2 * kCus) return 0;
    if (m <= 48 && blocks(16, 64) <= kCus) return 0;
    if (k < 2048 && (m <= 16 || blocks(16, 16) <= 7 * kCus)) return 0;
    if (k < 3072 && blocks(16, 64) <= kCus * 3 / 4) return 0;
    auto rounds = [&](int tn, int tm) { return (static_cast<int64_t>((n + tn - 1) / tn + 7) / 8 * ((m + tm - 1) / tm) + 31) / 32; };
    const int64_t of[5] = {rounds(32, 64), rounds(64, 64), rounds(64, 128), rounds(128, 64), rounds(128, 128)};
    const int64_t cost[5] = {6 + 9 * of[0], 17 * of[1], 23 * of[2], 26 * of[3], k >= 1536 && k <= 6656 ? 35 * of[4] : int64_t{1} << 40};
    int best = 0;
    for (int i = 1; i < 5; ++i)
      if (cost[i] < cost[best]) best = i;
    if (k >= 2048 || m <= 32 || of[best] == 1) return 4 + best;
  }
  if (m <= 32 || (m <= 64 && blocks(64, 64) <= kCus)) return 0;
  if (m > 64 && blocks(16, 16) <= (k < 2048 ? 7 : 4) * kCus) return 0;
  if (m > 512 && blocks(64, 128) >= 2 * kCus) return 3;
  return blocks(32, 64) <= kCus ? 1 : 2;
}

// src/kernels/mxfp8_gemm.cu:217-243.
template <typename Out>
int gemm(const uint8_t* a, const uint8_t* as, const uint8_t* w, const uint8_t* ws, Out* out, int m, int n, int k,
         void* stream, size_t stride, int output_tile) {
  const char* who = "MXFP8 GEMM";
  if (m <= 0 || n <= 0) return DGPP_OK;
  if (k <= 0 || k % 64) return report_invalid(std::string(who) + ": k must be a positive multiple of 64");
  if (stride == 0) stride = static_cast<size_t>(n);
  if (stride < static_cast<size_t>(n)) return report_invalid(std::string(who) + ": output stride is too small");
  if (output_tile != 0 && output_tile != 8 && output_tile != 16 && output_tile != 32 && output_tile != 64)
    return report_invalid(std::string(who) + ": output tile must be 0, 8, 16, 32 or 64");
  if (!a || !as || !w || !ws || !out) return report_invalid(std::string(who) + ": null pointer");
  if (((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15u) != 0)
    return report_invalid(std::string(who) + ": payloads must be 16-byte aligned");
  // The tile override is a diagnostic of the reference's kernel; every value gives the same chain here.
  // Waves per block from k alone (an output element's chain must not depend on m or n): sixteen once every
  // wave has a step of its own.
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (tiles_for(m, n, k)) {
    case 1: return report_hip(launch_gemm_tiled<Out, 1, 2, 4>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 2: return report_hip(launch_gemm_tiled<Out, 2, 2, 2>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 3: return report_hip(launch_gemm_tiled<Out, 2, 4, 2>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 4: return report_hip(launch_gemm_ring<Out, 2, 2, 1, 2, 4, 17, 4>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 5: return report_hip(launch_gemm_ring<Out, 4, 2, 1, 2, 4, 17, 4>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 6: return report_hip(launch_gemm_ring<Out, 2, 4, 2, 2, 4, 17, 4>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 7: return report_hip(launch_gemm_ring<Out, 4, 2, 2, 2, 4, 17, 4>(a, as, w, ws, out, m, n, k, stride, s), who);
    case 8: return report_hip(launch_gemm_ring<Out, 2, 4, 4, 2, 3, 13, 1>(a, as, w, ws, out, m, n, k, stride, s), who);
    default: break;
  }
  const hipError_t err = k >= 16 * 128 ? launch_gemm_waves<Out, 16>(a, as, w, ws, out, m, n, k, stride, s)
                                       : launch_gemm_waves<Out, 4>(a, as, w, ws, out, m, n, k, stride, s);
  return report_hip(err, who);
}

// src/kernels/mxfp8_gemm.cu:246-268. A lane reads 8 bytes and writes 4, so besides the reference's rules
// (32-wide groups, a stride of at least k and a multiple of four elements) the rows start 8-byte aligned.
int quantize(const uint16_t* x, const uint16_t* up, bool fused, size_t stride, int rows, int k, float alpha, float limit,
             uint8_t* codes, uint8_t* scales, void* stream, const char* who) {
  if (rows <= 0) return DGPP_OK;
  if (k <= 0 || k % 32 || stride < static_cast<size_t>(k) || stride % 4)
    return report_invalid(std::string(who) + ": requires 32-wide groups and aligned input rows");
  if (!x || !codes || !scales || (fused && !up)) return report_invalid(std::string(who) + ": null pointer");
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(up)) & 7u) != 0 ||
      (reinterpret_cast<uintptr_t>(codes) & 3u) != 0)
    return report_invalid(std::string(who) + ": input rows must be 8-byte aligned, codes 4-byte aligned");
  if (rows > 65535) return report_invalid(std::string(who) + ": more than 65535 rows");
  const dim3 grid(static_cast<unsigned>((k / 4 + kQuantThreads - 1) / kQuantThreads), static_cast<unsigned>(rows));
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (fused)
    hipLaunchKernelGGL((mxfp8_quantize_kernel<true>), grid, dim3(kQuantThreads), 0, s, x, up, stride, k, alpha, limit, codes, scales);
  else
    hipLaunchKernelGGL((mxfp8_quantize_kernel<false>), grid, dim3(kQuantThreads), 0, s, x, up, stride, k, 0.f, 0.f, codes, scales);
  return report_hip(hipGetLastError(), who);
}

}  // namespace
}  // namespace dgpp_amd

using namespace dgpp_amd;

extern "C" {

int dgpp_bench_mxfp8_form(int m, int n, int k) { return m <= 0 || n <= 0 || k <= 0 || k % 64 != 0 ? -1 : tiles_for(m, n, k); }

int dgpp_launch_mxfp8_quantize_rows(const uint16_t* x, size_t x_stride, int rows, int k, uint8_t* codes, uint8_t* scales,
                                    void* stream) {
  return quantize(x, nullptr, false, x_stride, rows, k, 0.f, 0.f, codes, scales, stream, "MXFP8 quantize");
}
int dgpp_launch_minimax_swiglu_mxfp8_rows(const uint16_t* gate, const uint16_t* up, size_t stride, int rows, int k, float alpha,
                                          float limit, uint8_t* codes, uint8_t* scales, void* stream) {
  return quantize(gate, up, true, stride, rows, k, alpha, limit, codes, scales, stream, "MiniMax SwiGLU MXFP8");
}
int dgpp_launch_mxfp8_gemm_bf16(const uint8_t* a, const uint8_t* a_scales, const uint8_t* w, const uint8_t* w_scales,
                                uint16_t* out, int m, int n, int k, void* stream, size_t out_stride, int output_tile) {
  return gemm<uint16_t>(a, a_scales, w, w_scales, out, m, n, k, stream, out_stride, output_tile);
}
int dgpp_launch_mxfp8_gemm_f32(const uint8_t* a, const uint8_t* a_scales, const uint8_t* w, const uint8_t* w_scales, float* out,
                               int m, int n, int k, void* stream, size_t out_stride, int output_tile) {
  return gemm<float>(a, a_scales, w, w_scales, out, m, n, k, stream, out_stride, output_tile);
}

}  // extern "C"
