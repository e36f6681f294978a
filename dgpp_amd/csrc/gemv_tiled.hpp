// The matrix-core form for many activation rows (prompt chunks): a block multiplies 128 weight rows with up to 128
// activation rows, so a weight is fetched and decoded once per 128 activation rows instead of once per 16
// (gemv_mfma_kernels.hpp). Included by gemv_kernels.hpp after the argument structs.
//
// With 16 rows per pass a prompt of T tokens decodes every weight T / 16 times and gathers the activations again for
// every 64 weight rows: the vector ALU and the gathers, not the matrix core, were the time. Here a wavefront owns two row
// groups (16 weight rows each) and CT column tiles: per 32 elements of k it decodes two operands and runs 2 CT MFMAs on
// them, and reads CT operands from LDS.
//
// What bounds it: the latency of a tile, with two wavefronts per SIMD to cover it. Counters (busy share of the chip's
// cycles, share of a wavefront's life): block FP8 1000 x 12288 x 6144 MFMA 33 %, vector ALU 42 %, LDS 17 %, waiting for
// data or a barrier 29 %, for an issue slot 33 %; MXFP4 prompt of 2048 tokens, gate + up MFMA 18 %, vector ALU 21 %, LDS
// 18 %, waiting 42 % and 33 %; NVFP4 activations, 16 rows a segment MFMA 13 %, waiting 61 %: 64-byte pieces of 16
// weight rows, one tile ahead. A pass of up to 32 rows pays for the registers and the LDS of one of 128. The grouped
// kernels spill around a pass, not in the walk over k (16 to 81 registers, MXFP4 gate + up 4): a short k pays most.
//
// Tile. k advances by 128 elements: the weights go from memory straight to the operand layout in registers (nothing
// of them is shared between wavefronts), the block's activation rows into one of two LDS stages of
// [row][16 units of 16 bytes], unit u of row r at u ^ (r % 16). The row-major writes and the FP8 operand reads (two
// units per lane and step) are conflict-free; of the FP4 reads (four units) the quarters meet in pairs, and half of their
// LDS cycles are conflicts. BF16 rows go from memory to LDS without passing registers, which the sums need. Loads of a
// tile are issued one tile ahead of its use; one barrier per tile. 64 KB of LDS and up to 256 registers: two blocks per
// CU, one computing while the other waits.
//
// Arithmetic. The sums of a (weight row, activation row) pair are those of the 16-row form: the same elements in the
// same MFMAs, K parts on their own, added in ascending order. A call's bits do not depend on which form takes it.
#pragma once

#include "gemv_mfma_kernels.hpp"

namespace dgpp_amd {

constexpr int kTileK = 128;                       // elements of k per tile
constexpr int kTiledCols = 128;                   // activation rows per pass
constexpr int kTiledRows = 128;                   // weight rows of a block (gate + up: 64 of each)
constexpr int kTiledStage = kTiledCols * 16;      // 16-byte units of one stage

// The two row groups of a wavefront: two groups of one matrix, or one of gate and one of up.
struct TiledRows {
  MatRef mat[2];
  int row0[2];
};

template <int FMT, bool A4, int CT>
struct TiledPass {
  static constexpr int kSub = MTraits<FMT>::kSub;
  static constexpr int kSteps = kTileK / MTraits<FMT>::kStepElems;   // steps of a row group per tile: 1 (FP4) or 2 (FP8)
  static constexpr int kCols = CT * kTileCols;
  static constexpr int kUnits = kCols * 16 / kBlockThreads;          // units of a stage per thread (BF16 rows)
  static constexpr int kCodeLoads = (kCols * 4 + kBlockThreads - 1) / kBlockThreads;   // 32-code loads per thread (A4)
  static constexpr int kActRegs = A4 ? kCodeLoads : kUnits;

  struct Regs {          // one tile on its way
    uint4 act[A4 ? kCodeLoads : 1];
    uint32_t act_s[A4 ? kCodeLoads : 1];
    uint4 w[2][kSteps];
    uint32_t s[2][kSteps];
  };

  const uint8_t* payload[2];
  uint32_t off[2];
  ScaleLane sl[2];
  int cs[2];
  const uint8_t* act;            // bytes
  const uint8_t* act_scales;
  uint32_t act_off[kActRegs];    // 16-byte units from `act`
  size_t act_srow[A4 ? kCodeLoads : 1];
  int k, chunks;

  __device__ __forceinline__ void load(int tile, Regs& r) const {
    const int q = (threadIdx.x & (kWave - 1)) >> 4;
    const bool full = (tile + 1) * kTileK <= k;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
#pragma unroll
      for (int s = 0; s < kSteps; ++s) {
        const int c = (tile * kSteps + s) * 4 + q;
        typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
        const __attribute__((address_space(1))) u32x4_t* src =
            (const __attribute__((address_space(1))) u32x4_t*)(uintptr_t)(payload[g] + off[g] + static_cast<uint32_t>(c) * 16u);
        r.w[g][s] = make_uint4(0u, 0u, 0u, 0u);
        if (full || c < chunks) {
          const u32x4_t v = *src;
          r.w[g][s] = make_uint4(v.x, v.y, v.z, v.w);
        }
        r.s[g][s] = load_scale<FMT>(sl[g], tile * kSteps + s, chunks, cs[g]);
      }
    }
    if constexpr (A4) {
      const int piece = threadIdx.x & 3;
#pragma unroll
      for (int i = 0; i < kCodeLoads; ++i) {
        r.act[i] = make_uint4(0u, 0u, 0u, 0u);
        r.act_s[i] = 0u;
        if (full || tile * kTileK + piece * 32 < k) {
          r.act[i] = *reinterpret_cast<const uint4*>(act + static_cast<size_t>(act_off[i]) * 16 + tile * 64 + piece * 16);
          r.act_s[i] = *reinterpret_cast<const uint16_t*>(act_scales + act_srow[i] + tile * 8 + piece * 2);
        }
      }
    }
  }

  // A tile's BF16 rows, from memory straight to their places in a stage: a wavefront's lanes fill 64 units in a row (four
  // rows' places), so it is the lane that reads the unit which belongs there. Waited for by the next __syncthreads().
  __device__ __forceinline__ void stage_rows(int tile, uint4* __restrict__ stage) const {
    const int u = (threadIdx.x & 15) ^ (threadIdx.x >> 4);   // row % 16 is threadIdx.x / 16 for each of the rows
    const int place = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * kWave;
    if ((tile + 1) * kTileK <= k) {
#pragma unroll
      for (int i = 0; i < kUnits; ++i)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) uint32_t*)(uintptr_t)(act + (static_cast<size_t>(act_off[i]) + tile * 16 + u) * 16),
            (__attribute__((address_space(3))) uint32_t*)(stage + place + i * 256), 16, 0, 0);
    } else {
#pragma unroll
      for (int i = 0; i < kUnits; ++i) {
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (tile * kTileK + u * 8 < k)
          v = *reinterpret_cast<const uint4*>(act + (static_cast<size_t>(act_off[i]) + tile * 16 + u) * 16);
        stage[threadIdx.x + i * 256] = v;
      }
    }
  }

  __device__ __forceinline__ void commit(uint4* __restrict__ stage, const Regs& r) const {
    if constexpr (A4) {
      const int piece = threadIdx.x & 3;
#pragma unroll
      for (int i = 0; i < kCodeLoads; ++i) {
        const int row = (threadIdx.x >> 2) + i * (kBlockThreads / 4);
        if (kCols * 4 >= kBlockThreads || row < kCols) {
          ChunkRegs ch;
          ch.w = r.act[i];
          ch.s = r.act_s[i];
          FragH f[4];
          decode_frags_nvfp4_f16(ch, f);
#pragma unroll
          for (int j = 0; j < 4; ++j) stage[row * 16 + ((piece * 4 + j) ^ (row & 15))] = __builtin_bit_cast(uint4, f[j].v);
        }
      }
    }
  }

  __device__ __forceinline__ void multiply(const uint4* __restrict__ stage, const uint4 (&w)[2][kSteps],
                                           const uint32_t (&sc)[2][kSteps], f32x4_t (&acc)[2][CT]) const {
    const int lane = threadIdx.x & (kWave - 1), c = lane & 15, q = lane >> 4;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if constexpr (A4) {
        FragH f[2][kSub];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          ChunkRegs ch;
          ch.w = w[g][s];
          ch.s = sc[g][s];
          decode_frags_nvfp4_f16(ch, f[g]);
        }
#pragma unroll
        for (int j = 0; j < kSub; ++j) {
          const uint4* at = stage + c * 16 + (((s * 4 + q) * kSub + j) ^ c);
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            const uint4 b = at[t * 256];
            acc[0][t] = mfma_f16(f[0][j], b, acc[0][t]);
            acc[1][t] = mfma_f16(f[1][j], b, acc[1][t]);
          }
        }
      } else {
        Frag f[2][kSub];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          ChunkRegs ch;
          ch.w = w[g][s];
          ch.s = sc[g][s];
          decode_frags<FMT>(ch, f[g]);
        }
#pragma unroll
        for (int j = 0; j < kSub; ++j) {
          const uint4* at = stage + c * 16 + (((s * 4 + q) * kSub + j) ^ c);
#pragma unroll
          for (int t = 0; t < CT; ++t) {
            const uint4 b = at[t * 256];
            acc[0][t] = mfma_bf16(f[0][j], b, acc[0][t]);
            acc[1][t] = mfma_bf16(f[1][j], b, acc[1][t]);
          }
        }
      }
    }
  }

  // `sum` receives the wavefront's two row groups against mt activation rows (row c: act_rows[c] when given, else c).
  // Rows from mt on repeat row mt - 1; their sums are not stored. Every thread of the block must call.
  __device__ __forceinline__ void run(const TiledRows& rows, int n, int k_, const uint8_t* act_, size_t act_stride_bytes,
                                      const int32_t* act_rows, int act_row0, int mt, const A4Src& a4, const MGeom& g,
                                      uint4* __restrict__ lds0, uint4* __restrict__ lds1, f32x4_t (&sum)[2][CT]) {
    const int lane = threadIdx.x & (kWave - 1);
    k = k_;
    chunks = k / MTraits<FMT>::kLoadElems;
    act = act_;
    act_scales = a4.scales;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = min(rows.row0[i] + (lane & 15), n - 1);   // rows past the end redo the last row
      payload[i] = rows.mat[i].payload;
      off[i] = static_cast<uint32_t>(r) * static_cast<uint32_t>(FmtTraits<FMT>::kIsFp4 ? k / 2 : k);
      sl[i] = scale_lane<FMT>(rows.mat[i], rows.row0[i], n, k);
      cs[i] = rows.mat[i].cs;
    }
#pragma unroll
    for (int i = 0; i < kActRegs; ++i) {
      const int c = min(A4 ? static_cast<int>(threadIdx.x >> 2) + i * (kBlockThreads / 4) : static_cast<int>(threadIdx.x >> 4) + i * 16,
                        mt - 1);
      const size_t row = act_rows ? static_cast<size_t>(act_rows[c]) : static_cast<size_t>(act_row0 + c);
      act_off[i] = static_cast<uint32_t>(row * act_stride_bytes >> 4);
      if constexpr (A4) act_srow[i] = row * a4.scale_stride;
    }
    const int tiles = (g.steps + kSteps - 1) / kSteps;
    const int part_tiles = g.part_steps / kSteps;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < CT; ++t) sum[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[2][CT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < CT; ++t) acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    Regs pre;
    load(0, pre);
    if constexpr (!A4) stage_rows(0, lds0);
    auto step = [&](int t, uint4* __restrict__ cur, uint4* __restrict__ other) {
      if constexpr (A4) commit(cur, pre);
      else __syncthreads();   // `cur` is whole, and its wavefronts are done with `other`
      uint4 w[2][kSteps];
      uint32_t sc[2][kSteps];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          w[i][s] = pre.w[i][s];
          sc[i][s] = pre.s[i][s];
        }
      if (t + 1 < tiles) {
        load(t + 1, pre);
        if constexpr (!A4) stage_rows(t + 1, other);
      }
      if constexpr (A4) __syncthreads();   // the stage is whole; its readers of two tiles before passed the barrier of the tile between
      multiply(cur, w, sc, acc);
    };
    auto add_part = [&](bool first) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          sum[i][t] = first ? acc[i][t] : sum[i][t] + acc[i][t];
          acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    };
    if constexpr (A4) {
      // Codes pass registers, so a stage is chosen by parity; the parts in a loop of their own keep 6 registers more free
      // than the flat loop below (256 experts, 6144 x 2048, 12 / 16 / 60 rows a segment: 2358 -> 2097, 2393 -> 2136, 3364
      // -> 3178 us a layer).
      for (int t0 = 0; t0 < tiles; t0 += part_tiles) {
        const int t1 = min(tiles, t0 + part_tiles);
        for (int t = t0; t < t1; ++t) step(t, t & 1 ? lds1 : lds0, nullptr);
        add_part(t0 == 0);
      }
    } else {
      int part_end = min(tiles, part_tiles);
      auto ends = [&](int done) {
        if (done != part_end) return false;
        add_part(part_end <= part_tiles);
        part_end = min(tiles, part_end + part_tiles);
        return done == tiles;
      };
      for (int t = 0;;) {   // the stages by name: the compiler then knows that a read of one need not wait for loads to the other
        step(t, lds0, lds1);
        if (ends(++t)) break;
        step(t, lds1, lds0);
        if (ends(++t)) break;
      }
    }
    __syncthreads();   // the stages are free for the next pass
  }
};

// Four adjacent weight rows r .. r + 3 of one activation row: one vector store where the row and the end allow it.
template <bool F32>
__device__ __forceinline__ void store4(void* out, size_t at, int r, int n, bool vec, const float (&v)[4]) {
  if constexpr (F32) {
    float* o = static_cast<float*>(out) + at + r;
    if (vec && r + 4 <= n) {
      *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r + i < n) o[i] = v[i];
  } else {
    uint16_t* o = static_cast<uint16_t*>(out) + at + r;
    uint16_t b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = f32_to_bf16(v[i]);
    if (vec && r + 4 <= n) {
      *reinterpret_cast<uint2*>(o) = make_uint2(b[0] | (static_cast<uint32_t>(b[1]) << 16), b[2] | (static_cast<uint32_t>(b[3]) << 16));
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r + i < n) o[i] = b[i];
  }
}

// One pass of a block over a segment's (or a dense batch's) rows c0 .. c0 + mt - 1, stored. GU as in
// mfma_grouped_kernel (a.gate_up 1: SwiGLU to out, 2: gate to out, up to out_up).
struct TiledOut {
  void* out;
  void* out_up;
  size_t out_stride;
  int out_f32;
  int gate_up;
  float limit;
  const float* a4_gs;
};
template <int FMT, bool GU, bool A4, int CT>
__device__ __forceinline__ void tiled_pass(const TiledRows& rows, const float (&divisor)[2], int n, int k, const uint8_t* act,
                                           size_t act_stride_bytes, const int32_t* act_rows, int act_row0, size_t out_row0,
                                           int mt, const A4Src& a4, const MGeom& g, const TiledOut& o, uint4* __restrict__ lds0,
                                           uint4* __restrict__ lds1) {
  TiledPass<FMT, A4, CT> pass;
  f32x4_t sum[2][CT];
  pass.run(rows, n, k, act, act_stride_bytes, act_rows, act_row0, mt, a4, g, lds0, lds1, sum);
  const int lane = threadIdx.x & (kWave - 1);
  const bool vec = ((reinterpret_cast<uintptr_t>(o.out) | (GU ? reinterpret_cast<uintptr_t>(o.out_up) : 0)) & 15u) == 0 &&
                   (o.out_stride & 3u) == 0;
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const int c = t * kTileCols + (lane & 15);
    if (c >= mt) continue;
    const size_t at = (out_row0 + c) * o.out_stride;
    float v[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (A4) {
        const float mul = o.a4_gs[act_rows ? act_rows[c] : act_row0 + c] * (1.0f / divisor[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = sum[i][t][e] * mul;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[i][e] = finish_dot<FMT>(sum[i][t][e], divisor[i]);
      }
    }
    if constexpr (GU) {
      const int r = rows.row0[0] + (lane >> 4) * 4;
      if (o.gate_up == 2) {
        store4<false>(o.out, at, r, n, vec, v[0]);
        store4<false>(o.out_up, at, r, n, vec, v[1]);
      } else {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = bf16_to_f32(swiglu_bf16(v[0][e], v[1][e], o.limit));
        store4<false>(o.out, at, r, n, vec, x);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = rows.row0[i] + (lane >> 4) * 4;
        if (o.out_f32) store4<true>(o.out, at, r, n, vec, v[i]);
        else store4<false>(o.out, at, r, n, vec, v[i]);
      }
    }
  }
}

// The narrowest pass that holds mt rows.
template <int FMT, bool GU, bool A4>
__device__ __forceinline__ void tiled_rows(const TiledRows& rows, const float (&divisor)[2], int n, int k, const uint8_t* act,
                                           size_t act_stride_bytes, const int32_t* act_rows, int act_row0, size_t out_row0,
                                           int mt, const A4Src& a4, const MGeom& g, const TiledOut& o, uint4* __restrict__ lds0,
                                           uint4* __restrict__ lds1) {
  if (mt > 64)
    tiled_pass<FMT, GU, A4, 8>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, lds0, lds1);
  else if (mt > 32)
    tiled_pass<FMT, GU, A4, 4>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, lds0, lds1);
  else
    tiled_pass<FMT, GU, A4, 2>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, lds0, lds1);
}

// Consecutive workgroups go to the eight XCDs in turn. Blocks of one segment share its activation rows and blocks of one
// row tile its weights, so the linear index is dealt such that an XCD (its own L2) keeps a segment's row tiles, or a row
// tile's column passes, to itself.
constexpr int kXcds = 8;

// The grouped launch's blocks. A table's segments go to the XCDs whole, one each in turn. Fewer segments than XCDs - a
// shared expert's, a dense product's by views - and those which the caller knows to be as long as the prompt (a shared
// expert behind the table's) go over all XCDs instead, an eighth of their (row tile, pass) pairs to each, and first, so
// that a long one is no tail: dealt whole, one segment had 32 of the 256 CUs. Measured, us, whole -> spread: one segment,
// block FP8 gate + up, 129 x 17408 x 5120 721 -> 205 (the 16-row form 378), 4096 x 512 x 4096 393 -> 89; NVFP4 product
// 1024 x 2048 x 6144 238 -> 95; whole layers with a shared expert: MXFP4, 256 experts and one in
// the table, 2048 tokens 2167 -> 1312; block FP8, 36 experts, 2048 tokens 739 -> 477. Spreading the up to
// seven segments by which a table misses a multiple of eight as well was slower: their blocks stand for the longest
// possible segment, and most have no pass (36 segments, 2048 tokens 176 -> 213).
struct TiledDeal {
  int whole;          // segments that go to an XCD whole
  int slots;          // blocks that share the passes of one of them and a row tile
  int spread;         // the others, behind them in the table
  int spread_slots;
  int spread_per_xcd; // blocks
  int row_tiles;
  unsigned whole_blocks() const {   // of one slot
    return static_cast<unsigned>((whole + kXcds - 1) / kXcds * kXcds) * static_cast<unsigned>(row_tiles);
  }
  // The grid: x the spread segments' blocks, then a slot's of the whole ones; y the slots. (One index for all would cost every
  // block, those without a pass too, another division: 1 us of a launch.)
  unsigned grid_x() const { return static_cast<unsigned>(spread_per_xcd) * kXcds + whole_blocks(); }
  unsigned grid_y() const { return static_cast<unsigned>(slots > 1 ? slots : 1); }
};
// max_rows: no segment has more; long_segs: so many at the table's end have that many. tuned > 0: slots (bench switch 16).
inline TiledDeal tiled_deal(int n_segs, int long_segs, int row_tiles, int max_rows, int tuned) {
  const int passes = (max_rows + kTiledCols - 1) / kTiledCols;
  auto side_by_side = [&](int64_t blocks) {   // all passes where the blocks of one slot are few, else some
    const int64_t want = tuned > 0 ? tuned : 8192 / blocks;
    return static_cast<int>(want < 1 ? 1 : (want < passes ? want : passes));
  };
  TiledDeal d;
  d.row_tiles = row_tiles;
  d.spread = n_segs < kXcds ? n_segs : long_segs;
  d.whole = n_segs - d.spread;
  d.slots = d.whole ? side_by_side(d.whole_blocks()) : 0;
  d.spread_slots = d.spread ? side_by_side(static_cast<int64_t>(d.spread) * row_tiles) : 0;
  d.spread_per_xcd = (d.spread * row_tiles * d.spread_slots + kXcds - 1) / kXcds;
  return d;
}
struct TiledPlace {
  int seg, tile, slot, slots;   // the block takes passes slot, slot + slots, ... of the segment; seg -1: none
};
__host__ __device__ __forceinline__ TiledPlace tiled_place(const TiledDeal& d, int x, int y) {
  const int xcd = x & (kXcds - 1), idx = (x >> 3) - d.spread_per_xcd;
  if (idx < 0) {
    const int of_seg = d.row_tiles * d.spread_slots, item = xcd * d.spread_per_xcd + (x >> 3);
    if (y > 0 || item >= d.spread * of_seg) return {-1, 0, 0, 1};
    return {d.whole + item / of_seg, item % of_seg / d.spread_slots, item % d.spread_slots, d.spread_slots};
  }
  const int seg = idx / d.row_tiles * kXcds + xcd;
  if (seg >= d.whole) return {-1, 0, 0, 1};
  return {seg, idx % d.row_tiles, y, d.slots};
}
static_assert(kXcds == 8, "the shifts above");

template <int FMT, bool GU, bool A4>
__global__ __launch_bounds__(kBlockThreads, 2) void tiled_grouped_kernel(GroupedArgs a, MGeom g, TiledDeal deal) {
  __shared__ uint4 lds0[kTiledStage], lds1[kTiledStage];
  const TiledPlace at = tiled_place(deal, static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y));
  if (at.seg < 0) return;
  const DgppMoeSegment seg = a.segs[at.seg];
  const int first_pass = at.slot * kTiledCols, tile = at.tile;
  if (first_pass >= seg.rows) return;
  const int wave = threadIdx.x >> 6;
  TiledRows rows;
  float divisor[2];
  const float* gp[2] = {nullptr, nullptr};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rows.mat[i] = mat_of_view<FMT>(a.views[seg.expert * 3 + (GU ? i : a.which)], &gp[i]);
    rows.row0[i] = GU ? (tile * kWavesPerBlock + wave) * kGroupRows : ((tile * kWavesPerBlock + wave) * 2 + i) * kGroupRows;
    divisor[i] = load_divisor<FMT>(gp[i]);
  }
  A4Src src;
  src.scales = a.a4_scales;
  src.scale_stride = a.a4_scale_stride;
  const TiledOut o = {a.out, a.out_up, a.out_stride, a.out_f32, a.gate_up, a.limit, a.a4_gs};
  for (int c0 = first_pass; c0 < seg.rows; c0 += at.slots * kTiledCols) {
    const int first = seg.row0 + c0;
    tiled_rows<FMT, GU, A4>(rows, divisor, a.n, a.k, reinterpret_cast<const uint8_t*>(a.act), A4 ? a.act_stride : a.act_stride * 2,
                            a.act_rows ? a.act_rows + first : nullptr, first, static_cast<size_t>(first),
                            min(kTiledCols, seg.rows - c0), src, g, o, lds0, lds1);
  }
}

// grid.x = kXcds * ceil(row tiles / kXcds) * column passes.
template <int FMT, bool A4>
__global__ __launch_bounds__(kBlockThreads, 2) void tiled_dense_kernel(DenseArgs a, MGeom g, int row_tiles, int passes) {
  __shared__ uint4 lds0[kTiledStage], lds1[kTiledStage];
  const int lin = static_cast<int>(blockIdx.x), idx = lin / kXcds;
  const int tile = idx / passes * kXcds + lin % kXcds, c0 = idx % passes * kTiledCols;
  if (tile >= row_tiles) return;
  const int wave = threadIdx.x >> 6;
  TiledRows rows;
  float divisor[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rows.mat[i] = a.mat;
    rows.row0[i] = ((tile * kWavesPerBlock + wave) * 2 + i) * kGroupRows;
    divisor[i] = load_divisor<FMT>(a.global);
  }
  A4Src src;
  src.scales = a.a4_scales;
  src.scale_stride = a.a4_scale_stride;
  const TiledOut o = {a.out, nullptr, a.out_stride, a.out_f32, 0, 0.f, a.a4_gs};
  tiled_rows<FMT, false, A4>(rows, divisor, a.n, a.k, reinterpret_cast<const uint8_t*>(a.act), A4 ? a.act_stride : a.act_stride * 2,
                             nullptr, c0, static_cast<size_t>(c0), min(kTiledCols, a.m - c0), src, g, o, lds0, lds1);
}

}  // namespace dgpp_amd
