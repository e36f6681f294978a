// The matrix-core form for many activation rows (prompt chunks): a block multiplies 128 weight rows with up to 128
// activation rows, so a weight is fetched and decoded once per 128 activation rows instead of once per 16
// (gemv_mfma_kernels.hpp). Included by gemv_kernels.hpp after the argument structs.
//
// With 16 rows per pass a prompt of T tokens decodes every weight T / 16 times and gathers the activations again for
// every 64 weight rows: the vector ALU and the gathers, not the matrix core, were the time. Here a wavefront owns two row
// groups (16 weight rows each) and CT column tiles: per 32 elements of k it decodes two operands and runs 2 CT MFMAs on
// them, and reads CT operands from LDS.
//
// Tile. k advances by one step of a row group, 128 elements (FP4) or 64 (FP8). Weights are of one wavefront and go to its
// registers, three tiles ahead of their use, two for the widest pass with NVFP4 activations; the block's activation rows
// go into a ring of LDS stages, three tiles ahead as well (BF16: from memory to LDS without passing registers) where four
// stages leave room for two blocks per CU, one tile ahead for FP4's widest pass. One barrier per tile, which waits for
// those of a wavefront's loads that the tile needs and no others (in the last turn, of up to three tiles, for all): waiting for all
// of them, the form before this one had one tile on its way and took the latency of a load per tile.
//
// Lanes. The matrix core wants 16 rows in 16 adjacent lanes, the memory pipe adjacent lanes in one row. Weights are
// therefore asked for row by row (four lanes to the 64 bytes of a row's tile), the FP4 scales of four tiles at once, and
// both pass through a region of LDS of the wavefront's own. The places in the stages and in that region are turned such
// that sixteen lanes that read together meet no bank twice (SQ_LDS_BANK_CONFLICT 0; before, half of the LDS cycles for FP4).
// Measured, us, uniform segments, lanes in the matrix core's order -> row by row: MXFP4 gate + up, 256 x 2 x 1024 x 4096, 16
// rows 323 -> 271, 64 388 -> 351, 128 538 -> 550; NVFP4 activations, 256 x 2048 x 6144, 16 rows 557 -> 439.
//
// What bounds it: at 128 rows a pass the matrix core and the LDS together (a read feeds two MFMAs; dense block FP8
// 1000 x 12288 x 6144 MFMA 42 % busy with a quarter of the places empty in the last round); at 16 rows the memory pipe,
// 4.2 TB/s for FP4 and 4.9 for FP8, with two blocks per CU.
// From the form before (a tile ahead, waiting for all): block FP8 gate + up, 128 x 2 x 768 x 2048, 777 tokens 193 -> 141 us,
// down 146 -> 80; MXFP4, 2048 tokens 744 -> 582 and 445 -> 339; NVFP4, 288 experts, 4096 x 512, 4096 tokens 706 -> 549 and
// 566 -> 401; NVFP4 activations, 512 tokens 708 -> 482; dense block FP8 1000 x 12288 x 6144 190 -> 166.
//
// Arithmetic. The sums of a (weight row, activation row) pair are those of the 16-row form: the same elements in the
// same MFMAs, K parts on their own, added in ascending order. A call's bits do not depend on which form takes it.
#pragma once

#include <type_traits>

#include "gemv_mfma_kernels.hpp"
#include "moe_rank.hpp"

namespace dgpp_amd {

constexpr int kTiledCols = 128;                   // activation rows of the widest pass
constexpr int kHalfCols = 64;
constexpr int kNarrowCols = 32;                   // of the kernel for short segments
constexpr int kTiledRows = 128;                   // weight rows of a block (gate + up: 64 of each)

// The two row groups of a wavefront: two groups of one matrix, or one of gate and one of up.
struct TiledRows {
  MatRef mat[2];
  int row0[2];
};

// All but the newest N of this wavefront's loads have arrived (a load to LDS with them), then the block's barrier. The
// stage that is read next is whole when every wavefront has waited for its own loads to it.
template <int N>
__device__ __forceinline__ void tiled_barrier() {
  __builtin_amdgcn_sched_barrier(0);   // nothing of the next tile comes forward: it would wait for loads of that tile here
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// RING: the LDS stages that the activation rows' tiles take in turn.
template <int FMT, bool A4, int CT, int RING>
struct TiledPass {
  static constexpr int kSub = MTraits<FMT>::kSub;
  static constexpr int kTileElems = MTraits<FMT>::kStepElems;        // elements of k of a tile: 128 (FP4) or 64 (FP8)
  static constexpr int kUnits = kTileElems / 8;                      // 16-byte units of a staged row
  static constexpr int kCols = CT * kTileCols;
  static constexpr int kRowLoads = kCols * kUnits / kBlockThreads;   // loads to LDS per thread and tile (BF16 rows)
  static constexpr int kCodeLoads = (kCols * 4 + kBlockThreads - 1) / kBlockThreads;   // 32-code loads per thread (A4)
  static constexpr int kActRegs = A4 ? kCodeLoads : kRowLoads;
  static_assert(A4 ? RING == 2 : RING == 2 || RING == 4, "tiles and stages are named in turns of four");
  static_assert(kRowLoads >= 1 && kRowLoads * kBlockThreads == kCols * kUnits, "whole loads");

  struct Regs {          // one tile on its way
    uint4 w[2];
    uint32_t s[2];
    uint4 act[A4 ? kCodeLoads : 1];
    uint32_t act_s[A4 ? kCodeLoads : 1];
  };

  // Weights are asked for row by row - lane l takes 16 bytes of row l / 4 - and pass through LDS of the wavefront's own into
  // the layout of the matrix core, lane (r, q) quarter q of row r; FP4 scales come for a turn of four tiles at once, a
  // tile's to a lane, the same way.
  static constexpr bool kFp4 = FmtTraits<FMT>::kIsFp4;
  static constexpr int kTileScale = FMT == kFmtNvfp4 ? 8 : 4;   // FP4: bytes of a row's scales of a tile
  using ScaleWord = std::conditional_t<FMT == kFmtNvfp4, uint2, uint32_t>;
  struct Exchange {
    uint4 w[2][64];
    ScaleWord s[kFp4 ? 2 : 1][kFp4 ? 64 : 1];
  };

  const uint8_t* payload[2];
  const uint8_t* scales[2];
  uint32_t off[2], soff[2];      // bytes: this lane's piece of the row it loads, of the first tile; the scales it loads
  uint32_t scale_bytes;          // FP4: of the matrix
  uint32_t row_at[2];            // rows that this lane multiplies
  int cs[2];
  const uint8_t* act;            // bytes; without a row list the pass's first row
  const uint8_t* act_scales;
  size_t act_off[kActRegs];      // bytes from `act`: the row, and of the row this thread's unit of the first tile
  size_t act_srow[A4 ? kCodeLoads : 1];
  int k, chunks, tid;

  // The place of sub-operand j of quarter q in row r of a stage: FP4 quarters at 0, 12, 4 and 8, FP8 ones side by side, the
  // row's number folded in. (A read instruction takes sixteen lanes at a time: eight rows of one quarter, the other eight
  // of the next. With the quarters in memory's order those met in pairs for FP4: half of the LDS cycles.)
  __device__ static __forceinline__ int fold(int r) { return kSub == 4 ? r & 15 : (r >> 1) & 7; }
  __device__ static __forceinline__ int place(int q, int j, int r) {
    return (kSub == 4 ? ((q >> 1) ^ ((q & 1) * 3)) * 4 + j : j * 4 + q) ^ fold(r);
  }
  __device__ static __forceinline__ int unit_at(int p, int r) {   // the unit of row r that belongs at place p
    const int at = p ^ fold(r), x = at >> 2;
    return kSub == 4 ? (((x & 1) * 2) ^ ((x >> 1) * 3)) * 4 + (at & 3) : (at & 3) * 2 + x;
  }

  typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
  template <class T>
  __device__ static __forceinline__ T global_at(const uint8_t* base, uint32_t byte) {
    return *(const __attribute__((address_space(1))) T*)(uintptr_t)(base + byte);
  }
  // The loads of the walk are buffer loads: the tile's offset is a scalar, a buffer of no bytes is one that reads nothing,
  // and the compiler counts those to LDS among the others (after a global_load_lds it waits for every load).
  __device__ static __forceinline__ const uint8_t* uniform(const void* p) {
    const uint64_t v = reinterpret_cast<uintptr_t>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<const uint8_t*>(static_cast<uintptr_t>(static_cast<uint64_t>(hi) << 32 | lo));
  }
  __device__ static __forceinline__ __amdgpu_buffer_rsrc_t buffer(const uint8_t* base, bool live) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, live ? 0xfffffff0u : 0u, 0x00027000);
  }

  // Block-FP8 scales come in whole words and are taken out of them where they are used: a byte that is carried over a loop as
  // it was loaded gets its upper bits cleared, and waited for, at the loop's end.
  __device__ __forceinline__ uint32_t fp8_scale_byte(int g, int tile) const {   // of a block-FP8 piece, from scales[g]
    const uint32_t col = (static_cast<uint32_t>(tile) * 64u + (static_cast<uint32_t>(tid & 63) >> 4) * 16u) >> cs[g];
    return soff[g] + col * (FMT == kFmtFp8F32 ? 4u : 1u);
  }
  __device__ __forceinline__ uint32_t fp8_scale_word(int g, int tile, bool live) const {
    uint32_t at = fp8_scale_byte(g, tile);
    const uint8_t* base = scales[g];
    if constexpr (FMT == kFmtFp8E8M0) {   // the aligned word that holds the byte
      const uint32_t low = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(base) & 3u);
      at = (at + low) & ~3u;
      base -= low;
    }
    return __builtin_amdgcn_raw_buffer_load_b32(buffer(base, live), at, 0, 0);
  }
  __device__ __forceinline__ uint32_t fp8_scale_shift(int g, int tile) const {
    if constexpr (FMT == kFmtFp8E8M0)
      return ((fp8_scale_byte(g, tile) + static_cast<uint32_t>(reinterpret_cast<uintptr_t>(scales[g]))) & 3u) * 8u;
    else return 0u;
  }
  __device__ __forceinline__ uint32_t scale_of(int g, int tile, uint32_t word) const {   // ChunkRegs::s
    if constexpr (FMT == kFmtFp8E8M0) return (word >> fp8_scale_shift(g, tile)) & 0xffu;
    else return word;
  }

  // The FP4 scales of the turn that starts at `tile`: this lane's tile of it. Past the matrix's end zeros come, and where a
  // turn passes the end of k what follows; nobody uses either.
  __device__ __forceinline__ void load_scales(int tile, ScaleWord (&to)[2]) const {
    if constexpr (kFp4) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(scales[g]), 0, scale_bytes, 0x00027000);
        if constexpr (FMT == kFmtNvfp4) {
          typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
          const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(b, soff[g], tile * kTileScale, 0);
          to[g] = make_uint2(v.x, v.y);
        } else {
          to[g] = __builtin_amdgcn_raw_buffer_load_b32(b, soff[g], tile * kTileScale, 0);
        }
      }
    }
  }
  // Lane l writes the 16 bytes that it loaded to place l of a group's region; which piece of row l / 4 that is, is turned by
  // the row.
  __device__ static __forceinline__ int turned(int r) { return (0x1320 >> ((r >> 2) & 3) * 4) & 3; }
  __device__ __forceinline__ void put_scales(Exchange& x, const ScaleWord (&from)[2]) const {
    if constexpr (kFp4) {
#pragma unroll
      for (int g = 0; g < 2; ++g) x.s[g][tid & 63] = from[g];
    }
  }
  // A tile's weights, from as they were loaded to as they are multiplied, and its FP4 scales (`at`: which tile of its turn).
  // LOADS: loads to LDS may be on their way. A scale is then read as the word that was written: a read of its bytes could, for
  // the compiler, be one of the stage that is being loaded, and waited for every load (MXFP4 2048 tokens 854 us for 833 so).
  template <bool LOADS = !A4>
  __device__ __forceinline__ void exchange(Exchange& x, int at, Regs& r) const {
    const int lane = tid & 63, row = lane & 15, q = lane >> 4;
#pragma unroll
    for (int g = 0; g < 2; ++g) x.w[g][lane] = r.w[g];
#pragma unroll
    for (int g = 0; g < 2; ++g) r.w[g] = x.w[g][row * 4 + (q ^ turned(row))];
    if constexpr (kFp4) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        if constexpr (LOADS) {
          const ScaleWord w = x.s[g][row * 4 + at];
          if constexpr (FMT == kFmtNvfp4) r.s[g] = ((q & 2) != 0 ? w.y : w.x) >> (q & 1) * 16 & 0xffffu;
          else r.s[g] = w >> q * 8 & 0xffu;
        } else {
          const uint8_t* p = reinterpret_cast<const uint8_t*>(x.s[g]) + (row * 4 + at) * kTileScale;
          if constexpr (FMT == kFmtNvfp4) r.s[g] = *reinterpret_cast<const uint16_t*>(p + q * 2);
          else r.s[g] = p[q];
        }
      }
    }
  }

  // A whole tile's weights and NVFP4 rows into registers, its BF16 rows to a stage. No branch around the loads: the waits
  // count them. Past the last whole tile they read nothing, and nobody uses it.
  __device__ __forceinline__ void load(int tile, int full, Regs& r) const {
    const bool live = tile < full;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(buffer(payload[g], live), off[g], tile * 64, 0);
      r.w[g] = make_uint4(v.x, v.y, v.z, v.w);
    }
    if constexpr (!kFp4) {
#pragma unroll
      for (int g = 0; g < 2; ++g) r.s[g] = fp8_scale_word(g, tile, live);
    }
    if constexpr (A4) {
#pragma unroll
      for (int i = 0; i < kCodeLoads; ++i) {
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(buffer(act, live), static_cast<uint32_t>(act_off[i]), tile * 64, 0);
        r.act[i] = make_uint4(v.x, v.y, v.z, v.w);
        r.act_s[i] = __builtin_amdgcn_raw_buffer_load_b32(buffer(act_scales, live), static_cast<uint32_t>(act_srow[i]), tile * 8, 0);
      }
    }
  }
  // The BF16 rows go from memory to LDS without passing registers: a wavefront's lanes fill 64 places in a row, so it is
  // the lane that reads the unit which belongs there.
  __device__ __forceinline__ void stage_rows(int tile, int full, uint4* __restrict__ stage) const {
    const int first = __builtin_amdgcn_readfirstlane(tid >> 6) * kWave;
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(act, tile < full), (__attribute__((address_space(3))) void*)(stage + first + i * kBlockThreads),
                                               16, static_cast<uint32_t>(act_off[i]), tile * kUnits * 16, 0, 0);
  }

  // The part of a tile past the last whole one (k is no multiple of it): zeros past the end of the rows.
  __device__ __forceinline__ void load_rest(int tile, Regs& r) const {
    const int q = (tid & (kWave - 1)) >> 4;
    const bool inside = tile * 4 + q < chunks;
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      r.w[g] = make_uint4(0u, 0u, 0u, 0u);
      r.s[g] = 0u;
      if (inside) {
        const u32x4_t v = global_at<u32x4_t>(payload[g] + static_cast<size_t>(tile) * 64, row_at[g] * static_cast<uint32_t>(kFp4 ? k / 2 : k) + q * 16u);
        r.w[g] = make_uint4(v.x, v.y, v.z, v.w);
        const uint32_t at = row_at[g] * static_cast<uint32_t>(k / (FMT == kFmtNvfp4 ? 16 : 32)) + static_cast<uint32_t>(tile) * kTileScale;
        if constexpr (FMT == kFmtFp8F32) r.s[g] = fp8_scale_word(g, tile, true);
        else if constexpr (FMT == kFmtNvfp4) r.s[g] = global_at<uint16_t>(scales[g], at + q * 2);
        else if constexpr (FMT == kFmtMxfp4) r.s[g] = global_at<uint8_t>(scales[g], at + q);
        else r.s[g] = static_cast<uint32_t>(global_at<uint8_t>(scales[g], fp8_scale_byte(g, tile))) << fp8_scale_shift(g, tile);
      }
    }
    if constexpr (A4) {
      const int piece = tid & 3;
#pragma unroll
      for (int i = 0; i < kCodeLoads; ++i) {
        r.act[i] = make_uint4(0u, 0u, 0u, 0u);
        r.act_s[i] = 0u;
        if (tile * kTileElems + piece * 32 < k) {
          r.act[i] = *reinterpret_cast<const uint4*>(act + act_off[i] + tile * 64);
          r.act_s[i] = static_cast<uint32_t>(*reinterpret_cast<const uint16_t*>(act_scales + act_srow[i] + tile * 8 + (piece & 1) * 2)) << (piece & 1) * 16;
        }
      }
    }
  }
  __device__ __forceinline__ void stage_rest(int tile, uint4* __restrict__ stage) const {
    const int u = unit_at(tid % kUnits, tid / kUnits);
#pragma unroll
    for (int i = 0; i < kRowLoads; ++i) {
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (tile * kTileElems + u * 8 < k)
        v = *reinterpret_cast<const uint4*>(act + act_off[i] + tile * kUnits * 16);
      stage[tid + i * kBlockThreads] = v;
    }
  }

  __device__ __forceinline__ void commit(uint4* __restrict__ stage, const Regs& r) const {
    if constexpr (A4) {
      const int piece = tid & 3;
#pragma unroll
      for (int i = 0; i < kCodeLoads; ++i) {
        const int row = (tid >> 2) + i * (kBlockThreads / 4);
        if (kCols * 4 >= kBlockThreads || row < kCols) {
          ChunkRegs ch;
          ch.w = r.act[i];
          ch.s = r.act_s[i] >> (piece & 1) * 16;
          FragH f[4];
          decode_frags_nvfp4_f16(ch, f);
#pragma unroll
          for (int j = 0; j < 4; ++j) stage[row * kUnits + place(piece, j, row)] = __builtin_bit_cast(uint4, f[j].v);
        }
      }
    }
  }

  // A use of a tile's weights and scales that costs nothing once they have arrived.
  __device__ __forceinline__ void keep(const Regs& r) const {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      asm volatile("" ::"v"(r.w[g].x), "v"(r.w[g].y), "v"(r.w[g].z), "v"(r.w[g].w));
      if constexpr (!kFp4) asm volatile("" ::"v"(r.s[g]));
    }
  }

  // The products of a tile. The operands from LDS are asked for kAhead products early, in an order that the compiler is held
  // to: left alone it reads one, waits for it and uses it, with one other wavefront on the SIMD to cover the wait.
  static constexpr int kAhead = CT < 4 ? CT * 2 : 4;
  template <class Middle>
  __device__ __forceinline__ void multiply(int tile, const uint4* __restrict__ stage, const Regs& r, f32x4_t (&acc)[2][CT], Middle middle) const {
    const int lane = tid & (kWave - 1), c = lane & 15, q = lane >> 4;
    using F = std::conditional_t<A4, FragH, Frag>;
    F f[2][kSub];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      ChunkRegs ch;
      ch.w = r.w[g];
      ch.s = scale_of(g, tile, r.s[g]);
      if constexpr (A4) decode_frags_nvfp4_f16(ch, f[g]);
      else decode_frags<FMT>(ch, f[g]);
    }
    const uint4* at[kSub];
#pragma unroll
    for (int j = 0; j < kSub; ++j) at[j] = stage + c * kUnits + place(q, j, c);
    constexpr int kReads = kSub * CT;
    uint4 b[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) b[i] = at[i / CT][i % CT * kTileCols * kUnits];
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      const int j = i / CT, t = i % CT, n = i + kAhead;
      if (i == kReads / 2) middle();
      if constexpr (A4) {
        acc[0][t] = mfma_f16(f[0][j], b[i % kAhead], acc[0][t]);
        acc[1][t] = mfma_f16(f[1][j], b[i % kAhead], acc[1][t]);
      } else {
        acc[0][t] = mfma_bf16(f[0][j], b[i % kAhead], acc[0][t]);
        acc[1][t] = mfma_bf16(f[1][j], b[i % kAhead], acc[1][t]);
      }
      if (n < kReads) b[i % kAhead] = at[n / CT][n % CT * kTileCols * kUnits];
    }
    __builtin_amdgcn_sched_group_barrier(0x100, kAhead, 0);   // reads from LDS
#pragma unroll
    for (int i = 0; i < kReads; ++i) {
      if (i == kReads / 2) {
        __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);    // the middle's writes to LDS and reads from it
        __builtin_amdgcn_sched_group_barrier(0x100, kFp4 ? 4 : 2, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);      // products
      if (i + kAhead < kReads) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  }

  __device__ __forceinline__ void set_weights(const TiledRows& rows, int n, int k_) {   // once tid is set
    const int lane = tid & (kWave - 1);
    k = k_;
    chunks = k / MTraits<FMT>::kLoadElems;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      payload[i] = uniform(rows.mat[i].payload);
      scales[i] = uniform(rows.mat[i].scales);
      cs[i] = rows.mat[i].cs;
      // rows past the end redo the last row
      const uint32_t r = static_cast<uint32_t>(min(rows.row0[i] + (lane >> 2), n - 1));
      row_at[i] = static_cast<uint32_t>(min(rows.row0[i] + (lane & 15), n - 1));
      off[i] = r * static_cast<uint32_t>(kFp4 ? k / 2 : k) + static_cast<uint32_t>((lane & 3) ^ turned(lane >> 2)) * 16u;
      if constexpr (kFp4) soff[i] = r * static_cast<uint32_t>(k / (FMT == kFmtNvfp4 ? 16 : 32)) + static_cast<uint32_t>(lane & 3) * kTileScale;
      else soff[i] = (row_at[i] >> rows.mat[i].rs) * ((static_cast<uint32_t>(k) + (1u << cs[i]) - 1) >> cs[i]) * (FMT == kFmtFp8F32 ? 4u : 1u);
    }
    scale_bytes = static_cast<uint32_t>(n) * static_cast<uint32_t>(k / (FMT == kFmtNvfp4 ? 16 : 32));
  }

  // `sum` receives the wavefront's two row groups against mt activation rows (row c: act_rows[c] when given, else c).
  // Rows from mt on repeat row mt - 1; their sums are not stored. Every thread of the block must call.
  __device__ __forceinline__ void run(const TiledRows& rows, int n, int k_, const uint8_t* act_, size_t act_stride_bytes,
                                      const int32_t* act_rows, int act_row0, int mt, const A4Src& a4, const MGeom& g,
                                      uint4* __restrict__ s0, uint4* __restrict__ s1, uint4* __restrict__ s2,
                                      uint4* __restrict__ s3, Exchange& __restrict__ x, f32x4_t (&sum)[2][CT]) {
    // A loop over passes would otherwise keep what every width computes from the thread's number in registers around all of them.
    tid = static_cast<int>(threadIdx.x);
    asm volatile("" : "+v"(tid));
    const int lane = tid & (kWave - 1);
    set_weights(rows, n, k_);
    act = uniform(act_ + (act_rows ? 0 : static_cast<size_t>(act_row0) * act_stride_bytes));
    if constexpr (A4) act_scales = uniform(a4.scales + (act_rows ? 0 : static_cast<size_t>(act_row0) * a4.scale_stride));
#pragma unroll
    for (int i = 0; i < kActRegs; ++i) {
      const int c = min(A4 ? (tid >> 2) + i * (kBlockThreads / 4) : tid / kUnits + i * (kBlockThreads / kUnits), mt - 1);
      const size_t row = static_cast<size_t>(act_rows ? act_rows[c] : c);
      if constexpr (A4) {
        act_off[i] = row * act_stride_bytes + (tid & 3) * 16;
        act_srow[i] = row * a4.scale_stride + (tid & 2) * 2;
      } else {
        act_off[i] = row * act_stride_bytes + unit_at(tid % kUnits, tid / kUnits) * 16;   // rows 256 / kUnits apart fold alike
      }
    }
    // A buffer load reaches 4 GB: a pass with a row that ends beyond takes the way of the last part of k all along.
    bool far = false;
    for (int c = lane; c < mt; c += kWave) {
      const size_t row = static_cast<size_t>(act_rows ? act_rows[c] : c);
      far = far || row * act_stride_bytes + static_cast<size_t>(k) * 2 > 0xfffffff0u || (A4 && row * a4.scale_stride + k > 0xfffffff0u);
    }
    const int full = __builtin_amdgcn_readfirstlane(__builtin_amdgcn_ballot_w64(far) != 0 ? 0 : k / kTileElems), part_tiles = g.part_steps;
    f32x4_t acc[2][CT];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int t = 0; t < CT; ++t) acc[i][t] = sum[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    auto add_part = [&](bool first) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          sum[i][t] = first ? acc[i][t] : sum[i][t] + acc[i][t];
          acc[i][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    };
    Regs r0, r1, r2, r3;
    ScaleWord sraw[2];
    // Tiles of weights on their way. The widest pass with codes has two and 32 bytes of scratch a lane as it is, its 32-row form 12, NVFP4's
    // plain 128-row form 8; the others none.
    constexpr int kDeep = A4 && CT == 8 ? 2 : 3;
    // One tile: its stage is whole and the one that is filled next is free after the barrier. Of a wavefront's loads
    // those may still be on their way then that are younger than its loads to the stage: the weights (and block-FP8 scales)
    // that followed those, and what the RING - 2 steps between asked for. (The FP4 scales of a turn are not counted: where
    // they are among them, up to two fewer may be left.)
    // The count stands on every one of those loads being in the program. Those of a whole turn are, all of them are read
    // on both ways out of the loop below. Those of the last turn are not: what it asks for past the last tile nobody reads,
    // and the compiler leaves out as much of it as it can tell. Its steps, three of a pass at most, wait for everything.
    constexpr int kTileLoads = kFp4 ? 2 : 4;
    constexpr int kYounger = kTileLoads + (RING - 2) * (kRowLoads + kTileLoads);
    auto step = [&](int t, auto at, auto last, const uint4* __restrict__ cur, uint4* __restrict__ next, const Regs& now, Regs& coming,
                    Regs& far) {
      constexpr int kAt = decltype(at)::value;   // in its turn
      if constexpr (A4) {
        tiled_barrier<63>();
      } else {
        tiled_barrier<decltype(last)::value ? 0 : kYounger>();
        stage_rows(t + RING - 1, full, next);
        asm volatile("" ::: "memory");   // the weights are asked for after the rows: kYounger
      }
      load(t + kDeep, full, far);
      if constexpr (kAt == 0) load_scales(t + 4, sraw);
      if constexpr (A4) commit(next, coming);
      multiply(t, cur, now, acc, [&] {
        if constexpr (kAt == 3) put_scales(x, sraw);
        exchange(x, (kAt + 1) & 3, coming);
      });
    };
    if (full > 0) {
      if constexpr (A4) {
        load(0, full, r0);
        load(1, full, r1);
        if constexpr (kDeep == 3) load(2, full, r2);
        commit(s0, r0);
        load_scales(0, sraw);
      } else if constexpr (RING == 2) {
        load_scales(0, sraw);
        load(0, full, r0);
        load(1, full, r1);
        asm volatile("" ::: "memory");
        stage_rows(0, full, s0);
        asm volatile("" ::: "memory");
        load(2, full, r2);
      } else {
        uint4* const st[3] = {s0, s1, s2};
        Regs* const reg[3] = {&r0, &r1, &r2};
        load_scales(0, sraw);
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          stage_rows(t, full, st[t]);
          asm volatile("" ::: "memory");
          load(t, full, *reg[t]);
          asm volatile("" ::: "memory");
        }
      }
      put_scales(x, sraw);
      exchange(x, 0, r0);
      // The stages and the tiles by name, in turns of four, and one way out of the loop: the compiler then waits for what a
      // step reads and no more.
      int t = 0, part_end = part_tiles;
      auto turn = [&](int steps, auto last) {   // whole: four steps; the last: one to three
        step(t, std::integral_constant<int, 0>{}, last, s0, RING == 2 ? s1 : s3, r0, r1, kDeep == 2 ? r2 : r3);
        if (steps == 1) return;
        step(t + 1, std::integral_constant<int, 1>{}, last, s1, s0, r1, r2, kDeep == 2 ? r3 : r0);
        if (steps == 2) return;
        step(t + 2, std::integral_constant<int, 2>{}, last, RING == 2 ? s0 : s2, s1, r2, r3, kDeep == 2 ? r0 : r1);
        if constexpr (!decltype(last)::value)
          step(t + 3, std::integral_constant<int, 3>{}, last, RING == 2 ? s1 : s3, RING == 2 ? s0 : s2, r3, r0, kDeep == 2 ? r1 : r2);
      };
      for (; t + 4 <= full;) {
        turn(4, std::false_type{});
        t += 4;
        if (t == part_end) {   // parts are whole turns
          add_part(t == part_tiles);
          part_end += part_tiles;
        }
      }
      if (t < full) turn(full - t, std::true_type{});
      tiled_barrier<0>();   // nothing is on its way to a stage, and no wavefront reads one
      if constexpr (!A4) {
        if (t == full) {    // what the last whole turn asked for is read here, by an instruction that is none (kYounger)
          keep(r0);
          keep(r1);
          keep(r2);
        }
      }
    }
    for (int t = full; t < g.steps; ++t) {
      load_rest(t, r0);
      if constexpr (A4) commit(s0, r0);
      else stage_rest(t, s0);
      __syncthreads();
      multiply(t, s0, r0, acc, [] {});
      __syncthreads();
      if ((t + 1) % part_tiles == 0 || t + 1 == g.steps) add_part(t < part_tiles);
    }
    if (full == g.steps && full % part_tiles != 0) add_part(full < part_tiles);
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
// A block's LDS stages, as large as the widest pass wants them: four, two where the rows pass registers (A4) and where four
// would leave room for one block per CU.
template <int FMT, bool A4, int COLS>
struct TiledStages {
  static constexpr int kUnits = COLS * MTraits<FMT>::kStepElems / 8;
  static constexpr int kRing = A4 || kUnits > 1024 ? 2 : 4;
  uint4 *s0, *s1, *s2, *s3;
  typename TiledPass<FMT, A4, COLS / kTileCols, kRing>::Exchange* x;   // of each wavefront
};
template <int FMT, bool GU, bool A4, int CT, int COLS>
__device__ __forceinline__ void tiled_pass(const TiledRows& rows, const float (&divisor)[2], int n, int k, const uint8_t* act,
                                           size_t act_stride_bytes, const int32_t* act_rows, int act_row0, size_t out_row0,
                                           int mt, const A4Src& a4, const MGeom& g, const TiledOut& o,
                                           const TiledStages<FMT, A4, COLS>& st) {
  TiledPass<FMT, A4, CT, TiledStages<FMT, A4, COLS>::kRing> pass;
  f32x4_t sum[2][CT];
  pass.run(rows, n, k, act, act_stride_bytes, act_rows, act_row0, mt, a4, g, st.s0, st.s1, st.s2, st.s3,
           reinterpret_cast<typename TiledPass<FMT, A4, CT, TiledStages<FMT, A4, COLS>::kRing>::Exchange&>(st.x[threadIdx.x >> 6]), sum);
  const int lane = pass.tid & (kWave - 1);
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
template <int FMT, bool GU, bool A4, int COLS>
__device__ __forceinline__ void tiled_rows(const TiledRows& rows, const float (&divisor)[2], int n, int k, const uint8_t* act,
                                           size_t act_stride_bytes, const int32_t* act_rows, int act_row0, size_t out_row0,
                                           int mt, const A4Src& a4, const MGeom& g, const TiledOut& o,
                                           const TiledStages<FMT, A4, COLS>& st) {
  if constexpr (COLS == kNarrowCols)
    tiled_pass<FMT, GU, A4, 2>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, st);
  else if (COLS > 64 && mt > 64)
    tiled_pass<FMT, GU, A4, COLS / kTileCols>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, st);
  else if (mt > 32)
    tiled_pass<FMT, GU, A4, 4>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, st);
  else
    tiled_pass<FMT, GU, A4, 2>(rows, divisor, n, k, act, act_stride_bytes, act_rows, act_row0, out_row0, mt, a4, g, o, st);
}

// The kernel's stages and exchange regions, by name.
#define DGPP_TILED_STAGES(st, FMT, A4, COLS)                                                                         \
  using Stages = TiledStages<FMT, A4, COLS>;                                                                         \
  __shared__ uint4 stage0[Stages::kUnits], stage1[Stages::kUnits];                                                   \
  __shared__ uint4 stage2[Stages::kRing == 4 ? Stages::kUnits : 1], stage3[Stages::kRing == 4 ? Stages::kUnits : 1]; \
  __shared__ typename TiledPass<FMT, A4, COLS / kTileCols, Stages::kRing>::Exchange exchange[kWavesPerBlock];         \
  const Stages st = {stage0, stage1, stage2, stage3, exchange}

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
// cols: rows of a pass.
inline TiledDeal tiled_deal(int n_segs, int long_segs, int row_tiles, int max_rows, int tuned, int cols = kTiledCols) {
  const int passes = (max_rows + cols - 1) / cols;
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

// A table whose rows the caller knows the number of: its passes sorted by width, the widest first, and dealt to the XCDs in
// turn. Segments differ by an order of magnitude (2048 tokens over 256 experts: a quarter have up to 16 rows, a tenth more
// than 128); dealt in the table's order, the places of the chip were filled to 70 % on average: the XCDs' shares differ, and
// wide passes come last. Every block sorts for itself, while it would wait for its segment anyway: a segment has `rows / 128`
// full passes and a rest, a thread counts those of its segments by class (more than 64, more than 32, fewer rows), a prefix sum
// over the block says whose the item is. Measured, us, the table's order -> sorted: MXFP4 gate + up, 2048 tokens 582 -> 475,
// down 339 -> 323; NVFP4, 288 experts, 4096 tokens 549 -> 430; block FP8, 128 experts, 777 tokens 141 -> 132 and 80 -> 77.
struct TiledPlan {
  TiledDeal deal;
  int items;          // 0: by the deal; else no fewer than there are passes, a multiple of the XCDs
  int n_segs;
  dim3 grid() const {
    return items > 0 ? dim3(static_cast<unsigned>(items) * static_cast<unsigned>(deal.row_tiles)) : dim3(deal.grid_x(), deal.grid_y());
  }
};
constexpr int kSortedSegs = 1 << 15;            // sorted_item counts segments in the halves of a word
constexpr int64_t kSortedBlocks = 1 << 24;      // a launch takes fewer than 2^32 threads
// Sorted once every XCD has several items; with fewer, where the rows are not known and beyond what it counts, by the deal.
inline TiledPlan tiled_plan(int n_segs, int long_segs, int row_tiles, int max_rows, int64_t total_rows, int tuned, int cols) {
  int64_t items = total_rows > 0 && tuned == 0 ? n_segs + total_rows / cols : 0;
  if (items < 8 * kXcds || n_segs >= kSortedSegs) items = 0;
  items = (items + kXcds - 1) / kXcds * kXcds;
  if (items >= kSortedBlocks || items * row_tiles >= kSortedBlocks) items = 0;
  return {tiled_deal(n_segs, long_segs, row_tiles, max_rows, tuned, cols), static_cast<int>(items), n_segs};
}
struct TiledItem {
  int expert, row0, rows;
};
template <int COLS>
__device__ __forceinline__ bool sorted_item(const DgppMoeSegment* segs, int n_segs, int item, TiledItem& out) {
  __shared__ int totals[2][kWavesPerBlock], found[2];
  const int tid = static_cast<int>(threadIdx.x), wave = tid >> 6;
  int wide = 0, rest = 0;   // passes more than half full; more than a quarter (upper half) and less
  auto wide_of = [](int rows) { return rows / COLS + (rows % COLS > COLS / 2 ? 1 : 0); };
  auto rest_of = [](int rows) {
    const int r = rows % COLS;
    return r > COLS / 2 ? 0 : r > COLS / 4 ? 1 << 16 : r > 0 ? 1 : 0;
  };
  for (int s = tid; s < n_segs; s += kBlockThreads) {
    const int rows = segs[s].rows;
    wide += wide_of(rows);
    rest += rest_of(rows);
  }
  int wide_before = wave_prefix_incl(wide), rest_before = wave_prefix_incl(rest);
  if ((tid & (kWave - 1)) == kWave - 1) {
    totals[0][wave] = wide_before;
    totals[1][wave] = rest_before;
  }
  if (tid < 2) found[tid] = -1;
  __syncthreads();
  wide_before -= wide;
  rest_before -= rest;
  int all_wide = 0, all_rest = 0;
#pragma unroll
  for (int w = 0; w < kWavesPerBlock; ++w) {
    if (w < wave) wide_before += totals[0][w], rest_before += totals[1][w];
    all_wide += totals[0][w];
    all_rest += totals[1][w];
  }
  int shift = 16, before = 0;   // of a narrower pass
  if (item >= all_wide) {
    item -= all_wide;
    if (item >= all_rest >> 16) {
      item -= all_rest >> 16;
      shift = 0;
    }
    before = rest_before >> shift & 0xffff;
    if (item >= before && item < before + (rest >> shift & 0xffff)) {
      for (int s = tid; s < n_segs; s += kBlockThreads) {
        const int rows = segs[s].rows;
        if ((rest_of(rows) >> shift & 0xffff) != 0 && before++ == item) found[0] = s, found[1] = rows / COLS * COLS;
      }
    }
  } else if (item >= wide_before && item < wide_before + wide) {
    for (int s = tid; s < n_segs; s += kBlockThreads) {
      const int n = wide_of(segs[s].rows);
      if (item >= wide_before && item < wide_before + n) found[0] = s, found[1] = (item - wide_before) * COLS;
      wide_before += n;
    }
  }
  __syncthreads();
  const int s = __builtin_amdgcn_readfirstlane(found[0]), c0 = __builtin_amdgcn_readfirstlane(found[1]);
  if (s < 0) return false;
  const DgppMoeSegment seg = segs[s];
  out = {seg.expert, seg.row0 + c0, min(COLS, seg.rows - c0)};
  return true;
}

// COLS: rows of a pass at most, 128, or 32 for short segments (three blocks per CU instead of two).
template <int FMT, bool GU, bool A4, int COLS>
__global__ __launch_bounds__(kBlockThreads, COLS == kNarrowCols ? 3 : 2) void tiled_grouped_kernel(GroupedArgs a, MGeom g, TiledPlan plan) {
  DGPP_TILED_STAGES(st, FMT, A4, COLS);
  TiledItem it;
  int tile, step;
  if (plan.items > 0) {
    const int lin = static_cast<int>(blockIdx.x), idx = lin / kXcds;
    tile = idx % plan.deal.row_tiles;
    step = COLS;
    if (!sorted_item<COLS>(a.segs, plan.n_segs, idx / plan.deal.row_tiles * kXcds + lin % kXcds, it)) return;
  } else {
    const TiledPlace at = tiled_place(plan.deal, static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y));
    if (at.seg < 0) return;
    const DgppMoeSegment seg = a.segs[at.seg];
    tile = at.tile;
    step = at.slots * COLS;
    it = {seg.expert, seg.row0 + at.slot * COLS, seg.rows - at.slot * COLS};
    if (it.rows <= 0) return;
  }
  const int wave = threadIdx.x >> 6;
  TiledRows rows;
  float divisor[2];
  const float* gp[2] = {nullptr, nullptr};
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rows.mat[i] = mat_of_view<FMT>(a.views[it.expert * 3 + (GU ? i : a.which)], &gp[i]);
    rows.row0[i] = GU ? (tile * kWavesPerBlock + wave) * kGroupRows : ((tile * kWavesPerBlock + wave) * 2 + i) * kGroupRows;
    divisor[i] = load_divisor<FMT>(gp[i]);
  }
  A4Src src;
  src.scales = a.a4_scales;
  src.scale_stride = a.a4_scale_stride;
  const TiledOut o = {a.out, a.out_up, a.out_stride, a.out_f32, a.gate_up, a.limit, a.a4_gs};
  for (int c0 = 0; c0 < it.rows; c0 += step) {
    const int first = it.row0 + c0;
    tiled_rows<FMT, GU, A4, COLS>(rows, divisor, a.n, a.k, reinterpret_cast<const uint8_t*>(a.act), A4 ? a.act_stride : a.act_stride * 2,
                                   a.act_rows ? a.act_rows + first : nullptr, first, static_cast<size_t>(first),
                                   min(COLS, it.rows - c0), src, g, o, st);
  }
}

// grid.x = kXcds * ceil(row tiles / kXcds) * column passes.
template <int FMT, bool A4, int COLS>
__global__ __launch_bounds__(kBlockThreads, COLS == kNarrowCols ? 3 : 2) void tiled_dense_kernel(DenseArgs a, MGeom g, int row_tiles, int passes) {
  DGPP_TILED_STAGES(st, FMT, A4, COLS);
  const int lin = static_cast<int>(blockIdx.x), idx = lin / kXcds;
  const int tile = idx / passes * kXcds + lin % kXcds, c0 = idx % passes * COLS;
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
  tiled_rows<FMT, false, A4, COLS>(rows, divisor, a.n, a.k, reinterpret_cast<const uint8_t*>(a.act), A4 ? a.act_stride : a.act_stride * 2,
                                   nullptr, c0, static_cast<size_t>(c0), min(COLS, a.m - c0), src, g, o, st);
}

// A streamed launch's product that the block belongs to; `lin`: the block's number in it.
__device__ __forceinline__ const DenseArgs& stream_problem(const DenseArgs& a, int&) { return a; }
__device__ __forceinline__ const DenseArgs& stream_problem(const DenseMultiArgs& ma, int& lin) {
  int which = 0;
#pragma unroll
  for (int i = 0; i + 1 < kMaxDenseProblems; ++i)
    if (i + 1 < ma.count && lin >= ma.tile_end[i]) which = i + 1;
  if (which != 0) lin -= ma.tile_end[which - 1];
  return ma.p[which];
}

// ---- up to sixteen activation rows ------------------------------------------------------------------------------------
// A dense product of one column tile reads every weight once and is bound by that read, if enough of it is on its way: a
// wavefront takes two row groups and ONE part of K, two to three tiles ahead, and meets nobody until the parts are folded, in
// the order of the forms above. The activation rows, the same few KB for all, come the way of the weights: asked for row by
// row and turned in LDS of the wavefront's own (in the matrix core's order, sixteen rows side by side, their loads took
// longer than the weights'). No barrier in the walk. 32 rows x 4 parts to a block of four wavefronts: a matrix of 17408
// rows has 544 blocks, all resident at once (three to a CU), where the blocks of sixteen wavefronts of the form with
// the parts side by side made just over one round. More rows go in column tiles, the weights out of the XCD's L2.
//
// What bounds it: the walk's latency where a wavefront has few tiles (4096 x 4096: 8 a part, 7.5 us in all), and otherwise the chain of a tile -
// loads, LDS, decoding, products, one behind the other - on CUs with one to three blocks. K = 5120, 8 rows, NVFP4 10.4 us for 256 blocks, 15.6 for 512,
// 18.9 for 544 (17408 rows: three blocks on 32 CUs) and 20.3 for 768; MXFP4 7.8, 11.5, 14.2, 15.5. With one thing left out, 544 blocks, NVFP4
// 18.9 / MXFP4 14.2: the decoding 15.4 / 14.2, the weights' loads 18.3 / 11.5, the rows and their way through LDS 17.7 / 12.6, the weights'
// way through LDS 18.2 / 13.6, the scales 18.7 / 13.8, the products 18.2 / 13.8. Nontemporal loads were slower (23.2 against 21.7, 20.6 against
// 19.3 when that was all): a tile takes half of a line, and the line did not stay for the other half. So two tiles are asked for one right after the
// other: 17408 x 5120, 16 rows, NVFP4 21.2 -> 20.2 us, MXFP4 17.6 -> 16.5, MXFP8 39.3 -> 36.9; 12288 x 4096, 40 rows, MXFP8 35.9 -> 33, block
// FP8 26.1 -> 23.2.
// ROWS: activation rows that are loaded, 8 or 16 (those from m on repeat the last).
// Args: DenseArgs, or DenseMultiArgs: up to four products of one k and one row count in one launch, their blocks one after the other
// (whole rounds of the XCDs each), each output bitwise its single launch's.
template <int FMT, int ROWS, class Args>
__global__ __launch_bounds__(kBlockThreads, 3) void stream_dense_kernel(Args args, MGeom g, int col_tiles) {
  int lin = static_cast<int>(blockIdx.x);
  DenseArgs a = stream_problem(args, lin);
  // An XCD keeps a row tile's column tiles to itself, one after the other.
  const int idx = lin / kXcds;
  const int tile = idx / col_tiles * kXcds + lin % kXcds, c0 = idx % col_tiles * kTileCols;
  a.act += static_cast<size_t>(c0) * a.act_stride;
  a.m = min(a.m - c0, kTileCols);
  using Weights = TiledPass<FMT, false, 2, 2>;
  using Regs = typename Weights::Regs;
  constexpr int kSub = Weights::kSub, kUnits = Weights::kUnits, kActLoads = ROWS * kUnits / kWave;
  static_assert(kActLoads * kWave == ROWS * kUnits && kWave / kUnits * 2 >= 8, "whole loads, whose rows fold alike");
  __shared__ typename Weights::Exchange exchange[kWavesPerBlock];
  __shared__ uint4 act_rows[kWavesPerBlock][2][ROWS * kUnits];   // of two tiles
  __shared__ f32x4_t fold[kWavesPerBlock][2][kWave];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % g.parts;
  const int row0 = (tile * (kWavesPerBlock / g.parts) + wave / g.parts) * 2 * kGroupRows;
  Weights w;
  w.tid = static_cast<int>(threadIdx.x);
  w.set_weights({{a.mat, a.mat}, {row0, row0 + kGroupRows}}, a.n, a.k);
  const int lane = threadIdx.x & (kWave - 1), c = lane & 15, q = lane >> 4;
  const int lo = min(part * g.part_steps, g.steps), hi = min(lo + g.part_steps, g.steps);
  const int full = min(a.k / Weights::kTileElems, hi);
  const uint8_t* act = Weights::uniform(a.act);
  uint32_t act_off[kActLoads];
  int act_k[kActLoads];   // first element of the tile that the lane loads
#pragma unroll
  for (int i = 0; i < kActLoads; ++i) {
    const int row = i * (kWave / kUnits) + lane / kUnits, unit = Weights::unit_at(lane % kUnits, row);
    act_k[i] = unit * 8;
    act_off[i] = static_cast<uint32_t>(min(row, a.m - 1)) * static_cast<uint32_t>(a.act_stride * 2) + unit * 16;
  }
  typename Weights::Exchange& x = exchange[wave];
  struct Acts { uint4 v[kActLoads]; };
  auto load_acts = [&](int tile, Acts& to) {
#pragma unroll
    for (int i = 0; i < kActLoads; ++i) {
      const typename Weights::u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(Weights::buffer(act, tile < full), act_off[i], tile * Weights::kTileElems * 2, 0);
      to.v[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
  };
  auto put_acts = [&](int half, const Acts& from) {
#pragma unroll
    for (int i = 0; i < kActLoads; ++i) act_rows[wave][half][i * kWave + lane] = from.v[i];
  };
  const int act_row = c & (ROWS - 1);
  f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  auto multiply = [&](int tile, int half, const Regs& r) {
    uint4 b[kSub];
#pragma unroll
    for (int j = 0; j < kSub; ++j) b[j] = act_rows[wave][half][act_row * kUnits + Weights::place(q, j, act_row)];
    Frag f[2][kSub];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      ChunkRegs ch;
      ch.w = r.w[i];
      ch.s = w.scale_of(i, tile, r.s[i]);
      decode_frags<FMT>(ch, f[i]);
    }
#pragma unroll
    for (int j = 0; j < kSub; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i] = mfma_bf16(f[i][j], b[j], acc[i]);
  };
  Regs r0, r1, r2, r3;
  Acts b0, b1, b2, b3;
  typename Weights::ScaleWord sraw[2];
  // Two tiles, the halves of a line, are asked for together, once the two before are multiplied: far0 and far1, at even steps.
  auto step = [&](int t, auto at, const Regs& now, Regs& coming, Regs& far0, Regs& far1, const Acts& coming_b, Acts& far_b) {
    constexpr int kAt = decltype(at)::value;
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (kAt % 2 == 0) {
      w.load(t + 2, full, far0);
      w.load(t + 3, full, far1);
    }
    load_acts(t + 3, far_b);
    if constexpr (kAt == 0) w.load_scales(t + 4, sraw);
    multiply(t, kAt & 1, now);
    if constexpr (kAt == 3) w.put_scales(x, sraw);
    w.template exchange<false>(x, (kAt + 1) & 3, coming);
    put_acts((kAt + 1) & 1, coming_b);
  };
  if (lo < full) {
    w.load_scales(lo, sraw);
    w.load(lo, full, r0);
    w.load(lo + 1, full, r1);
    load_acts(lo, b0);
    load_acts(lo + 1, b1);
    load_acts(lo + 2, b2);
    w.put_scales(x, sraw);
    w.template exchange<false>(x, 0, r0);
    put_acts(0, b0);
    int t = lo;
    auto turn = [&](int steps) {   // a constant where this is inlined, or the last turn's
      step(t, std::integral_constant<int, 0>{}, r0, r1, r2, r3, b1, b3);
      if (steps == 1) return;
      step(t + 1, std::integral_constant<int, 1>{}, r1, r2, r2, r3, b2, b0);
      if (steps == 2) return;
      step(t + 2, std::integral_constant<int, 2>{}, r2, r3, r0, r1, b3, b1);
      if (steps == 3) return;
      step(t + 3, std::integral_constant<int, 3>{}, r3, r0, r0, r1, b0, b2);
    };
    for (; t + 4 <= full; t += 4) turn(4);
    if (t < full) turn(full - t);
  }
  if (lo <= full && full < hi) {   // the part of a tile past the last whole one, in the part of K that it belongs to (a part may be empty)
    w.load_rest(full, r0);
#pragma unroll
    for (int i = 0; i < kActLoads; ++i) {
      b0.v[i] = make_uint4(0u, 0u, 0u, 0u);
      if (full * Weights::kTileElems + act_k[i] < a.k)
        b0.v[i] = *reinterpret_cast<const uint4*>(act + act_off[i] + static_cast<size_t>(full) * Weights::kTileElems * 2);
    }
    put_acts(0, b0);
    multiply(full, 0, r0);
  }
  if (g.parts > 1) {
#pragma unroll
    for (int i = 0; i < 2; ++i) fold[wave][i][lane] = acc[i];
    __syncthreads();
    if (part != 0) return;
  }
  const float divisor = load_divisor<FMT>(a.global);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    f32x4_t s = acc[i];
    if (g.parts >= 2) s = s + fold[wave + 1][i][lane];
    if (g.parts == 4) s = (s + fold[wave + 2][i][lane]) + fold[wave + 3][i][lane];
    store_tile<FMT>(s, divisor, a.out, a.out_f32, static_cast<size_t>(c0 + c) * a.out_stride, row0 + i * kGroupRows, a.n, c < a.m);
  }
}

}  // namespace dgpp_amd
