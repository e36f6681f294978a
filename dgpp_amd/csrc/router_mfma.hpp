// The router's score rows of a prompt chunk on the matrix core. Included by moe_router.hip after store_score.
//
// A (token, expert) dot is 64 chains of fmas and a tree over them (router_dots_tile_kernel): chain l takes the eight-element
// vectors l, l + 64, ... in element order. v_mfma_f32_16x16x4_f32 is four fmas in ascending order, each rounded to FP32, subnormal
// numbers kept (checked bit for bit against the host's fmaf over random and subnormal operands), so a chain is a row of those
// instructions, and the sums are the other form's, bit for bit.
//
// A block is a tile of TT tokens and 32 experts, eight wavefronts. Wavefront j runs the chains l = 8 h + j, h in
// bit-reversed order, so that the tree's first three levels (l ^ 32, 16, 8) need three sums in registers; the last three are the
// eight wavefronts', over LDS. An item is four vectors a chain of the eight chains of one h: four 128-byte lines of every row, loaded
// to a ring of LDS stages. Tiles of 32 tokens have two stages and two blocks per CU, which cover each other's barriers; tiles of 16,
// for batches that leave CUs without one of 32, have four stages, three items on their way. (Tiles of 32 hold 128 registers and 12 bytes
// of scratch a lane, at four wavefronts per SIMD.)
//
// Lanes. The instruction wants one element of a row from each of four lanes: a lane reads the words that hold its two elements
// of a vector and places the halves by v_perm. (Whole vectors and swaps between lanes took twice the vector instructions, which
// run on the units of this one: 133 us for the 107 below.)
//
// What bounds it: the FP32 matrix instruction, 120 TFLOP/s measured alone: 4096 tokens, 256 experts x 4096 99 TFLOP/s. From the sums in
// lanes, us: 4096 tokens, 288 x 4096 181 -> 107 (five rounds of blocks, the last half empty), 256 x 4096 161 -> 87; 2048 tokens 83 -> 46;
// 512 tokens, 256 x 6144 35 -> 26.
#pragma once

namespace dgpp_amd {
namespace {

constexpr int kChainWaves = 8, kChainExperts = 32, kChainSteps = 4;
constexpr int kChainThreads = kChainWaves * 64;
constexpr int chain_stage_units(int tokens) { return (tokens + kChainExperts) * kChainSteps * 8; }   // 16-byte units

// All but the newest N loads of this wavefront have arrived and its LDS reads are done, then the block's barrier.
template <int N>
__device__ __forceinline__ void chain_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}

template <int TT, int RING>
struct RouterChains {
  static constexpr int kE = kChainExperts / 16, kT = TT / 16;          // 16-row groups
  static constexpr int kRows = TT + kChainExperts;
  static constexpr int kLoads = kRows * kChainSteps * 8 / kChainThreads;   // a thread's per item: 16 rows each
  static_assert(RING == 2 || RING == 4, "stages are named in turns of two or four");
  typedef float f32x4_t __attribute__((ext_vector_type(4)));
  using Acc = f32x4_t[kE][kT];

  const uint8_t* gate;
  const uint8_t* hidden;
  uint32_t gate_bytes, hidden_bytes, row_bytes;
  uint32_t first_byte;     // this thread's, of its row of the first sixteen
  int tid, wave, lines, items;   // lines: 128-byte ones of a row; items: of one h

  __device__ __forceinline__ static int reversed(int h) { return ((h & 1) << 2) | (h & 2) | ((h >> 2) & 1); }

  // Item `at` of the h-th group: past a row's end the next row's bytes or zeros come, which nobody multiplies; past the tile's
  // rows zeros; past the last item nothing is read (the waits count the loads all the same). Place ((row x 4 + step) x 8 + piece)
  // of a stage, the step and the piece turned by the row: sixteen rows that are read together meet no bank twice.
  __device__ __forceinline__ void fetch(int h, int at, uint4* __restrict__ stage) const {
    const bool live = h < 8;
    const uint32_t off = first_byte + (static_cast<uint32_t>(at) * 4096u + static_cast<uint32_t>(reversed(h)) * 128u);
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
      const uint32_t rows = (i < kE ? i : i - kE) * 16u, bytes = i < kE ? gate_bytes : hidden_bytes, skip = rows * row_bytes;
      const __amdgpu_buffer_rsrc_t b = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>((i < kE ? gate : hidden) + skip), 0,
                                                                         live && bytes > skip ? bytes - skip : 0u, 0x00027000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(b, (__attribute__((address_space(3))) void*)(stage + (i * kChainWaves + wave) * 64), 16, off, 0, 0, 0);
    }
  }
  __device__ __forceinline__ void set_thread() {
    tid = static_cast<int>(threadIdx.x);
    wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const uint32_t row = static_cast<uint32_t>(wave * 2 + (lane >> 5));
    const uint32_t step = (static_cast<uint32_t>(lane >> 3) ^ (row >> 3)) & 3u, piece = (static_cast<uint32_t>(lane) ^ row) & 7u;
    first_byte = row * row_bytes + step * 1024u + piece * 16u;
  }

  // Lane (r, q) multiplies elements q and q + 4 of a vector: half of word q / 2, and of the second next.
  __device__ __forceinline__ void multiply(const uint4* __restrict__ stage, int left, Acc& acc) const {
    const int lane = tid & 63, r = lane & 15, q = lane >> 4;
    const uint32_t* at[2];   // of even and of odd steps
#pragma unroll
    for (int i = 0; i < 2; ++i)
      at[i] = reinterpret_cast<const uint32_t*>(stage + (r * 4 + (i ^ (r >> 3))) * 8 + (wave ^ (r & 7))) + (q >> 1);
    const uint32_t half = (q & 1) != 0 ? 0x07060c0cu : 0x05040c0cu;   // the BF16 number's place, zeros below
    uint32_t v[kE + kT][kChainSteps][2];
#pragma unroll
    for (int s = 0; s < kChainSteps; ++s)
#pragma unroll
      for (int g = 0; g < kE + kT; ++g)
#pragma unroll
        for (int i = 0; i < 2; ++i) v[g][s][i] = at[s & 1][g * 16 * 128 + (s >> 1) * 64 + i * 2];
    auto step = [&](int s) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        float f[kE + kT];
#pragma unroll
        for (int g = 0; g < kE + kT; ++g) f[g] = bits_f32(__builtin_amdgcn_perm(v[g][s][i], 0u, half));
#pragma unroll
        for (int g = 0; g < kE; ++g)
#pragma unroll
          for (int t = 0; t < kT; ++t) acc[g][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[g], f[kE + t], acc[g][t], 0, 0, 0);
      }
    };
    if (left >= kChainSteps) {
#pragma unroll
      for (int s = 0; s < kChainSteps; ++s) step(s);
    } else {
#pragma unroll
      for (int s = 0; s < kChainSteps - 1; ++s)
        if (s < left) step(s);
    }
  }
  __device__ __forceinline__ static void add(const Acc& a, Acc& to) {
#pragma unroll
    for (int g = 0; g < kE; ++g)
#pragma unroll
      for (int t = 0; t < kT; ++t) to[g][t] = a[g][t] + to[g][t];
  }
  __device__ __forceinline__ static void move(const Acc& a, Acc& to) {
#pragma unroll
    for (int g = 0; g < kE; ++g)
#pragma unroll
      for (int t = 0; t < kT; ++t) to[g][t] = a[g][t];
  }

  // `sum`: this wavefront's chains, three levels of the tree done: expert group g, token group t; lane (token c, q) register i is
  // expert 4 q + i. Every thread of the block must call.
  __device__ __forceinline__ void run(uint4* __restrict__ s0, uint4* __restrict__ s1, uint4* __restrict__ s2, uint4* __restrict__ s3,
                                      Acc& sum) {
    int fh = 0, fi = 0;   // the item that is fetched next
    auto fetch_next = [&](uint4* __restrict__ stage) {
      fetch(fh, fi, stage);
      if (++fi == items) fi = 0, ++fh;
    };
    fetch_next(s0);
    if constexpr (RING == 4) {
      fetch_next(s1);
      fetch_next(s2);
    }
    Acc acc, level1, level2;
#pragma unroll
    for (int g = 0; g < kE; ++g)
#pragma unroll
      for (int t = 0; t < kT; ++t) acc[g][t] = level1[g][t] = level2[g][t] = sum[g][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    int h = 0, i = 0;
    auto item = [&](const uint4* __restrict__ mine, uint4* __restrict__ free_stage) {
      chain_barrier<(RING - 2) * kLoads>();   // this item is whole, and nobody reads the one before any more
      fetch_next(free_stage);
      multiply(mine, (lines - reversed(h) + 7) / 8 - i * kChainSteps, acc);
      if (++i == items) {
        if ((h & 1) == 0) {
          move(acc, level1);
        } else {
          add(level1, acc);
          if ((h & 2) == 0) {
            move(acc, level2);
          } else {
            add(level2, acc);
            add(acc, sum);   // the first half is added to zeros
          }
        }
#pragma unroll
        for (int g = 0; g < kE; ++g)
#pragma unroll
          for (int t = 0; t < kT; ++t) acc[g][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        i = 0, ++h;
      }
    };
    for (int t = 0; t < 8 / RING * items; ++t) {
      if constexpr (RING == 2) {
        item(s0, s1);
        item(s1, s0);
      } else {
        item(s0, s3);
        item(s1, s0);
        item(s2, s1);
        item(s3, s2);
      }
    }
    chain_barrier<0>();
  }
};

template <int kMode, int TT>
__device__ __forceinline__ void router_chain_tile(const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ gate,
                                                  const float* __restrict__ bias, float* __restrict__ scores, float* __restrict__ biased,
                                                  int tokens, int hidden_dim, int n_experts, int t0, int e0) {
  constexpr int kRing = TT == 32 ? 2 : 4;
  using R = RouterChains<TT, kRing>;
  constexpr int kPitch = kChainExperts + 4;   // floats of a token's sums in LDS
  static_assert(kChainWaves * TT * kPitch * 4 <= chain_stage_units(TT) * kRing * 16, "the sums fit where the stages were");
  __shared__ uint4 stage[kRing][chain_stage_units(TT)];
  R r;
  r.row_bytes = static_cast<uint32_t>(hidden_dim) * 2u;
  r.set_thread();
  r.lines = hidden_dim / 64;
  r.items = (hidden_dim / 64 + 31) / 32;
  r.gate = reinterpret_cast<const uint8_t*>(gate + static_cast<size_t>(e0) * hidden_dim);
  r.hidden = reinterpret_cast<const uint8_t*>(hidden + static_cast<size_t>(t0) * hidden_dim);
  r.gate_bytes = static_cast<uint32_t>(min(n_experts - e0, kChainExperts)) * r.row_bytes;
  r.hidden_bytes = static_cast<uint32_t>(min(tokens - t0, TT)) * r.row_bytes;
  typename R::Acc sum;
  r.run(stage[0], stage[1], stage[kRing - 2], stage[kRing - 1], sum);
  float* sums = reinterpret_cast<float*>(&stage[0][0]);
  const int lane = r.tid & 63;
#pragma unroll
  for (int g = 0; g < R::kE; ++g)
#pragma unroll
    for (int t = 0; t < R::kT; ++t)
      *reinterpret_cast<typename R::f32x4_t*>(sums + (r.wave * TT + t * 16 + (lane & 15)) * kPitch + g * 16 + (lane >> 4) * 4) = sum[g][t];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TT * kChainExperts / kChainThreads; ++i) {
    const int at = r.tid + i * kChainThreads, t = at / kChainExperts, e = at % kChainExperts;
    float v[kChainWaves];
#pragma unroll
    for (int j = 0; j < kChainWaves; ++j) v[j] = sums[(j * TT + t) * kPitch + e];
    const float dot = ((v[0] + v[4]) + (v[2] + v[6])) + ((v[1] + v[5]) + (v[3] + v[7]));
    if (t0 + t < tokens && e0 + e < n_experts)
      store_score<kMode>(dot, bias, e0 + e, static_cast<size_t>(t0 + t) * n_experts + e0 + e, scores, biased);
  }
}

// The expert tiles of a token tile follow each other on one XCD, whose L2 then holds the tokens' rows (and all of the gate).
template <int kMode, int TT>
__global__ __launch_bounds__(kChainThreads, TT == 32 ? 4 : 2) void router_dots_chain_kernel(
    const uint16_t* __restrict__ hidden, const uint16_t* __restrict__ gate, const float* __restrict__ bias, float* __restrict__ scores,
    float* __restrict__ biased, int tokens, int hidden_dim, int n_experts) {
  const int expert_tiles = (n_experts + kChainExperts - 1) / kChainExperts;
  const int within = static_cast<int>(blockIdx.x >> 3);
  const int t0 = ((within / expert_tiles) * 8 + static_cast<int>(blockIdx.x & 7)) * TT;
  if (t0 >= tokens) return;
  router_chain_tile<kMode, TT>(hidden, gate, bias, scores, biased, tokens, hidden_dim, n_experts, t0, within % expert_tiles * kChainExperts);
}

template <int TT>
void launch_dots_chain(int mode, hipStream_t stream, const uint16_t* hidden, const uint16_t* gate, const float* bias, float* scores,
                       float* biased, int tokens, int hidden_dim, int n_experts) {
  const int token_tiles = (tokens + TT - 1) / TT, expert_tiles = (n_experts + kChainExperts - 1) / kChainExperts;
  const dim3 grid((token_tiles + 7) / 8 * 8 * expert_tiles), block(kChainThreads);
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, block, 0, stream, hidden, gate, bias, scores, biased, tokens, hidden_dim, n_experts);
  };
  if (mode == DGPP_ROUTER_SOFTMAX_TOPK) go(router_dots_chain_kernel<DGPP_ROUTER_SOFTMAX_TOPK, TT>);
  else if (mode == DGPP_ROUTER_SQRT_SOFTPLUS_BIAS) go(router_dots_chain_kernel<DGPP_ROUTER_SQRT_SOFTPLUS_BIAS, TT>);
  else go(router_dots_chain_kernel<DGPP_ROUTER_SIGMOID_BIAS, TT>);
}

}  // namespace
}  // namespace dgpp_amd
