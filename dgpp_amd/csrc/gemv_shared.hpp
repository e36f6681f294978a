// A small decode batch's routed experts and its block-FP8 shared expert in one launch per pass: the blocks of either are those of
// the launches that they would have (gemv_kernels.hpp), bit for bit, and run beside each other where they ran one after the other.
//
// What bounds these passes is a launch's start and end: NVFP4, 288 experts of 512 x 4096 and a shared one of 512, 3 tokens, us: gate + up
// 16.4 routed and 6.2 shared, down 11.6 and 5.4, accumulation 3.2; a layer 52.8 -> 38.7 so, one token 31 -> 22.
#pragma once

#include "gemv_kernels.hpp"

namespace dgpp_amd {

// The shared expert's part of a grid, whose blocks come first: they wait for nothing, and its rows are twice as long.
struct SharedPart {
  SlotArgs a;
  RowGeom g;
  int steps;
  int tiles;    // of a run of `run` tokens
  int blocks;
  int run;
};

// SELECT: one token, whose selection every routed block repeats.
template <int FMT, int NB, int RUN, bool SPLIT, bool NT, bool SELECT>
__global__ __launch_bounds__(kBlockThreads, kMinWavesPerSimd) void gate_up_shared_kernel(SlotArgs a, SelectArgs sel, RowGeom g, int steps,
                                                                                        int tiles, SharedPart s) {
  extern __shared__ uint4 lds[];
  int b = static_cast<int>(blockIdx.x);
  if (b < s.blocks) {
    const int p = b / s.tiles * s.run * (s.a.top_k + 1) + s.a.top_k;   // the shared slot of a run's first token
    slot_gate_up_body<kFmtFp8F32, NB, RUN, SPLIT, false>(s.a, s.g, s.steps, lds, p, b % s.tiles);
    return;
  }
  b -= s.blocks;
  if constexpr (SELECT) {
    int32_t* ids = reinterpret_cast<int32_t*>(lds + FmtTraits<FMT>::kPieces * (a.k / FmtTraits<FMT>::kElemsPerChunk));
    if (threadIdx.x < kWave) select_to_lds(sel, a.top_k, ids, b == 0);
    __syncthreads();
    a.ids = ids;
  }
  slot_gate_up_body<FMT, NB, RUN, SPLIT, NT>(a, g, steps, lds, b / tiles, b % tiles);
}

// token_down_accum_kernel with the shared slot's row at the end of the chain: wavefronts from top_k on take a part of the tile's rows
// of the shared matrix each (SHARED of them: a block-FP8 row is as long as two of FP4).
struct SharedDown {
  MatRef mat;
  RowGeom g;
  int k;
};
// NB, NBS: loads in flight of a routed and of a shared row (the chain per row does not depend on them).
template <int FMT, int NB, int NBS, bool SPLIT, int SHARED>
__global__ __launch_bounds__(1024) void token_down_shared_kernel(TokenDownArgs a, RowGeom g, int steps, SharedDown s) {
  extern __shared__ uint4 lds[];
  constexpr int kPieces = FmtTraits<FMT>::kPieces, kSharedPieces = FmtTraits<kFmtFp8F32>::kPieces;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  int t, tile;
  token_tile(a, static_cast<int>(blockIdx.x), t, tile);
  const int rows_per_block = (kWave >> g.l2) * steps, tile_row0 = tile * rows_per_block;
  const int row_vecs = kPieces * (a.k / FmtTraits<FMT>::kElemsPerChunk);
  const int shared_vecs = kSharedPieces * (s.k / FmtTraits<kFmtFp8F32>::kElemsPerChunk);
  float* part = reinterpret_cast<float*>(lds + a.top_k * row_vecs + SHARED * shared_vecs);   // [top_k + 1][rows_per_block]
  const uint16_t* x = a.act + (static_cast<size_t>(t) * (a.top_k + 1) + min(wave, a.top_k)) * a.act_stride;
  // One slot's rows of the tile from row `first` on, `count` of them, to dots[0 ...].
  auto walk = [&](auto fmt, auto loads, auto nt, const MatRef& m, const float* global, const RowGeom& rg, int k, uint4* my_x, int first,
                  int count, float* dots) {
    constexpr int F = decltype(fmt)::value, N = decltype(loads)::value, XV = kSplitStageVecs;
    constexpr bool kNT = decltype(nt)::value;
    const int chunks = k / FmtTraits<F>::kElemsPerChunk, vecs = FmtTraits<F>::kPieces * chunks, rpw = kWave >> rg.l2;
    auto lr = lane_row<F, kNT>(m, first, a.n, k, rg.l2);
    ChunkRegs regs[N];
    if constexpr (SPLIT) {
      StageRegs<XV> xr;
      stage_issue<F, XV>(x, k, lane, kWave, xr);
      issue_pass<F, N>(lr, 0, rg.l2, m.cs, regs);
      stage_commit<F, XV>(xr, k, lane, kWave, my_x);
    } else {
      const bool aligned = (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
      for (int v = lane; v < vecs; v += kWave) {
        const int c = v / FmtTraits<F>::kPieces, q = v - c * FmtTraits<F>::kPieces;
        my_x[q * chunks + c] = load_vec8(x, v, aligned);
      }
    }
    // The staged row is this wavefront's own: LDS keeps a wavefront's writes and reads in order, no block barrier.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float d = load_divisor<F>(global);
    for (int r = 0; r < count && first + r < a.n; r += rpw) {
      float acc[1];
      if (SPLIT && r == 0) {
        row_dots_pre<F, 1, N>(lr, rg, m.cs, my_x, chunks, 1, regs, acc);
      } else {
        lr = lane_row<F, kNT>(m, first + r, a.n, k, rg.l2);
        row_dots<F, 1, N>(lr, rg, m.cs, my_x, chunks, 1, acc);
      }
      if (lr.li == 0) dots[r + (lane >> rg.l2)] = finish_dot<F>(acc[0], d);
    }
  };
  if (wave < a.top_k) {
    const float* gd = nullptr;
    const MatRef md = mat_of_view<FMT>(a.views[a.ids[static_cast<size_t>(t) * a.top_k + wave] * 3 + 2], &gd);
    walk(std::integral_constant<int, FMT>{}, std::integral_constant<int, NB>{}, std::true_type{}, md, gd, g, a.k, lds + wave * row_vecs, tile_row0, rows_per_block, part + wave * rows_per_block);
  } else {
    const int i = wave - a.top_k, count = rows_per_block / SHARED;
    walk(std::integral_constant<int, kFmtFp8F32>{}, std::integral_constant<int, NBS>{}, std::false_type{}, s.mat, nullptr, s.g, s.k,
         lds + a.top_k * row_vecs + i * shared_vecs, tile_row0 + i * count, count, part + a.top_k * rows_per_block + i * count);
  }
  __syncthreads();
  for (int r = threadIdx.x; r < rows_per_block; r += blockDim.x) {
    const int row = tile_row0 + r;
    if (row >= a.n) break;
    float v = 0.f;
    for (int j = 0; j < a.top_k; ++j)
      v = fmaf(a.weights[static_cast<size_t>(t) * a.top_k + j], part[j * rows_per_block + r], v);
    v = fmaf(1.0f, part[a.top_k * rows_per_block + r], v);
    static_cast<uint16_t*>(a.out)[static_cast<size_t>(t) * a.n + row] = f32_to_bf16(v);
  }
}

// ask: only whether the call is of this form. One token comes with its selection (the fast set-up) or past 4096 of k without.
template <int FMT>
bool launch_gate_up_shared_fmt(const SlotArgs& a, const SlotArgs& sh, const SelectArgs* sel, bool ask, hipStream_t stream, hipError_t& err) {
  const RowGeom g = geom_for<FMT>(a.k);
  SharedPart s;
  s.g = geom_for<kFmtFp8F32>(sh.k);
  if (s.g.P % g.nb != 0 || use_mfma_core()) return false;   // one number of loads in flight for both
  const bool split = tune_get(kTuneSplitStage) != 1 && a.k <= 8 * kSplitStageVecs * kBlockThreads && (a.x_stride & 7u) == 0 && (reinterpret_cast<uintptr_t>(a.x) & 15u) == 0;
  const int tokens = a.slots / (a.top_k + 1);
  if (tokens == 1 ? (sel != nullptr) != split : sel != nullptr || !a.match || !a.once || run_cap_for(a, kGateUpRun) != kGateUpRun) return false;
  if (ask) return true;
  const int rows_per_step = kWavesPerBlock * (kWave >> g.l2), shared_step = kWavesPerBlock * (kWave >> s.g.l2);
  const int per_slot = (a.n + rows_per_step - 1) / rows_per_step;
  const int steps = tokens > 1 ? 2 : pick_steps(static_cast<long long>(per_slot) * a.slots);   // as launch_slot_gate_up_fmt
  const int tiles = (per_slot + steps - 1) / steps;
  s.a = sh;
  s.steps = 1;
  s.tiles = (sh.n + shared_step - 1) / shared_step;
  s.run = tokens > 1 ? kGateUpRun : 1;
  s.blocks = s.tiles * ((tokens + s.run - 1) / s.run);
  const dim3 grid(static_cast<unsigned>(s.blocks) + static_cast<unsigned>(tiles) * static_cast<unsigned>(a.slots));
  const size_t lds = stage_bytes(s.run, a.k) + (sel != nullptr ? kWave * sizeof(int32_t) : 0);
  err = hipSuccess;
  dispatch_nb(g.nb, [&](auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    auto go = [&](auto kern) {
      err = ensure_lds(kern, lds);
      if (err == hipSuccess) hipLaunchKernelGGL(kern, grid, dim3(kBlockThreads), lds, stream, a, sel != nullptr ? *sel : SelectArgs{}, g, steps, tiles, s);
    };
    if (sel != nullptr) go(gate_up_shared_kernel<FMT, NB, 1, true, true, true>);
    else if (split) go(gate_up_shared_kernel<FMT, NB, kGateUpRun, true, true, false>);
    else go(gate_up_shared_kernel<FMT, NB, kGateUpRun, false, false, false>);
  });
  if (err == hipSuccess) err = hipGetLastError();
  note_launch(kFormShared);
  return true;
}

template <int FMT>
bool launch_token_down_shared_fmt(const TokenDownArgs& a, const MatRef& shared, int k_shared, bool ask, hipStream_t stream, hipError_t& err) {
  constexpr int SHARED = FMT == kFmtFp8F32 ? 1 : 2;
  const RowGeom g = geom_for<FMT>(a.k);
  SharedDown s;
  s.mat = shared;
  s.k = k_shared;
  s.g = geom_for<kFmtFp8F32>(k_shared);
  if (s.g.P % g.nb != 0 || use_mfma_core()) return false;
  if ((a.top_k + SHARED) * kWave > 1024) return false;
  const int rpw = kWave >> g.l2, shared_rpw = kWave >> s.g.l2;
  const long long wave_steps = static_cast<long long>((a.n + rpw - 1) / rpw) * a.tokens * a.top_k;
  int steps = static_cast<int>(wave_steps / 16384);   // as launch_token_down_fmt
  steps = steps < 2 ? 2 : (steps > 8 ? 8 : steps);
  const int rows_per_block = rpw * steps;
  if (rows_per_block % (SHARED * shared_rpw) != 0) return false;
  TokenDownArgs b = a;
  b.tiles = (a.n + rows_per_block - 1) / rows_per_block;
  b.xcd_group = a.tokens > 1 && a.tokens * a.top_k * 4 >= 256 && b.tiles % 8 == 0 ? 1 : 0;
  if (static_cast<long long>(b.tiles) * a.tokens > 0x7FFFFFFFLL) return false;
  const size_t lds = static_cast<size_t>(a.top_k) * stage_bytes(1, a.k) + SHARED * stage_bytes(1, k_shared) +
                     static_cast<size_t>(a.top_k + 1) * rows_per_block * sizeof(float);
  if (lds > kMaxLdsBytes) return false;
  if (ask) return true;
  const bool split = tune_get(kTuneSplitStage) != 1 && a.k <= 8 * kSplitStageVecs * kWave && k_shared <= 8 * kSplitStageVecs * kWave && (a.act_stride & 7u) == 0 &&
                     (reinterpret_cast<uintptr_t>(a.act) & 15u) == 0;
  const dim3 grid(static_cast<unsigned>(b.tiles) * static_cast<unsigned>(a.tokens));
  err = hipSuccess;
  dispatch_nb(g.nb, [&](auto nbc) {
    constexpr int NB = decltype(nbc)::value;
    auto go = [&](auto kern) {
      err = ensure_lds(kern, lds);
      if (err == hipSuccess) hipLaunchKernelGGL(kern, grid, dim3((a.top_k + SHARED) * kWave), lds, stream, b, g, steps, s);
    };
    auto go_loads = [&](auto loads) {
      constexpr int NBS = decltype(loads)::value;
      if (split) go(token_down_shared_kernel<FMT, NB, NBS, true, SHARED>);
      else go(token_down_shared_kernel<FMT, NB, NBS, false, SHARED>);
    };
    if constexpr (FMT != kFmtFp8F32 && NB <= 4) {
      if (s.g.P % (2 * NB) == 0) return go_loads(std::integral_constant<int, 2 * NB>{});
    }
    go_loads(std::integral_constant<int, NB>{});
  });
  if (err == hipSuccess) err = hipGetLastError();
  note_launch(kFormShared);
  return true;
}

}  // namespace dgpp_amd
