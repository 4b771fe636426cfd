// Rows of an input product of one token: norm prologue, dot products, activation epilogue, as a body that
// a launch of its own (mixer_gemv.hip) and the one beside a mixer (mixer_beside.hip) run.
#pragma once
#include "gemv_kernel.h"
#include "mixer_common.h"

namespace cake {

struct MixInArgs {
  const float* resid;
  const uint16_t* norm_w;
  const uint16_t* w;       // [N][K]
  float* out;
  const uint16_t* bias;    // the up rows'; may be null
  uint16_t* act;
  float eps, off;
  int ln, Kn, K, N, n_raw, actf;
};

__host__ __device__ __forceinline__ int mixer_in_pairs(const MixInArgs& a) { return (a.N + 1) >> 1; }

// lanes 0 and 1 of a wave store a pair's rows
template <int DT>
__device__ __forceinline__ void mixer_in_store(const MixInArgs& a, int p, float da, float db, int lane) {
  const int r = 2 * p + lane;
  if (lane > 1 || r >= a.N) return;
  const float d = lane == 0 ? da : db;
  if (r < a.n_raw) a.out[r] = d;
  else a.act[r - a.n_raw] = from_f32<DT>(mix_act(a.actf, a.bias ? d + to_f32<DT>(a.bias[r - a.n_raw]) : d));
}

// rows [0, n_raw) -> out f32; rows [n_raw, N) -> act = actf(. + bias) in 16 bit.  ln: a layer
// norm instead of the RMS norm.  Workgroup blk of nblk, NT threads, xs [K] f32.
template <int DT, int U, int PFC, int NX, int NT>
__device__ __forceinline__ void mixer_in_rows(const MixInArgs& a, int blk, int nblk, float* xs) {
  constexpr int kWaves = NT / 64;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int npairs = mixer_in_pairs(a);
  const int p0 = blk * kWaves + wave;
  auto map = [&](int p, const uint16_t*& wa, const uint16_t*& wb) {
    wa = a.w + (size_t)(2 * p) * a.K;
    wb = a.w + (size_t)min(2 * p + 1, a.N - 1) * a.K;
  };
  Regs<PFC> pre;
  NormPre<DT, NX, NT> xp;
  const uint16_t *wa0, *wb0;
  map(p0 < npairs ? p0 : npairs - 1, wa0, wb0);
  if constexpr (NX > 0) xp.load(a.resid, a.norm_w, a.K);
  __builtin_amdgcn_sched_barrier(0);  // x loads strictly before the weights (in-order vmcnt)
  if (NX > 0 || (PFC > 0 && p0 < npairs)) prefetch_rows<PFC>(wa0, wb0, pre);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NX > 0) xp.finish_off(a.eps, a.K, a.Kn, a.off, a.ln, xs);
  else stage_norm_off<DT>(a.resid, a.norm_w, a.eps, a.K, a.Kn, a.off, a.ln, xs);
  auto epi = [&](int p, float da, float db) { mixer_in_store<DT>(a, p, da, db, lane); };
  // (of rounds of two there is one left over at most: asked for at once 2048 rows of 2560 took 5.1 us, 4.8)
  run_pairs<DT, true, U, PFC, (U > 2)>(map, epi, xs, a.K, npairs, p0, nblk * kWaves, pre);
}

}  // namespace cake
