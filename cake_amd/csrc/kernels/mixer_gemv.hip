// Batch-1 decode projections of the hybrid designs (16-bit weights).
//
// In a parallel layer one norm feeds every projection, so its input side is ONE launch over the
// concatenated rows [mixer projections | feed-forward up] (the norm is the prologue, the
// feed-forward activation the epilogue of the up rows) and its output side ONE launch over
// the concatenated columns [mixer output | feed-forward down] with the residual sum in the
// epilogue; between them runs the mixer (mixer_attn.hip, mixer_delta.hip; with the up rows beside it where
// mixer_beside.hip takes them, the first launch is the mixer's rows then).  A serial layer runs
// the same two kernels around its mixer and again around its feed-forward.
#include "mixer_gemv.h"

namespace cake {

template <int DT, int U, int PFC, int NX>
__global__ __launch_bounds__(kGemvThreads) void mixer_in_kernel(MixInArgs a) {
  extern __shared__ float xs[];
  mixer_in_rows<DT, U, PFC, NX, kGemvThreads>(a, blockIdx.x, gridDim.x, xs);
}

// Up to a workgroup a CU: a wave has one pair, and all R rounds of 512 columns of it are asked for before the norm.  Rounds
// behind it are round trips of their own, and with one workgroup on a CU nothing hides them.  A few more pairs than four
// waves a CU take: five, so that no CU has two workgroups.  2048 rows of 1536 / 2560 / 3584 / 4096 columns, two or four rounds
// before the norm, 3.9 / 4.8 / 5.9 / 6.7 us, 3.7 / 4.6 / 5.5 / 6.1 so; 2560 rows 4.3 / 5.6 / 6.6 / 7.1, 4.0 / 5.0 / 6.0 / 6.4; 3072
// of 4096 on five waves 8.4, on four with the whole pair asked for 7.6, as mixer_in_kernel has them 7.4.
template <int DT, int R, int NT>
__global__ __launch_bounds__(NT) void mixer_in_pair_kernel(MixInArgs a) {
  extern __shared__ float xs[];
  constexpr int NX = (R * 512 + 4 * NT - 1) / (4 * NT);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nch = a.K >> 3, npairs = mixer_in_pairs(a);
  const int p = blockIdx.x * (NT / 64) + wave, at = min(p, npairs - 1);
  const uint4* wa = reinterpret_cast<const uint4*>(a.w + (size_t)(2 * at) * a.K);
  const uint4* wb = reinterpret_cast<const uint4*>(a.w + (size_t)min(2 * at + 1, a.N - 1) * a.K);
  NormPre<DT, NX, NT> xp;
  xp.load(a.resid, a.norm_w, a.K);
  __builtin_amdgcn_sched_barrier(0);
  uint4 va[R], vb[R];
#pragma unroll
  for (int c = 0; c < R; ++c) {
    const int i = c + 1 < R ? c * 64 + lane : min(c * 64 + lane, nch - 1);
    va[c] = ld_nt16(wa + i);
    vb[c] = ld_nt16(wb + i);
  }
  __builtin_amdgcn_sched_barrier(0);
  xp.finish_off(a.eps, a.K, a.Kn, a.off, a.ln, xs);
  float da = 0.f, db = 0.f;
#pragma unroll
  for (int c = 0; c < R; ++c)
    if (c + 1 < R || c * 64 + lane < nch) fma_chunk<DT, true>(xs, c * 64 + lane, va[c], vb[c], da, db);
  da = wave_sum(da);
  db = wave_sum(db);
  if (p < npairs) mixer_in_store<DT>(a, p, da, db, lane);
}

// Few rows (a router's): a workgroup has one pair of them, each of its waves a quarter of k.  With a pair a wave, the
// workgroups are as few as the rows are, and one CU reads 64 KB at 25 KB a us (64 / 512 / 1024 rows of 4096 4.9 / 5.4 /
// 5.6 us, 3.2 / 4.0 / 4.5 so; 2048 6.6, 6.4; of 2048 columns 64 / 1024 3.5 / 3.9, 2.7 / 3.6, 4096 5.6, 6.2).
template <int DT, int PFC, int NX>
__global__ __launch_bounds__(kGemvThreads) void mixer_in_split_kernel(MixInArgs a) {
  extern __shared__ float xs[];
  __shared__ float part[2][kGemvWaves];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nch = a.K >> 3;
  const uint4* wa = reinterpret_cast<const uint4*>(a.w + (size_t)(2 * blockIdx.x) * a.K);
  const uint4* wb = reinterpret_cast<const uint4*>(a.w + (size_t)min(2 * (int)blockIdx.x + 1, a.N - 1) * a.K);
  NormPre<DT, NX> xp;
  xp.load(a.resid, a.norm_w, a.K);
  __builtin_amdgcn_sched_barrier(0);
  uint4 va[PFC], vb[PFC];
#pragma unroll
  for (int c = 0; c < PFC; ++c) {
    const int i = min((c * kGemvWaves + wave) * 64 + lane, nch - 1);
    va[c] = wa[i];
    vb[c] = wb[i];
  }
  __builtin_amdgcn_sched_barrier(0);
  xp.finish_off(a.eps, a.K, a.Kn, a.off, a.ln, xs);
  float da = 0.f, db = 0.f;
#pragma unroll
  for (int c = 0; c < PFC; ++c) {
    const int i = (c * kGemvWaves + wave) * 64 + lane;
    if (i < nch) fma_chunk<DT, true>(xs, i, va[c], vb[c], da, db);
  }
  da = wave_sum(da);
  db = wave_sum(db);
  if (lane == 0) {
    part[0][wave] = da;
    part[1][wave] = db;
  }
  __syncthreads();
  const float *qa = part[0], *qb = part[1];
  mixer_in_store<DT>(a, blockIdx.x, (qa[0] + qa[1]) + (qa[2] + qa[3]), (qb[0] + qb[1]) + (qb[2] + qb[3]), threadIdx.x);
}

// y[r] = x[r] + alpha ((W a)[r] + bias[r]), a 16-bit; bias may be null
template <int DT, int U, int PFC, int NX>
__global__ __launch_bounds__(kGemvThreads) void mixer_out_kernel(
    const uint16_t* __restrict__ a, const uint16_t* __restrict__ w, int K, int N, float alpha,
    const uint16_t* __restrict__ bias, const float* x, float* y) {
  extern __shared__ float smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int npairs = (N + 1) >> 1;
  const int p0 = blockIdx.x * kGemvWaves + wave;
  auto map = [&](int p, const uint16_t*& wa, const uint16_t*& wb) {
    wa = w + (size_t)(2 * p) * K;
    wb = w + (size_t)min(2 * p + 1, N - 1) * K;
  };
  Regs<PFC> pre;
  Plain16Pre<NX> xp;
  const uint16_t *wa0, *wb0;
  const int pc = p0 < npairs ? p0 : npairs - 1;
  map(pc, wa0, wb0);
  if constexpr (NX > 0) xp.load(a, K);
  __builtin_amdgcn_sched_barrier(0);
  if (NX > 0 || (PFC > 0 && p0 < npairs)) prefetch_rows<PFC>(wa0, wb0, pre);
  // the residual words of the first pair, requested now (no other wave writes them)
  const float r0 = x[min(2 * pc + (lane & 1), N - 1)];
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NX > 0) xp.finish(K, xs);
  else stage_plain16(a, K, xs);
  auto epi = [&](int p, float da, float db) {
    if (lane > 1) return;
    const int r = 2 * p + lane;
    if (r >= N) return;
    const float d = (lane == 0 ? da : db) + (bias ? to_f32<DT>(bias[r]) : 0.f);
    y[r] = fmaf(alpha, d, p == p0 ? r0 : x[r]);
  };
  run_pairs<DT, false, U, PFC, (U > 2)>(map, epi, xs, K, npairs, p0, gridDim.x * kGemvWaves, pre);
}

// y = W [x ; x0] + step (x, x0 f32 [W] each; w [W][K], K = 2 W padded to 8); y is neither
template <int DT, int U, int PFC>
__global__ __launch_bounds__(kGemvThreads) void mixer_loop_kernel(
    const float* __restrict__ x, const float* __restrict__ x0, const float* __restrict__ step,
    const uint16_t* __restrict__ w, int W, int K, float* __restrict__ y) {
  extern __shared__ float xs[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int npairs = (W + 1) >> 1;
  const int p0 = blockIdx.x * kGemvWaves + wave;
  auto map = [&](int p, const uint16_t*& wa, const uint16_t*& wb) {
    wa = w + (size_t)(2 * p) * K;
    wb = w + (size_t)min(2 * p + 1, W - 1) * K;
  };
  Regs<PFC> pre;
  const uint16_t *wa0, *wb0;
  map(p0 < npairs ? p0 : npairs - 1, wa0, wb0);
  if (PFC > 0 && p0 < npairs) prefetch_rows<PFC>(wa0, wb0, pre);
  if (W % 4 == 0) {
    for (int i = threadIdx.x * 4; i < K; i += kGemvThreads * 4)
      *reinterpret_cast<float4*>(xs + i) =
          i < W ? *reinterpret_cast<const float4*>(x + i)
                : i < 2 * W ? *reinterpret_cast<const float4*>(x0 + i - W)
                            : make_float4(0.f, 0.f, 0.f, 0.f);
  } else {
    for (int i = threadIdx.x; i < K; i += kGemvThreads)
      xs[i] = i < W ? x[i] : i < 2 * W ? x0[i - W] : 0.f;
  }
  __syncthreads();
  auto epi = [&](int p, float da, float db) {
    if (lane > 1) return;
    const int r = 2 * p + lane;
    if (r < W) y[r] = (lane == 0 ? da : db) + step[r];
  };
  run_pairs<DT, true, U, PFC>(map, epi, xs, K, npairs, p0, gridDim.x * kGemvWaves, pre);
}

}  // namespace cake

using namespace cake;

#define CAKE_MIX_LAUNCH(KERN, G, LDS, ...)                                            \
  do {                                                                                \
    auto kern_ = KERN;                                                                \
    if (!allow_lds(kern_, LDS)) return (int)hipErrorInvalidValue;                     \
    hipLaunchKernelGGL(kern_, dim3(G), dim3(kGemvThreads), LDS, st, __VA_ARGS__);     \
    return (int)hipGetLastError();                                                    \
  } while (0)

CAKE_API int cake_mixer_in(int dt, const float* resid, const void* norm_w, float eps, float off,
                           int ln, int Kn, const void* w, int K, int N, int n_raw, float* out,
                           int actf, const void* bias, void* act, hipStream_t st) {
  const size_t lds = (size_t)K * sizeof(float);
  if (K % 8 || K <= 0 || Kn < 1 || Kn > K || N <= 0 || n_raw < 0 || n_raw > N ||
      lds > 160 * 1024 || actf < 0 || actf >= kMixActs)
    return (int)hipErrorInvalidValue;
  const int g = grid_for((N + 1) / 2, 1024);
  const MixInArgs a{resid, (const uint16_t*)norm_w, (const uint16_t*)w, out, (const uint16_t*)bias,
                    (uint16_t*)act, eps, off, ln, Kn, K, N, n_raw, actf};
  // few rows and up to a workgroup a CU: above
  if (K >= 1024 && K <= 4096 && N <= 1024) {
    const int gs = mixer_in_pairs(a);
    DISPATCH_DT(dt, if (K <= 2048) CAKE_MIX_LAUNCH((mixer_in_split_kernel<DT, 1, 2>), gs, lds, a);
                else CAKE_MIX_LAUNCH((mixer_in_split_kernel<DT, 2, 4>), gs, lds, a));
  }
  if (K >= 1024 && K <= 4096 && N <= 2560) {
    const int rounds = (K + 511) / 512, waves = N <= 2048 ? 4 : 5;
#define CAKE_PAIR(R, W)                                                                                            \
  if (rounds == R && waves == W) {                                                                                 \
    hipLaunchKernelGGL((mixer_in_pair_kernel<DT, R, 64 * W>), dim3((mixer_in_pairs(a) + W - 1) / W), dim3(64 * W), \
                       lds, st, a);                                                                                \
    return (int)hipGetLastError();                                                                                 \
  }
#define CAKE_PAIRS(W) \
  CAKE_PAIR(2, W) CAKE_PAIR(3, W) CAKE_PAIR(4, W) CAKE_PAIR(5, W) CAKE_PAIR(6, W) CAKE_PAIR(7, W) CAKE_PAIR(8, W)
    DISPATCH_DT(dt, CAKE_PAIRS(4) CAKE_PAIRS(5));
#undef CAKE_PAIRS
#undef CAKE_PAIR
  }
#define CAKE_MIN(PF, NX) CAKE_MIX_LAUNCH((mixer_in_kernel<DT, 2, PF, NX>), g, lds, a)
  DISPATCH_DT(dt, if (K / 8 < 128) CAKE_MIN(0, 0); else if (K / 8 < 256) CAKE_MIN(2, 2);
              else if (K <= 4096) CAKE_MIN(4, 4);
              else if (K <= 8192) CAKE_MIN(4, 8); else CAKE_MIN(4, 0));
#undef CAKE_MIN
}

CAKE_API int cake_mixer_out(int dt, const void* a, const void* w, int K, int N, float alpha,
                            const void* bias, const float* x, float* y, hipStream_t st) {
  const size_t lds = (size_t)K * 2;
  if (K % 8 || K <= 0 || N <= 0 || lds > 160 * 1024) return (int)hipErrorInvalidValue;
  const int g = grid_for((N + 1) / 2, 1024);
#define CAKE_MOUT(PF, NX)                                                                   \
  CAKE_MIX_LAUNCH((mixer_out_kernel<DT, 4, PF, NX>), g, lds, (const uint16_t*)a,            \
                  (const uint16_t*)w, K, N, alpha, (const uint16_t*)bias, x, y)
  // (one or two rounds of 512 columns: 2048 rows of 512 / 1024 2.6 / 3.0 us, as left over of four 2.8 / 3.2)
  if (K <= 1024)
    DISPATCH_DT(dt, CAKE_MIX_LAUNCH((mixer_out_kernel<DT, 2, 0, 0>), g, lds, (const uint16_t*)a, (const uint16_t*)w, K, N,
                                    alpha, (const uint16_t*)bias, x, y));
  DISPATCH_DT(dt, if (K / 8 < 256) CAKE_MOUT(0, 0); else if (K <= 4096) CAKE_MOUT(4, 2);
              else if (K <= 8192) CAKE_MOUT(4, 4); else if (K <= 16384) CAKE_MOUT(4, 8);
              else if (K <= 28672) CAKE_MOUT(4, 14); else CAKE_MOUT(4, 0));
#undef CAKE_MOUT
}

CAKE_API int cake_mixer_loop(int dt, const float* x, const float* x0, const float* step,
                             const void* w, int W, int K, float* y, hipStream_t st) {
  const size_t lds = (size_t)K * sizeof(float);
  if (K % 8 || W <= 0 || K < 2 * W || y == x || y == x0 || lds > 160 * 1024)
    return (int)hipErrorInvalidValue;
  const int g = grid_for((W + 1) / 2, 1024);
#define CAKE_MLOOP(PF)                                                                          \
  CAKE_MIX_LAUNCH((mixer_loop_kernel<DT, 4, PF>), g, lds, x, x0, step, (const uint16_t*)w, W, K, y)
  DISPATCH_DT(dt, if (K / 8 < 256) CAKE_MLOOP(0); else CAKE_MLOOP(4));
#undef CAKE_MLOOP
}
