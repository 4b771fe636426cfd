// Routed experts of the hybrid designs: every token runs the `top` experts of largest router
// logit on its row times that expert's score (a sigmoid, not renormalised).
//
//   * rows: expert_route (choice and scores), expert_plan (rows sorted by expert and the tile
//     list of the grouped products), the grouped GEMM (gemm_grouped.hip; f32: here) over
//     gathered, scaled rows, expert_sum (each row's experts into the residual);
//   * one token, 16-bit: expert_up picks the experts in its prologue and streams only their up
//     rows, expert_down sums the chosen experts' output columns onto the residual.
#include <algorithm>

#include "gemv_kernel.h"
#include "mixer_common.h"

namespace cake {

constexpr int kMaxExperts = 1024, kMaxTop = 32;

// One wave: the k-th largest of E logits (ties: the smaller index), k = 0 .. top - 1, into
// id / score of lane k.  VPL = 64-logit blocks.
template <int VPL>
__device__ __forceinline__ void wave_top(const float* logits, int E, int top, int lane, int& id,
                                         float& score) {
  float v[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) v[j] = lane + 64 * j < E ? logits[lane + 64 * j] : -INFINITY;
  id = 0;
  score = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = v[0];
#pragma unroll
    for (int j = 1; j < VPL; ++j) best = fmaxf(best, v[j]);
    best = wave_max(best);
    int e = 0x7fffffff;  // the smallest index that holds it
#pragma unroll
    for (int j = VPL - 1; j >= 0; --j) {
      const unsigned long long hit =
          __builtin_amdgcn_ballot_w64(v[j] == best && lane + 64 * j < E);
      if (hit != 0ull) e = 64 * j + __builtin_ctzll(hit);
    }
    e = min(e, E - 1);  // logits that compare to nothing (NaN) still give a valid expert
#pragma unroll
    for (int j = 0; j < VPL; ++j)
      if (lane + 64 * j == e) v[j] = -INFINITY;
    if (lane == k) {
      id = e;
      score = 1.f / (1.f + expf(-best));
    }
  }
}

template <int VPL>
__global__ __launch_bounds__(256) void expert_route_kernel(const float* logits, long long ldl,
                                                           int N, int E, int top, int* ids,
                                                           float* score) {
  const int n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= N) return;
  int id;
  float s;
  wave_top<VPL>(logits + n * ldl, E, top, lane, id, s);
  if (lane < top) {
    ids[(long long)n * top + lane] = id;
    score[(long long)n * top + lane] = s;
  }
}

// Rows of a tile of the grouped products up (F columns) and down (W) on all CUs: the height whose rounds cost least.
// A height from the mean alone overflows its tiles: up and down of 64 experts 2048 x 1856, 135 skewed rows each 291 us
// (192 rows a tile), 258 (256) by the counts.
//
// A product of more than kGroupedShort k takes the tiles of gemm_ws.h: t = rounds (step k / 64 + end) us, a last round of less
// than an eighth of the CUs at less, at least the memory's (5.8 TB/s) and half of what the last round leaves idle; of few
// tiles, of 128 columns, a share of the step.  A shorter one takes the tiles of gemm_4w.h: t = rounds (step k / 64 + end), at
// least the memory's; tiles of a 224-row list run at 192 rows and fewer or at 256, in between.  The up product's k says which
// heights there are.  Over 20 expert sizes in even and independent groups of 66 .. 500 rows 0.32 % off the best height on the
// average where both k are long, 0.56 % where one or both are short (as if both products ran on the up product's tiles, without
// the idle half, 0.37 and 0.72: 16 of 2816 x 1024 at 240 independent rows 94.0 us, 84.9 so; 256 of 512 x 4096 at 192 719, 653).
constexpr int kHeights[4] = {160, 192, 224, 256}, kHeightsShort[4] = {128, 160, 192, 256};
__device__ __forceinline__ int tile_rows(int W, int q) { return W > kGroupedShort ? kHeights[q] : kHeightsShort[q]; }
__device__ inline float height_us(int rows, int tiles, int N, int K, float bytes) {
  if (K <= kGroupedShort) {
    constexpr float kStep[5] = {1.106f, 1.161f, 1.38f, 1.422f, 1.547f}, kEnd[5] = {5.4f, 7.76f, 8.64f, 9.39f, 11.64f};
    const int q = rows / 32 - 4;
    return fmaxf((tiles * ((N + 255) / 256) + 255) / 256 * (kStep[q] * ((K + 63) / 64) + kEnd[q]), bytes / 8.2e6f);
  }
  constexpr float kStep[4] = {1.124f, 1.152f, 1.299f, 1.339f}, kEnd[4] = {5.53f, 7.80f, 7.07f, 8.42f};
  const int q = max(rows / 32 - 5, 0);
  const bool few = tiles * ((N + 255) / 256) <= (q == 0 ? 128 : 64);   // (gemm_inst_grouped.hip)
  const int body = few && q > 0 ? 3 : q;
  const float r = tiles * (few ? (N + 127) / 128 : (N + 255) / 256) / 256.f, whole = floorf(r), part = r - whole;
  const float rounds = whole + (part > 0.f ? fminf(1.f, 0.82f + 1.42f * part) : 0.f), mem = bytes / 5.8e6f;
  const float one = kStep[body] * (few ? 0.448f : 1.f) * ((K + 63) / 64) + kEnd[body] * (few ? 1.54f : 1.f);
  return fmaxf(rounds * one, whole > 0.f ? mem + 0.5f * (rounds - r) * one : mem);
}
__device__ inline int tile_height(const int (&tiles)[4], int E, int M, int F, int W) {
  const float bytes = ((float)E * F * W + (float)M * (F + W)) * 2;
  int best = 0;
  float least = 0.f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const float us = height_us(tile_rows(W, q), tiles[q], F, W, bytes) + height_us(tile_rows(W, q), tiles[q], W, F, bytes);
    if (q == 0 || us < least) {
      best = q;
      least = us;
    }
  }
  return tile_rows(W, best);
}

// Entries (token, k) sorted by expert: scale[p] = score of sorted row p, where[entry] = p; the tile
// list [expert, first sorted row, rows, 0] of BM-row tiles (0: tile_height of an expert's F x W up
// matrix), entry max_tiles [their number, BM, 0, 0].  VPL > 0: the choice of a few rows (kPlanEntries entries
// at most) is made here from the logits, whose launch would be mostly its own time (13 rows of 64 experts 3.5 +
// 5.8 us, 6.3 so).
constexpr int kPlanEntries = 1024;
template <int VPL>
__global__ __launch_bounds__(1024) void expert_plan_kernel(const float* logits, long long ldl, const int* ids,
                                                           const float* score, int N, int top, int E, int BM,
                                                           int F, int W, float* scale, int* where, int4* tiles,
                                                           int max_tiles) {
  __shared__ int cnt[kMaxExperts], scan[2][kMaxExperts], fit[4];
  __shared__ int own_id[VPL > 0 ? kPlanEntries : 1];
  __shared__ float own_score[VPL > 0 ? kPlanEntries : 1];
  constexpr int U = VPL > 0 ? 1 : 16;  // entries in flight per thread
  const int tid = threadIdx.x, M = N * top;
  if constexpr (VPL > 0) {
    const int lane = tid & 63;
    for (int n = tid >> 6; n < N; n += 16) {
      int id;
      float s;
      wave_top<VPL>(logits + n * ldl, E, top, lane, id, s);
      if (lane < top) {
        own_id[n * top + lane] = id;
        own_score[n * top + lane] = s;
      }
    }
    ids = own_id;
    score = own_score;
  }
  cnt[tid] = 0;
  if (tid < 4) fit[tid] = 0;
  __syncthreads();
  for (int i0 = tid; i0 < M; i0 += 1024 * U) {
    int e[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = i0 + 1024 * u < M ? ids[i0 + 1024 * u] : -1;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e[u] >= 0) atomicAdd(&cnt[e[u]], 1);
  }
  __syncthreads();
  const int c = cnt[tid];
  if (BM == 0) {   // tiles of every height, over all experts
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      int n = (c + tile_rows(W, q) - 1) / tile_rows(W, q);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o);
      if ((tid & 63) == 0) atomicAdd(&fit[q], n);
    }
    __syncthreads();
    BM = tile_height(fit, E, M, F, W);
  }
  // inclusive scans of the counts and of the tile counts (one thread per expert)
  const int nt = (c + BM - 1) / BM;
  scan[0][tid] = c;
  scan[1][tid] = nt;
  for (int o = 1; o < 1024 && o < E; o <<= 1) {
    __syncthreads();
    const int a = tid >= o ? scan[0][tid - o] : 0, b = tid >= o ? scan[1][tid - o] : 0;
    __syncthreads();
    scan[0][tid] += a;
    scan[1][tid] += b;
  }
  const int first = scan[0][tid] - c, tile0 = scan[1][tid] - nt;
  for (int t = 0; t < nt; ++t)
    if (tile0 + t < max_tiles)
      tiles[tile0 + t] = make_int4(tid, first + t * BM, min(BM, c - t * BM), 0);
  if (tid == E - 1) tiles[max_tiles] = make_int4(min(scan[1][tid], max_tiles), BM, 0, 0);
  cnt[tid] = first;  // cursors
  __syncthreads();
  for (int i0 = tid; i0 < M; i0 += 1024 * U) {
    int e[U];
    float s[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int i = i0 + 1024 * u;
      e[u] = i < M ? ids[i] : -1;
      s[u] = i < M ? score[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (e[u] >= 0) {
        const int i = i0 + 1024 * u, p = atomicAdd(&cnt[e[u]], 1);
        scale[p] = s[u];
        where[i] = p;
      }
  }
}

// x[n] += alpha * sum over k of y[where[n][k]].  Bound by its bytes at many tokens and by round trips
// at few: the row of x and eight experts' rows are asked for at once (2048 x 4096, six each, 168 MB: 38.1 ->
// 32.2 us, 5.2 TB/s; 13 x 2048 6.9 -> 6.3).
template <int DT>
__global__ __launch_bounds__(256) void expert_sum_kernel(const void* y, long long ldy,
                                                         const int* where, int top, int W,
                                                         float alpha, float* x, long long ldx) {
  using E = typename St<DT>::E;
  using V = std::conditional_t<DT == kF32, float4, uint2>;
  constexpr int U = 8;
  const long long n = blockIdx.x;
  const int* wp = where + n * top;
  const bool wide = ldx % 4 == 0 && ((uintptr_t)x & 15) == 0;
  for (int i = threadIdx.x * 4; i < W; i += 1024) {  // ldy a multiple of 4: whole reads
    float* xr = x + n * ldx + i;
    const bool whole = wide && i + 4 <= W;
    float o[4] = {0.f, 0.f, 0.f, 0.f};
    if (whole) {
      const float4 v = *reinterpret_cast<const float4*>(xr);
      o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < W) o[e] = xr[e];
    }
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < top; k0 += U) {
      V v[U];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + k < top)
          v[k] = *reinterpret_cast<const V*>(reinterpret_cast<const E*>(y) + (long long)wp[k0 + k] * ldy + i);
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + k < top) {
          if constexpr (DT == kF32) {
            s[0] += v[k].x; s[1] += v[k].y; s[2] += v[k].z; s[3] += v[k].w;
          } else {
            s[0] += to_f32<DT>((uint16_t)(v[k].x & 0xffffu));
            s[1] += to_f32<DT>((uint16_t)(v[k].x >> 16));
            s[2] += to_f32<DT>((uint16_t)(v[k].y & 0xffffu));
            s[3] += to_f32<DT>((uint16_t)(v[k].y >> 16));
          }
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = fmaf(alpha, s[e], o[e]);
    if (whole)
      *reinterpret_cast<float4*>(xr) = make_float4(o[0], o[1], o[2], o[3]);
    else
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (i + e < W) xr[e] = o[e];
  }
}

// The same of 16-bit rows up to 4096 NV wide, and the norm of the new row for what reads it next: out[n] =
// norm(x[n]) (off + w).  A thread has four columns (NV times), so that a row stays in registers between the
// sum and the norm.
template <int DT, int NV>
__global__ __launch_bounds__(1024) void expert_sum_norm_kernel(const uint16_t* y, long long ldy, const int* where,
                                                               int top, int W, float alpha, float* x, long long ldx,
                                                               const float* w, float off, float eps, int ln,
                                                               uint16_t* out, long long ldo) {
  constexpr int U = 8;
  __shared__ float red[16];
  const long long n = blockIdx.x;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int* wp = where + n * top;
  float* xr = x + n * ldx;
  float4 v[NV], wv[NV];
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * nt + tid) * 4;
    v[j] = wv[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= W) continue;
    const float4 old = *reinterpret_cast<const float4*>(xr + i);
    wv[j] = *reinterpret_cast<const float4*>(w + i);
    float s[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < top; k0 += U) {
      uint2 p[U];
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + k < top) p[k] = *reinterpret_cast<const uint2*>(y + (long long)wp[k0 + k] * ldy + i);
#pragma unroll
      for (int k = 0; k < U; ++k)
        if (k0 + k < top) {
          s[0] += to_f32<DT>((uint16_t)(p[k].x & 0xffffu));
          s[1] += to_f32<DT>((uint16_t)(p[k].x >> 16));
          s[2] += to_f32<DT>((uint16_t)(p[k].y & 0xffffu));
          s[3] += to_f32<DT>((uint16_t)(p[k].y >> 16));
        }
    }
    v[j] = make_float4(fmaf(alpha, s[0], old.x), fmaf(alpha, s[1], old.y), fmaf(alpha, s[2], old.z),
                       fmaf(alpha, s[3], old.w));
    *reinterpret_cast<float4*>(xr + i) = v[j];
    sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  const float mean = ln ? block_sum(sum, red) / (float)W : 0.f;
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if ((j * nt + tid) * 4 >= W) continue;
    v[j].x -= mean; v[j].y -= mean; v[j].z -= mean; v[j].w -= mean;
    ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
  }
  const float f = 1.f / sqrtf(block_sum(ss, red) / (float)W + eps);
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * nt + tid) * 4;
    if (i >= W) continue;
    const uint16_t o[4] = {from_f32<DT>(v[j].x * f * (off + wv[j].x)), from_f32<DT>(v[j].y * f * (off + wv[j].y)),
                           from_f32<DT>(v[j].z * f * (off + wv[j].z)), from_f32<DT>(v[j].w * f * (off + wv[j].w))};
    *reinterpret_cast<uint2*>(out + n * ldo + i) = make_uint2(o[0] | (uint32_t)o[1] << 16, o[2] | (uint32_t)o[3] << 16);
  }
}

// f32 grouped product: out[row0 + r] = act(a[row0 + r] W[expert]^T) for the tiles' rows (BM 32),
// act < 0: none.  K % 8 == 0.
__global__ __launch_bounds__(256) void expert_gemm32_kernel(const float* a, long long lda,
                                                            const float* w, long long ldw,
                                                            long long w_expert, const int4* tiles,
                                                            int N, int K, int act, float* out,
                                                            long long ldo) {
  if ((int)blockIdx.x >= tiles[gridDim.x].x) return;
  const int4 t = tiles[blockIdx.x];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l15 = lane & 15, g = lane >> 4;
  const int n = blockIdx.y * 64 + wave * 16 + l15;
  const float* wr = w + t.x * w_expert + (long long)min(n, N - 1) * ldw;
  const float* ar[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) ar[j] = a + (long long)(t.y + min(16 * j + l15, t.z - 1)) * lda;
  cf32x4 acc[2] = {cf32x4{0.f, 0.f, 0.f, 0.f}, cf32x4{0.f, 0.f, 0.f, 0.f}};
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  for (int k0 = 0; k0 < K; k0 += 16) {  // K % 8 == 0: the last step may be half a step
    const int k = k0 + 4 * g;
    const uint4 bw = k < K ? *reinterpret_cast<const uint4*>(wr + k) : zero;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      acc[j] = mm_piece<kF32>(k < K ? *reinterpret_cast<const uint4*>(ar[j] + k) : zero, bw, acc[j]);
  }
  if (n >= N) return;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = 16 * j + 4 * g + e;
      if (r < t.z) out[(long long)(t.y + r) * ldo + n] = act < 0 ? acc[j][e] : mix_act(act, acc[j][e]);
    }
}

// ---------------------------------------------------------------------------
// one token, 16-bit weights
// ---------------------------------------------------------------------------
struct ExpertUpArgs {
  const float* resid;
  const uint16_t* norm_w;
  float eps, off;
  int ln, Kn;
  const float* logits;   // [E]
  int E, top;
  const uint16_t* w;     // [E][FP][K]
  int K, FP, act;
  uint16_t* out;         // [top][FP]
  int* sel;              // [top] chosen experts
};

// norm prologue, choice of the experts by every wave (VPL logits a lane: it stands before the first weight; 6 of 64 with four
// a lane 31.9 us of 3648 x 4096, with one 31.2; of 1856 x 2048 11.2, 10.5), out[k] = act(score_k * (W_up x))
template <int DT, int U, int PFC, int NX, int VPL>
__global__ __launch_bounds__(kGemvThreads) void expert_up_kernel(ExpertUpArgs a) {
  extern __shared__ float xs[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int half = a.FP >> 1, npairs = a.top * half, K = a.K;
  const int p0 = blockIdx.x * kGemvWaves + wave;
  NormPre<DT, NX> xp;
  if constexpr (NX > 0) xp.load(a.resid, a.norm_w, K);
  int id;
  float score;
  wave_top<VPL>(a.logits, a.E, a.top, lane, id, score);
  if (blockIdx.x == 0 && wave == 0 && lane < a.top) a.sel[lane] = id;
  auto map = [&](int p, const uint16_t*& wa, const uint16_t*& wb) {
    const int k = p / half;
    const int e = __builtin_amdgcn_readlane(id, __builtin_amdgcn_readfirstlane(k));
    wa = a.w + ((size_t)e * a.FP + 2 * (p - k * half)) * K;
    wb = wa + K;
  };
  Regs<PFC> pre;
  const uint16_t *wa0, *wb0;
  map(p0 < npairs ? p0 : npairs - 1, wa0, wb0);
  if (NX > 0 || (PFC > 0 && p0 < npairs)) prefetch_rows<PFC>(wa0, wb0, pre);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NX > 0) xp.finish_off(a.eps, K, a.Kn, a.off, a.ln, xs);
  else stage_norm_off<DT>(a.resid, a.norm_w, a.eps, K, a.Kn, a.off, a.ln, xs);
  auto epi = [&](int p, float da, float db) {
    const int k = p / half;
    const float s = __builtin_bit_cast(
        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, score),
                                         __builtin_amdgcn_readfirstlane(k)));
    if (lane > 1) return;
    a.out[(size_t)k * a.FP + 2 * (p - k * half) + lane] =
        from_f32<DT>(mix_act(a.act, s * (lane == 0 ? da : db)));
  };
  run_pairs<DT, true, U, PFC>(map, epi, xs, K, npairs, p0, gridDim.x * kGemvWaves, pre);
}

struct ExpertDownArgs {
  const uint16_t* a;     // [top][FP]
  const int* sel;
  int top;
  const uint16_t* w;     // [E][W][FP]
  int FP, W;
  float alpha;
  const float* x;
  float* y;              // may be x
};

// y[r] = x[r] + alpha sum_k W_down[sel_k][r] a_k: the chosen experts' rows as one row of top FP
// columns, U 16-byte chunks of a row pair in flight per lane
template <int DT, int NW>
__global__ __launch_bounds__(64 * NW) void expert_down_kernel(ExpertDownArgs a,
                                                                   uint32_t inv_nch) {
  constexpr int U = 4;
  extern __shared__ float smem[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(smem);
  __shared__ uint32_t first[kMaxTop];  // chunk of an expert's row 0, less its flat position
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int npairs = (a.W + 1) >> 1, nch = a.FP >> 3, stride = gridDim.x * NW;
  const int total = a.top * nch, p0 = blockIdx.x * NW + wave;
  const uint4* w = reinterpret_cast<const uint4*>(a.w);
  if ((int)threadIdx.x < a.top)
    first[threadIdx.x] = (uint32_t)a.sel[threadIdx.x] * (uint32_t)a.W * nch - threadIdx.x * nch;
  __syncthreads();
  uint4 va[U], vb[U];
  auto load = [&](int p, int c0) __attribute__((always_inline)) {
    const uint32_t ra = (uint32_t)(2 * p) * nch, rb = (uint32_t)min(2 * p + 1, a.W - 1) * nch;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(c0 + 64 * u + lane, total - 1);
      const uint32_t f = first[inv_nch ? __umulhi((uint32_t)c, inv_nch) : c] + c;  // c / nch
      va[u] = ld_nt16(w + (f + ra));
      vb[u] = ld_nt16(w + (f + rb));
    }
  };
  if (p0 < npairs) load(p0, 0);  // ahead of the input row
  for (int i = threadIdx.x * 8; i < a.top * a.FP; i += 64 * NW * 8)
    *reinterpret_cast<uint4*>(xs + i) = *reinterpret_cast<const uint4*>(a.a + i);
  __syncthreads();
  for (int p = p0; p < npairs; p += stride) {
    const int ra = 2 * p, rb = min(2 * p + 1, a.W - 1);
    const float r = a.x[lane & 1 ? rb : ra];
    float aa = 0.f, ab = 0.f;
    for (int c0 = 0; c0 < total; c0 += 64 * U) {
      uint4 ca[U], cb[U];
#pragma unroll
      for (int u = 0; u < U; ++u) { ca[u] = va[u]; cb[u] = vb[u]; }
      const bool same = c0 + 64 * U < total;
      if (same || p + stride < npairs) load(same ? p : p + stride, same ? c0 + 64 * U : 0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + 64 * u + lane;
        if (c < total) fma_chunk<DT, false>(xs, c, ca[u], cb[u], aa, ab);
      }
    }
    aa = wave_sum(aa);
    ab = wave_sum(ab);
    if (lane < 2 && ra + lane < a.W) a.y[ra + lane] = fmaf(a.alpha, lane == 0 ? aa : ab, r);
  }
}

}  // namespace cake

using namespace cake;

static bool routing_ok(int E, int top) {
  return E > 0 && E <= kMaxExperts && top > 0 && top <= kMaxTop && top <= E;
}

CAKE_API int cake_expert_route(const float* logits, long long ldl, int N, int E, int top, int* ids,
                               float* score, hipStream_t st) {
  if (!routing_ok(E, top) || N < 0 || ldl < E) return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  const dim3 g((N + 3) / 4);
  if (E <= 64)
    hipLaunchKernelGGL((expert_route_kernel<1>), g, dim3(256), 0, st, logits, ldl, N, E, top, ids, score);
  else if (E <= 256)
    hipLaunchKernelGGL((expert_route_kernel<4>), g, dim3(256), 0, st, logits, ldl, N, E, top, ids, score);
  else
    hipLaunchKernelGGL((expert_route_kernel<16>), g, dim3(256), 0, st, logits, ldl, N, E, top, ids, score);
  return (int)hipGetLastError();
}

// max_tiles >= sum over experts of ceil(rows / BM): N top / BM + min(E, N top) is enough; the list
// has one entry more (their number)
// BM 0: the height that suits the groups, of experts of F x W (up) and W x F
CAKE_API int cake_expert_plan(const int* ids, const float* score, int N, int top, int E, int BM, int F,
                              int W, float* scale, int* where, void* tiles, int max_tiles, hipStream_t st) {
  if (!routing_ok(E, top) || N <= 0 || BM < 0 || (BM == 0 && (F <= 0 || W <= 0)) ||
      max_tiles < (long long)N * top / (BM > 0 ? BM : kHeightsShort[0]) + (E < (long long)N * top ? E : N * top))
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((expert_plan_kernel<0>), dim3(1), dim3(1024), 0, st, nullptr, 0, ids, score, N, top, E, BM, F, W,
                     scale, where, (int4*)tiles, max_tiles);
  return (int)hipGetLastError();
}

// cake_expert_route and cake_expert_plan of a few rows (N top <= 1024) in one launch
CAKE_API int cake_expert_route_plan(const float* logits, long long ldl, int N, int top, int E, int BM, int F, int W,
                                    float* scale, int* where, void* tiles, int max_tiles, hipStream_t st) {
  if (!routing_ok(E, top) || N <= 0 || ldl < E || BM < 0 || (BM == 0 && (F <= 0 || W <= 0)) ||
      (long long)N * top > kPlanEntries ||
      max_tiles < N * top / (BM > 0 ? BM : kHeightsShort[0]) + (E < N * top ? E : N * top))
    return (int)hipErrorInvalidValue;
#define CAKE_PLAN(VPL)                                                                                           \
  hipLaunchKernelGGL((expert_plan_kernel<VPL>), dim3(1), dim3(1024), 0, st, logits, ldl, nullptr, nullptr, N, top, E, \
                     BM, F, W, scale, where, (int4*)tiles, max_tiles)
  if (E <= 64) CAKE_PLAN(1); else if (E <= 256) CAKE_PLAN(4); else CAKE_PLAN(16);
#undef CAKE_PLAN
  return (int)hipGetLastError();
}

CAKE_API int cake_expert_sum(int dt, const void* y, long long ldy, const int* where, int N, int top,
                             int W, float alpha, float* x, long long ldx, hipStream_t st) {
  if (N < 0 || top <= 0 || W <= 0 || ldy < (W + 3) / 4 * 4 || ldy % 4 || ldx < W)
    return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((expert_sum_kernel<DT>), dim3(N), dim3(256), 0, st, y, ldy,
                                     where, top, W, alpha, x, ldx));
  return (int)hipGetLastError();
}

// ... and the norm of the new rows: 16-bit types, W % 4 == 0 up to 8192, w [W] f32, out [N][ldo]
CAKE_API int cake_expert_sum_norm(int dt, const void* y, long long ldy, const int* where, int N, int top, int W,
                                  float alpha, float* x, long long ldx, const float* w, float off, float eps, int ln,
                                  void* out, long long ldo, hipStream_t st) {
  if (N < 0 || top <= 0 || W <= 0 || W % 4 || W > 8192 || ldy < W || ldy % 4 || ldx < W || ldx % 4 || ldo < W ||
      ldo % 4 || (((uintptr_t)x | (uintptr_t)w) & 15) || (((uintptr_t)y | (uintptr_t)out) & 7) ||
      !(dt == kBF16 || dt == kF16))
    return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  const int nt = W > 2048 ? 1024 : W > 1024 ? 512 : 256;
#define CAKE_SUM_NORM(DT, NV)                                                                                   \
  hipLaunchKernelGGL((expert_sum_norm_kernel<DT, NV>), dim3(N), dim3(nt), 0, st, (const uint16_t*)y, ldy, where, \
                     top, W, alpha, x, ldx, w, off, eps, ln, (uint16_t*)out, ldo)
  if (dt == kBF16) { if (W <= 4096) CAKE_SUM_NORM(kBF16, 1); else CAKE_SUM_NORM(kBF16, 2); }
  else { if (W <= 4096) CAKE_SUM_NORM(kF16, 1); else CAKE_SUM_NORM(kF16, 2); }
#undef CAKE_SUM_NORM
  return (int)hipGetLastError();
}

CAKE_API int cake_expert_gemm32(const float* a, long long lda, const float* w, long long ldw,
                                long long w_expert, const void* tiles, int max_tiles, int N, int K,
                                int act, float* out, long long ldo, hipStream_t st) {
  if (max_tiles <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 4 || ldw % 4 || w_expert % 4 || ldo < N ||
      act >= kMixActs)
    return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(expert_gemm32_kernel, dim3(max_tiles, (N + 63) / 64), dim3(256), 0, st, a, lda,
                     w, ldw, w_expert, (const int4*)tiles, N, K, act, out, ldo);
  return (int)hipGetLastError();
}

CAKE_API int cake_expert_up(int dt, const float* resid, const void* norm_w, float eps, float off,
                            int ln, int Kn, const float* logits, int E, int top, const void* w,
                            int K, int FP, int act, void* out, int* sel, hipStream_t st) {
  const size_t lds = (size_t)K * sizeof(float);
  if (!routing_ok(E, top) || K <= 0 || K % 8 || Kn < 1 || Kn > K || FP <= 0 || FP % 8 || act < 0 ||
      act >= kMixActs || lds > 160 * 1024)
    return (int)hipErrorInvalidValue;
  const ExpertUpArgs a{resid, (const uint16_t*)norm_w, eps, off, ln, Kn, logits, E, top,
                       (const uint16_t*)w, K, FP, act, (uint16_t*)out, sel};
  const dim3 g(grid_for(top * (FP / 2), 1024));
#define CAKE_EUP_RUN(KERN)                                                     \
  do {                                                                         \
    auto kern_ = KERN;                                                         \
    if (!allow_lds(kern_, lds)) return (int)hipErrorInvalidValue;              \
    hipLaunchKernelGGL(kern_, g, dim3(kGemvThreads), lds, st, a);              \
    return (int)hipGetLastError();                                             \
  } while (0)
#define CAKE_EUP(PF, NX)                                                       \
  do {                                                                         \
    if (E <= 64) CAKE_EUP_RUN((expert_up_kernel<DT, 2, PF, NX, 1>));           \
    if (E <= 256) CAKE_EUP_RUN((expert_up_kernel<DT, 2, PF, NX, 4>));          \
    CAKE_EUP_RUN((expert_up_kernel<DT, 2, PF, NX, 16>));                       \
  } while (0)
  DISPATCH_DT(dt, if (K / 8 < 256) CAKE_EUP(0, 0); else if (K <= 4096) CAKE_EUP(4, 4);
              else if (K <= 8192) CAKE_EUP(4, 8); else CAKE_EUP(4, 0));
#undef CAKE_EUP
#undef CAKE_EUP_RUN
}

CAKE_API int cake_expert_down(int dt, const void* in, const int* sel, int top, const void* w,
                              int E, int FP, int W, float alpha, const float* x, float* y,
                              hipStream_t st) {
  const size_t lds = (size_t)top * FP * 2;
  // 16-byte chunks of all experts within 32-bit indexes
  if (!routing_ok(E, top) || FP <= 0 || FP % 8 || W <= 0 || lds > 156 * 1024 ||
      (long long)E * W * (FP / 8) >= 0xffffffffll)
    return (int)hipErrorInvalidValue;
  const ExpertDownArgs a{(const uint16_t*)in, sel, top, (const uint16_t*)w, FP, W, alpha, x, y};
  // ceil(2^32 / nch): exact quotients for chunk indexes below 2^16 (0: one chunk per row)
  const uint32_t inv = (uint32_t)((0x100000000ull + FP / 8 - 1) / (FP / 8));
  const auto run = [&](auto kern, int waves) {
    if (!allow_lds(kern, lds)) return (int)hipErrorInvalidValue;
    const int g = std::min(((W + 1) / 2 + waves - 1) / waves, 4096 / waves);
    hipLaunchKernelGGL(kern, dim3(g), dim3(64 * waves), lds, st, a, inv);
    return (int)hipGetLastError();
  };
  // every workgroup stages the whole input row: eight waves a workgroup halve those reads where they
  // still reach every compute unit (6 of 3616 columns to 4096 rows: 31.7 -> 30.2 us) and leave none
  // with more row pairs than four would (4 of 2048 to 6000 rows, 375 workgroups: 16.7 -> 18.1)
  const int n4 = ((W + 1) / 2 + 3) / 4, n8 = (n4 + 1) / 2;
  const bool wide = (W + 1) / 2 >= 2048 && (n8 + 255) / 256 * 2 <= (n4 + 255) / 256;
  DISPATCH_DT(dt, return wide ? run(expert_down_kernel<DT, 8>, 8) : run(expert_down_kernel<DT, 4>, 4));
}
