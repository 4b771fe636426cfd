// Products of up to eight rows whose weights are small: an output product that adds to the residual rows, and a
// gated product that norms them itself.
//
// A launch costs 1.6 us whatever it does, and weights of 8 .. 70 MB take 1.3 .. 10 us, so what counts is the launches and
// how long each takes to get under way.  A workgroup of eight waves takes four weight rows at a time (gated: four and
// their partners), every wave 128 of each 1024 k: a load is 256 bytes of four rows, in whole lines (the 16-row fragments
// of gemm_direct_kernel are 64 bytes of sixteen, which the address unit passes at half the rate), two steps of them under
// way.  They are the operands of 4 x 4 x 4 MFMAs as they come, sixteen blocks of k side by side; x lies in the LDS.  The
// residual rows are asked for before the weights (loads return in order) and normed while these come in, by every
// workgroup for itself: they are few.
// Output, norm and gate / up of 2048 wide rows, 8192 behind the gates, at 2 / 5 / 8 rows in three launches (slabs, their
// sum and norm, gated product) 23.7 / 23.5 / 24.5 us, in these two 17.5 / 19.3 / 20.6 (75 MB: 11.6 us).
#include <algorithm>

#include "gemm_kernel.h"

namespace cake {

struct FewArgs {
  const uint16_t* a;    // [M][lda]; NORM: null
  const float* h;       // NORM: rows [M][lda] to norm (RMS) with weights ln
  const uint16_t* ln;
  const uint16_t* b;    // [N][ldb], gated [2 N][ldb]
  uint16_t* c;          // gated: [M][ldc]
  float* r;             // else: [M][ldc] += x w^T
  long long lda, ldb, ldc;
  float eps;
  int M, N, K;
};

constexpr int kFewRows = 8, kFewNormK = 3072, kFewLds = 150 * 1024;

typedef short fs16x4 __attribute__((ext_vector_type(4)));
typedef _Float16 fh16x4 __attribute__((ext_vector_type(4)));

// sixteen 4 x 4 products over 4 k each: lane 4 b + i holds row i of block b of either operand
template <int DT>
__device__ __forceinline__ cf32x4 few_mfma(uint2 a, uint2 b, cf32x4 c) {
  if constexpr (DT == kBF16)
    return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(__builtin_bit_cast(fs16x4, a), __builtin_bit_cast(fs16x4, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_4x4x4f16(__builtin_bit_cast(fh16x4, a), __builtin_bit_cast(fh16x4, b), c, 0, 0, 0);
}

// the sum over the sixteen blocks: lane 16 q + j + 4 s (any s) gets row {0, 2, 1, 3}[q] of column j
__device__ __forceinline__ float few_sum(cf32x4 v) {
  const auto add32 = [](float x, float y) {
    const auto p = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(y), false, false);
    return __int_as_float((int)p[0]) + __int_as_float((int)p[1]);
  };
  const float a = add32(v[0], v[1]), b = add32(v[2], v[3]);
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_int(a), __float_as_int(b), false, false);
  float s = __int_as_float((int)p[0]) + __int_as_float((int)p[1]);
  s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x128, 0xf, 0xf, false));   // row_ror:8
  s += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(s), 0x124, 0xf, 0xf, false));   // row_ror:4
  return s;
}

// LDS bytes from a row of x to the next: 64 past a multiple of 256, so that the four rows that sixteen lanes read lie in
// banks of their own
__host__ __device__ constexpr int few_stride(int K) { return (K + 127) / 128 * 256 + 64; }
constexpr int few_lds(int MG, int QG, int K) { return 2 * 8 * ((QG * MG + 3) / 4 * 64) * 4 + 4 * MG * few_stride(K); }

// MG: groups of four rows of x; QG: groups of four weight rows at a time (gated: the second half of them gates' partners)
template <int DT, bool GATED, int MG, int QG>
__global__ __launch_bounds__(512, 4) void gemm_few_kernel(FewArgs g) {
  constexpr bool NORM = GATED;
  constexpr int NW = 8, TILES = QG * MG, COLS = QG * 4 / (GATED ? 2 : 1);
  constexpr int RED = (TILES + 3) / 4 * 64;   // floats of a wave's sums
  extern __shared__ __attribute__((aligned(16))) uint8_t few_smem[];
  float* const red = reinterpret_cast<float*>(few_smem);   // [2][NW][RED]
  uint8_t* const xs = few_smem + 2 * NW * RED * 4;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int chunks = (g.K + 127) / 128, cpw = (chunks + NW - 1) / NW, XS = few_stride(g.K);
  const int groups = (g.N + COLS - 1) / COLS;
  const int mine = (groups - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;   // >= 1
  const int r = lane & 3, kl = (lane >> 2) * 8;

  // rows past the last are the last one
  const uint16_t* wp[QG];
  const auto aim = [&](int grp) {
#pragma unroll
    for (int q = 0; q < QG; ++q) {
      const int n = grp * COLS + (GATED ? q % (QG / 2) : q) * 4 + r;
      wp[q] = g.b + (size_t)(min(n, g.N - 1) + (GATED && q >= QG / 2 ? g.N : 0)) * g.ldb + kl;
    }
  };
  uint4 w[2][QG];
  int lg = 0, lc = 0;   // the step to ask for: which of this workgroup's groups, of this wave's chunks of k
  aim(blockIdx.x);
  const auto ask = [&](uint4 (&to)[QG]) {
    const int k = (lc * NW + wave) * 128;
#pragma unroll
    for (int q = 0; q < QG; ++q) to[q] = make_uint4(0, 0, 0, 0);
    if (lg < mine && k + kl < g.K)
#pragma unroll
      for (int q = 0; q < QG; ++q) to[q] = ld_nt16(reinterpret_cast<const uint4*>(wp[q] + k));
    if (++lc == cpw) {
      lc = 0;
      if (++lg < mine) aim(blockIdx.x + lg * gridDim.x);
    }
  };
  if constexpr (NORM) {   // wave m norms row m
    constexpr int NV = kFewNormK / 256;
    float4 v[NV];
    uint2 lw[NV];
    const bool has = wave < g.M;
    const float* hr = g.h + (size_t)min(wave, g.M - 1) * g.lda;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = (j * 64 + lane) * 4;
      v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
      lw[j] = make_uint2(0, 0);
      if (has && i < g.K) {
        v[j] = *reinterpret_cast<const float4*>(hr + i);
        lw[j] = *reinterpret_cast<const uint2*>(g.ln + i);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    ask(w[0]);
    ask(w[1]);
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
    ss = wave_sum(ss);
    const float f = 1.f / sqrtf(ss / (float)g.K + g.eps);
    if (wave < 4 * MG)
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        const int i = (j * 64 + lane) * 4;
        if (i >= chunks * 128) continue;
        const uint16_t y[4] = {from_f32<DT>(v[j].x * f * to_f32<DT>((uint16_t)(lw[j].x & 0xffff))),
                               from_f32<DT>(v[j].y * f * to_f32<DT>((uint16_t)(lw[j].x >> 16))),
                               from_f32<DT>(v[j].z * f * to_f32<DT>((uint16_t)(lw[j].y & 0xffff))),
                               from_f32<DT>(v[j].w * f * to_f32<DT>((uint16_t)(lw[j].y >> 16)))};
        *reinterpret_cast<uint2*>(xs + wave * XS + i * 2) =
            has ? make_uint2(y[0] | (uint32_t)y[1] << 16, y[2] | (uint32_t)y[3] << 16) : make_uint2(0, 0);
      }
  } else {
    const int cpr = chunks * 16, total = 4 * MG * cpr;   // 16-byte pieces
    constexpr int XB = 4;
    for (int i0 = tid; i0 < total; i0 += 512 * XB) {
      uint4 v[XB];
#pragma unroll
      for (int u = 0; u < XB; ++u) {
        const int i = i0 + u * 512, t = i / cpr, c = i - t * cpr;
        v[u] = make_uint4(0, 0, 0, 0);
        if (i < total && t < g.M && c * 8 < g.K) v[u] = *reinterpret_cast<const uint4*>(g.a + (size_t)t * g.lda + c * 8);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i0 == tid) {
        ask(w[0]);
        ask(w[1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < XB; ++u) {
        const int i = i0 + u * 512, t = i / cpr, c = i - t * cpr;
        if (i < total) *reinterpret_cast<uint4*>(xs + t * XS + c * 16) = v[u];
      }
    }
    if (total <= tid) {   // (a thread without a piece)
      ask(w[0]);
      ask(w[1]);
    }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  const uint8_t* const xl = xs + r * XS + (lane >> 2) * 16;
  cf32x4 acc[QG][MG];
  int c = 0, done = 0;
  const auto step = [&](uint4 (&wv)[QG]) {
    if (c == 0) {
#pragma unroll
      for (int q = 0; q < QG; ++q)
#pragma unroll
        for (int m = 0; m < MG; ++m) acc[q][m] = cf32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int k = c * NW + wave;
    if (k < chunks) {
      uint4 x[MG];
#pragma unroll
      for (int m = 0; m < MG; ++m) x[m] = *reinterpret_cast<const uint4*>(xl + m * 4 * XS + k * 256);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int q = 0; q < QG; ++q)
#pragma unroll
          for (int m = 0; m < MG; ++m)
            acc[q][m] = few_mfma<DT>(h ? make_uint2(wv[q].z, wv[q].w) : make_uint2(wv[q].x, wv[q].y),
                                     h ? make_uint2(x[m].z, x[m].w) : make_uint2(x[m].x, x[m].y), acc[q][m]);
    }
    ask(wv);
    if (++c < cpw) return;
    c = 0;
    // the waves' sums meet in the LDS, four tiles in a row's sixteen lanes; two banks of it, so one barrier a group
    float* const rb = red + (done & 1) * (NW * RED);
#pragma unroll
    for (int t0 = 0; t0 < TILES; t0 += 4) {
      float s[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = t0 + t < TILES ? few_sum(acc[(t0 + t) / MG % QG][(t0 + t) % MG]) : 0.f;
      const int b = lane >> 2 & 3;
      rb[wave * RED + t0 * 16 + lane] = b == 0 ? s[0] : b == 1 ? s[1] : b == 2 ? s[2] : s[3];
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int grp = blockIdx.x + done * gridDim.x;
    if (tid < COLS * MG * 4) {
      const int col = tid % COLS, m = tid / COLS, n = grp * COLS + col;
      if (m < g.M && n < g.N) {
        float y[2];
#pragma unroll
        for (int h = 0; h < (GATED ? 2 : 1); ++h) {
          const int tile = (col / 4 + h * (QG / 2)) * MG + m / 4, i = col % 4;
          const int at = tile / 4 * 64 + (i == 1 ? 2 : i == 2 ? 1 : i) * 16 + tile % 4 * 4 + m % 4;
          y[h] = 0.f;
#pragma unroll
          for (int v = 0; v < NW; ++v) y[h] += rb[v * RED + at];
        }
        if constexpr (GATED) g.c[(size_t)m * g.ldc + n] = from_f32<DT>(silu(y[0]) * y[1]);
        else g.r[(size_t)m * g.ldc + n] += y[0];
      }
    }
    ++done;
  };
  const int steps = mine * cpw;
  for (int s = 0; s < steps; s += 2) {
    step(w[0]);
    if (s + 1 < steps) step(w[1]);
  }
}

template <int DT, bool GATED, int MG, int QG>
static int launch_few(const FewArgs& g, hipStream_t st) {
  static const hipError_t raised =
      hipFuncSetAttribute((const void*)gemm_few_kernel<DT, GATED, MG, QG>, hipFuncAttributeMaxDynamicSharedMemorySize, kFewLds);
  const int cols = QG * 4 / (GATED ? 2 : 1), groups = (g.N + cols - 1) / cols, lds = few_lds(MG, QG, g.K);
  if (raised != hipSuccess) return (int)raised;
  if (lds > kFewLds) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((gemm_few_kernel<DT, GATED, MG, QG>), dim3(std::min(groups, 512)), dim3(512), lds, st, g);
  return (int)hipGetLastError();
}
template <bool GATED, int QG>
static int run_few(int dt, const FewArgs& g, hipStream_t st) {
  if (dt == kBF16) return g.M <= 4 ? launch_few<kBF16, GATED, 1, QG>(g, st) : launch_few<kBF16, GATED, 2, QG>(g, st);
  return g.M <= 4 ? launch_few<kF16, GATED, 1, QG>(g, st) : launch_few<kF16, GATED, 2, QG>(g, st);
}

}  // namespace cake

using namespace cake;

// Whether the output product [H][K] and the gated one [2 I][H] of M rows are better off here: of H 32 .. 3072, K 64 .. 4096,
// I 64 .. 43000 within this line a block takes 0.79 .. 1.02 of the time.  Below 1024 columns some of a workgroup's eight waves
// have none, and many narrow rows are many of its turns: a block of H 256, I 2048 / 8192 / 32768 at 5 rows 24.2 / 27.5 / 36.5
// us in launches of its own, 23.5 / 28.8 / 43.9 here; H 512, I 4096 / 16384 27.9 / 34.4, 27.4 / 36.7.  4096 wide ones at 5 rows
// are not better off (output 9.9 us and norm in the next, 8.2 and 3.5; 28672 x 4096 38.1 and its norm, 37.6): a workgroup's x
// is as much as its weights, and the stream form moves those as fast.
CAKE_API int cake_gemm_few_pair(int M, int H, int K, long long I) {
  return M >= 1 && M <= kFewRows && H >= 8 && H <= kFewNormK && H % 8 == 0 && K >= 8 && K <= 4096 && K % 8 == 0 && I >= 1 &&
         I * H <= 44LL << 20 && (H >= 1024 || I <= 12LL * H);
}

// r [M][ldr] += a [M][lda] b^T, b [N][ldb]; M <= 8, rows of a and b on 16 bytes
CAKE_API int cake_gemm_few_add(int dt, const void* a, long long lda, const void* b, long long ldb, float* r, long long ldr,
                               int M, int N, int K, hipStream_t st) {
  if (!(dt == kBF16 || dt == kF16) || M < 1 || M > kFewRows || N < 1 || K < 8 || K % 8 || K > 4096 || lda < K || ldb < K ||
      ldr < N || lda % 8 || ldb % 8 || !a || !b || !r || (((uintptr_t)a | (uintptr_t)b) & 15))
    return (int)hipErrorInvalidValue;
  const FewArgs g{(const uint16_t*)a, nullptr, nullptr, (const uint16_t*)b, nullptr, r, lda, ldb, ldr, 0.f, M, N, K};
  return run_few<false, 1>(dt, g, st);
}

// c [M][ldc] = silu(x b0^T) (x b1^T), b0 the first N rows of b, b1 the others; x the RMS norm of h [M][ldh] with weights ln
// [K], in 16 bits; M <= 8, K <= 3072
CAKE_API int cake_gemm_few_gated(int dt, const float* h, long long ldh, const void* ln, float eps, const void* b,
                                 long long ldb, void* c, long long ldc, int M, int N, int K, hipStream_t st) {
  if (!(dt == kBF16 || dt == kF16) || M < 1 || M > kFewRows || N < 1 || K < 8 || K % 8 || K > kFewNormK || ldh < K ||
      ldb < K || ldc < N || ldh % 4 || ldb % 8 || !h || !ln || !b || !c || (((uintptr_t)h | (uintptr_t)b) & 15) ||
      ((uintptr_t)ln & 7))
    return (int)hipErrorInvalidValue;
  const FewArgs g{nullptr, h, (const uint16_t*)ln, (const uint16_t*)b, (uint16_t*)c, nullptr, ldh, ldb, ldc, eps, M, N, K};
  return run_few<true, 2>(dt, g, st);
}
