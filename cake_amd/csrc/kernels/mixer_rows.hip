// Row kernels of the hybrid designs: embedding rows, RMS / layer norm with an offset weight, and
// the input of a looped pass.  Residual rows are f32 [N][ldx], ldx = width padded to 8, zeros past
// the width; the activations they produce are [N][ldo] in the storage type, zero-padded.
#include "mixer_common.h"

namespace cake {

template <int DT>
__global__ __launch_bounds__(256) void mixer_embed_kernel(const void* table, const int* tok, int ld,
                                                          float* x, float* x0) {
  using E = typename St<DT>::E;
  const E* row = reinterpret_cast<const E*>(table) + (long long)tok[blockIdx.x] * ld;
  const long long o = (long long)blockIdx.x * ld;
  for (int i = threadIdx.x * 4; i < ld; i += 1024) {  // ld % 8 == 0
    float4 v;
    if constexpr (DT == kF32) {
      v = *reinterpret_cast<const float4*>(row + i);
    } else {
      const uint2 w = *reinterpret_cast<const uint2*>(row + i);
      v = make_float4(St<DT>::ld((uint16_t)(w.x & 0xffffu)), St<DT>::ld((uint16_t)(w.x >> 16)),
                      St<DT>::ld((uint16_t)(w.y & 0xffffu)), St<DT>::ld((uint16_t)(w.y >> 16)));
    }
    *reinterpret_cast<float4*>(x + o + i) = v;
    if (x0) *reinterpret_cast<float4*>(x0 + o + i) = v;
  }
}

struct NormArgs {
  const float* x;       // [*][ldx], columns [W, ldo) zero
  long long ldx;
  const int* rows;      // row of x per output row (null: the same)
  const int* where;     // or: output rows of each row of x, `copies` of them (else null, 1)
  int copies;
  const float* scale;   // factor per output row (null: 1)
  const float* w;       // [ldo], zeros past W
  float off, eps;
  int ln, W, ldo;
  void* out;            // [N][ldo]
};
constexpr int kNormCopies = 32;

// out[r] = scale[r] * norm(x[rows ? rows[r] : r]) * (off + w): the RMS norm x / rms, or (LN)
// the layer norm (x - mean) / sqrt(variance + eps).  Of a few rows a launch is its round trips to the
// memory, so the weights are asked for with the row (24 rows of 4096 3.1 us, after the sums 3.6);
// of many rows it is the bytes: a row that goes to several places is read and summed once (2048 rows
// of 4096 to six places each 20.3 us, gathered six times over 46).
template <int DT, bool LN, int NV>
__global__ __launch_bounds__(256) void mixer_norm_kernel(NormArgs a) {
  using E = typename St<DT>::E;
  __shared__ float red[16], fac[kNormCopies];
  __shared__ int dst[kNormCopies];
  const long long n = blockIdx.x;
  const int ldo = a.ldo, W = a.W, tid = threadIdx.x;
  const float* xr = a.x + (a.rows ? a.rows[n] : n) * a.ldx;
  float4 v[NV], wv[NV];  // rows up to 1024 NV stay in registers (ldo % 8 == 0, zeros past W)
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * 256 + tid) * 4;
    v[j] = wv[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i < ldo) {
      v[j] = *reinterpret_cast<const float4*>(xr + i);
      wv[j] = *reinterpret_cast<const float4*>(a.w + i);
    }
  }
  if (tid < a.copies) {   // read after the sums' barriers
    const int r = a.where ? a.where[n * a.copies + tid] : (int)n;
    dst[tid] = r;
    fac[tid] = a.scale ? a.scale[r] : 1.f;
  }
  float ss = 0.f, sum = 0.f;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if constexpr (LN) sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
    else ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
  }
  for (int i = 1024 * NV + tid; i < ldo; i += 256) {
    if constexpr (LN) sum += xr[i];
    else ss += xr[i] * xr[i];
  }
  float mean = 0.f;
  if constexpr (LN) {
    mean = block_sum(sum, red) / (float)W;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = (j * 256 + tid) * 4;
      v[j].x = i < W ? v[j].x - mean : 0.f;
      v[j].y = i + 1 < W ? v[j].y - mean : 0.f;
      v[j].z = i + 2 < W ? v[j].z - mean : 0.f;
      v[j].w = i + 3 < W ? v[j].w - mean : 0.f;
      ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
    }
    for (int i = 1024 * NV + tid; i < W; i += 256) ss += (xr[i] - mean) * (xr[i] - mean);
  }
  const float norm = sqrtf(block_sum(ss, red) / (float)W + a.eps);
  for (int c = 0; c < a.copies; ++c) {
    const float f = fac[c] / norm;
    E* o = reinterpret_cast<E*>(a.out) + (long long)dst[c] * ldo;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const int i = (j * 256 + tid) * 4;
      if (i >= ldo) continue;
      const float y[4] = {v[j].x * f * (a.off + wv[j].x), v[j].y * f * (a.off + wv[j].y),
                          v[j].z * f * (a.off + wv[j].z), v[j].w * f * (a.off + wv[j].w)};
      if constexpr (DT == kF32) {
        *reinterpret_cast<float4*>(o + i) = make_float4(y[0], y[1], y[2], y[3]);
      } else {
        *reinterpret_cast<uint2*>(o + i) = make_uint2(
            (uint32_t)St<DT>::st(y[0]) | ((uint32_t)St<DT>::st(y[1]) << 16),
            (uint32_t)St<DT>::st(y[2]) | ((uint32_t)St<DT>::st(y[3]) << 16));
      }
    }
    for (int i = 1024 * NV + tid; i < ldo; i += 256)
      o[i] = St<DT>::st(i < W ? (xr[i] - mean) * f * (a.off + a.w[i]) : 0.f);
  }
}

// a[n] = [x[n] | x0[n] | 0] (storage type), y[n] = step (zeros past W)
template <int DT>
__global__ __launch_bounds__(256) void mixer_loop_rows_kernel(const float* x, const float* x0,
                                                              int ldx, const float* step, int W,
                                                              void* a, int lda, float* y) {
  using E = typename St<DT>::E;
  const long long n = blockIdx.x;
  E* o = reinterpret_cast<E*>(a) + n * lda;
  if (DT != kF32 && W % 8 == 0 && lda % 4 == 0) {
    for (int i = threadIdx.x * 4; i < lda; i += 1024) {
      const float4 v = i < W ? *reinterpret_cast<const float4*>(x + n * ldx + i)
                       : i < 2 * W ? *reinterpret_cast<const float4*>(x0 + n * ldx + i - W)
                                   : make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<uint2*>(o + i) =
          make_uint2((uint32_t)St<DT>::st(v.x) | ((uint32_t)St<DT>::st(v.y) << 16),
                     (uint32_t)St<DT>::st(v.z) | ((uint32_t)St<DT>::st(v.w) << 16));
    }
    for (int i = threadIdx.x * 4; i < ldx; i += 1024)
      *reinterpret_cast<float4*>(y + n * ldx + i) =
          i < W ? *reinterpret_cast<const float4*>(step + i) : make_float4(0.f, 0.f, 0.f, 0.f);
    return;
  }
  for (int i = threadIdx.x; i < lda; i += 256)
    o[i] = St<DT>::st(i < W ? x[n * ldx + i] : i < 2 * W ? x0[n * ldx + i - W] : 0.f);
  for (int i = threadIdx.x; i < ldx; i += 256) y[n * ldx + i] = i < W ? step[i] : 0.f;
}

// out[n][c] = act(in[n][c] + bias[c]), f32 storage path of the up projection
__global__ __launch_bounds__(256) void mixer_act_kernel(int act, const float* in, long long ldi,
                                                        const float* bias, int N, int F, float* out,
                                                        long long ldo) {
  const long long total = (long long)N * F;
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (long long)gridDim.x * 256) {
    const long long n = i / F;
    const int c = (int)(i - n * F);
    out[n * ldo + c] = mix_act(act, in[n * ldi + c] + (bias ? bias[c] : 0.f));
  }
}

}  // namespace cake

using namespace cake;

CAKE_API int cake_mixer_embed(int dt, const void* table, const int* tok, int N, int ld, float* x,
                              float* x0, hipStream_t st) {
  if (N < 0 || ld <= 0 || ld % 8) return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((mixer_embed_kernel<DT>), dim3(N), dim3(256), 0, st, table,
                                     tok, ld, x, x0));
  return (int)hipGetLastError();
}

// rows: row of x per output row; or where [N][copies]: output rows of each of x's N rows
CAKE_API int cake_mixer_norm(int dt, const float* x, long long ldx, const int* rows, const int* where,
                             int copies, const float* scale, const float* w, float off, float eps,
                             int ln, int N, int W, void* out, int ldo, hipStream_t st) {
  // w holds ldo f32 values (zeros past W); x has ldo readable columns
  if (N < 0 || W <= 0 || W > ldo || ldo % 8 || ldx % 4 || ldx < ldo || copies < 1 ||
      copies > kNormCopies || (where ? rows != nullptr : copies != 1))
    return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  const NormArgs a{x, ldx, rows, where, copies, scale, w, off, eps, ln, W, ldo, out};
#define CAKE_NORM(LN, NV) hipLaunchKernelGGL((mixer_norm_kernel<DT, LN, NV>), dim3(N), dim3(256), 0, st, a)
#define CAKE_NORM_NV(LN) \
  if (ldo <= 2048) CAKE_NORM(LN, 2); else if (ldo <= 4096) CAKE_NORM(LN, 4); else CAKE_NORM(LN, 8)
  CAKE_MIX_DT(dt, { if (ln) { CAKE_NORM_NV(true); } else { CAKE_NORM_NV(false); } });
#undef CAKE_NORM_NV
#undef CAKE_NORM
  return (int)hipGetLastError();
}

CAKE_API int cake_mixer_loop_rows(int dt, const float* x, const float* x0, int ldx,
                                  const float* step, int N, int W, void* a, int lda, float* y,
                                  hipStream_t st) {
  if (N < 0 || W <= 0 || W > ldx || lda < 2 * W) return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((mixer_loop_rows_kernel<DT>), dim3(N), dim3(256), 0, st, x,
                                     x0, ldx, step, W, a, lda, y));
  return (int)hipGetLastError();
}

CAKE_API int cake_mixer_act(int act, const float* in, long long ldi, const float* bias, int N,
                            int F, float* out, long long ldo, hipStream_t st) {
  if (N < 0 || F <= 0 || ldi < F || ldo < F || act < 0 || act >= kMixActs)
    return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  long long g = ((long long)N * F + 255) / 256;
  if (g > 8192) g = 8192;
  hipLaunchKernelGGL(mixer_act_kernel, dim3((unsigned)g), dim3(256), 0, st, act, in, ldi, bias, N,
                     F, out, ldo);
  return (int)hipGetLastError();
}
