// What follows a product that left its sums in slabs ([slabs][M][N] f32, cake_gemm_slabs): the sum of a
// row's slabs goes straight into the work that reads the row next.
//
//   cake_slab_norm  x += alpha (sum + bias), and the norm of the new row (or the sum alone, or the norm);
//   cake_slab_rope  q, k, v rows of a Llama block: rotation, keys and values into the cache;
//   cake_slab_attn  the same and the rows' causal attention, for a short prompt from position 0.
//
// Of few rows a launch is its round trips to the memory, whatever it reads: the sum of eight slabs of 45
// rows of 4096 (4.2 us) and the norm behind it (4.0) are one launch here, and neither a strip's parts in the
// stream form (gemm_rows.h) nor the splits of a tile meet in memory first.
#include "gemm_kernel.h"

namespace cake {

struct SlabNormArgs {
  const float* ws;       // [slabs][M][N]
  float* x;              // residual rows [M][ldx]
  const uint16_t* bias;  // [N] or null
  const void* w;         // norm weights [N], 16-bit or (w32) f32; null: no norm
  void* out;             // [M][ldo]
  long long slab, ldx, ldo;
  int N, slabs, w32, ln;
  float alpha, off, eps;
};

// A workgroup has a row, a thread NV times four columns of it with SL slabs in flight; everything a row
// reads is asked for before the first sum.
template <int DT, int NV, int SL>
__global__ __launch_bounds__(1024) void slab_norm_kernel(SlabNormArgs a) {
  __shared__ float red[16];
  const int m = blockIdx.x, tid = threadIdx.x, nt = blockDim.x;
  float* xr = a.x + m * a.ldx;
  const float* row = a.ws + (size_t)m * a.N;
  float4 v[NV], wv[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * nt + tid) * 4;
    v[j] = wv[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (i >= a.N) continue;
    const float4 old = *reinterpret_cast<const float4*>(xr + i);
    if (a.w != nullptr) {
      if (a.w32) {
        wv[j] = *reinterpret_cast<const float4*>(static_cast<const float*>(a.w) + i);
      } else {
        const uint2 h = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(a.w) + i);
        wv[j] = make_float4(to_f32<DT>((uint16_t)(h.x & 0xffff)), to_f32<DT>((uint16_t)(h.x >> 16)),
                            to_f32<DT>((uint16_t)(h.y & 0xffff)), to_f32<DT>((uint16_t)(h.y >> 16)));
      }
    }
    float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.slabs == 0) { v[j] = old; continue; }
    if (a.bias != nullptr) {
      const uint2 h = *reinterpret_cast<const uint2*>(a.bias + i);
      s = make_float4(to_f32<DT>((uint16_t)(h.x & 0xffff)), to_f32<DT>((uint16_t)(h.x >> 16)),
                      to_f32<DT>((uint16_t)(h.y & 0xffff)), to_f32<DT>((uint16_t)(h.y >> 16)));
    }
    for (int s0 = 0; s0 < a.slabs; s0 += SL) {
      float4 p[SL];
#pragma unroll
      for (int e = 0; e < SL; ++e)
        p[e] = *reinterpret_cast<const float4*>(row + min(s0 + e, a.slabs - 1) * a.slab + i);
#pragma unroll
      for (int e = 0; e < SL; ++e)
        if (s0 + e < a.slabs) { s.x += p[e].x; s.y += p[e].y; s.z += p[e].z; s.w += p[e].w; }
    }
    v[j] = make_float4(fmaf(a.alpha, s.x, old.x), fmaf(a.alpha, s.y, old.y), fmaf(a.alpha, s.z, old.z),
                       fmaf(a.alpha, s.w, old.w));
    *reinterpret_cast<float4*>(xr + i) = v[j];
  }
  if (a.w == nullptr) return;
  float mean = 0.f, ss = 0.f;
  if (a.ln) {
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
    mean = block_sum(sum, red) / (float)a.N;
  }
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    if ((j * nt + tid) * 4 >= a.N) continue;
    v[j].x -= mean; v[j].y -= mean; v[j].z -= mean; v[j].w -= mean;
    ss += v[j].x * v[j].x + v[j].y * v[j].y + v[j].z * v[j].z + v[j].w * v[j].w;
  }
  const float f = 1.f / sqrtf(block_sum(ss, red) / (float)a.N + a.eps);
  uint16_t* o = static_cast<uint16_t*>(a.out) + m * a.ldo;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = (j * nt + tid) * 4;
    if (i >= a.N) continue;
    const uint16_t y[4] = {from_f32<DT>(v[j].x * f * (a.off + wv[j].x)), from_f32<DT>(v[j].y * f * (a.off + wv[j].y)),
                           from_f32<DT>(v[j].z * f * (a.off + wv[j].z)), from_f32<DT>(v[j].w * f * (a.off + wv[j].w))};
    *reinterpret_cast<uint2*>(o + i) = make_uint2(y[0] | (uint32_t)y[1] << 16, y[2] | (uint32_t)y[3] << 16);
  }
}

struct SlabRopeArgs {
  const float* ws;       // [slabs][T][(nh + 2 nkv) hd]: q heads, k heads, v heads
  uint16_t* q;           // [T][ldq], rotated
  uint16_t *kc, *vc;     // cache rows [nkv][S][hd]
  const float* inv_freq; // [hd / 2]
  long long slab;
  int slabs, ldq, nh, nkv, hd, pos0, S;
};

// An item is four columns of a head's first half and the four of the second half that turn with them, or
// four of each half of a value row.  A row's items take several workgroups, since one CU would read all
// slabs of it alone.
template <int DT, int SL>
__global__ __launch_bounds__(256) void slab_rope_kernel(SlabRopeArgs a) {
  __shared__ float s_sn[128], s_cs[128];
  const int t = blockIdx.x, pos = a.pos0 + t, half = a.hd >> 1, hv = half >> 2;
  const int heads = a.nh + 2 * a.nkv;
  const int p = blockIdx.y * 256 + threadIdx.x;
  const bool on = p < heads * hv;
  const int head = on ? p / hv : 0, i0 = on ? (p - head * hv) * 4 : 0;
  const float* src = a.ws + (size_t)t * heads * a.hd + head * a.hd + i0;
  float4 u = make_float4(0.f, 0.f, 0.f, 0.f), w = u;
  for (int s0 = 0; s0 < a.slabs; s0 += SL) {
    float4 x[SL], y[SL];
#pragma unroll
    for (int e = 0; e < SL; ++e) {
      const float* r = src + min(s0 + e, a.slabs - 1) * a.slab;
      x[e] = *reinterpret_cast<const float4*>(r);
      y[e] = *reinterpret_cast<const float4*>(r + half);
    }
    if (s0 == 0) {   // beside the loads
      for (int i = threadIdx.x; i < half; i += 256) sincosf((float)pos * a.inv_freq[i], &s_sn[i], &s_cs[i]);
      __syncthreads();
    }
#pragma unroll
    for (int e = 0; e < SL; ++e)
      if (s0 + e < a.slabs) {
        u.x += x[e].x; u.y += x[e].y; u.z += x[e].z; u.w += x[e].w;
        w.x += y[e].x; w.y += y[e].y; w.z += y[e].z; w.w += y[e].w;
      }
  }
  if (!on) return;
  const bool turns = head < a.nh + a.nkv;
  float c[4], s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    c[e] = turns ? s_cs[i0 + e] : 1.f;
    s[e] = turns ? s_sn[i0 + e] : 0.f;
  }
  const float lo[4] = {u.x, u.y, u.z, u.w}, hi[4] = {w.x, w.y, w.z, w.w};
  uint16_t ol[4], oh[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    ol[e] = from_f32<DT>(turns ? lo[e] * c[e] - hi[e] * s[e] : lo[e]);
    oh[e] = from_f32<DT>(turns ? lo[e] * s[e] + hi[e] * c[e] : hi[e]);
  }
  uint16_t* dst = head < a.nh ? a.q + (size_t)t * a.ldq + head * a.hd
                  : turns     ? a.kc + ((size_t)(head - a.nh) * a.S + pos) * a.hd
                              : a.vc + ((size_t)(head - a.nh - a.nkv) * a.S + pos) * a.hd;
  *reinterpret_cast<uint2*>(dst + i0) = make_uint2(ol[0] | (uint32_t)ol[1] << 16, ol[2] | (uint32_t)ol[3] << 16);
  *reinterpret_cast<uint2*>(dst + i0 + half) = make_uint2(oh[0] | (uint32_t)oh[1] << 16, oh[2] | (uint32_t)oh[3] << 16);
}

struct SlabAttnArgs {
  SlabRopeArgs r;        // (q, ldq unused)
  uint16_t* out;         // [T][ldo]
  long long ldo;
  int T;
  float scale_log2;
};

// Short prompts from position 0 (T <= 64): every key is one of these rows, so a workgroup of a query head sums
// and rotates its q, k and v, keeps them in LDS and runs the attention at once.  Bound by a launch's round trips:
// rotation and attention as two launches 9.2 us at 5 rows of 16 heads and 10.8 at 45 of 32, of which the
// attention's 6 read back what the rotation had written.  The heads that share a key head sum its rows each.
//
// S^T = K Q^T with the keys of a 32-key group dealt to the two 16-row tiles so that a lane's scores are eight
// keys in a row: they are the second operand of O^T = V^T P^T as they are.
template <int DT, int HD, int SL>
__global__ __launch_bounds__(512) void slab_attn_kernel(SlabAttnArgs b) {
  constexpr int LQ = HD + 8, LV = 64 + 8, HV = HD / 8, NKS = HD / 32, NT = HD / 32;
  __shared__ __attribute__((aligned(16))) uint16_t qs[64 * LQ], ks[64 * LQ], vt[HD * LV];
  const SlabRopeArgs& a = b.r;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, rep = a.nh / a.nkv, kv = h / rep;
  const bool writes = h % rep == 0;
  const int cols = (a.nh + 2 * a.nkv) * HD;
  const int head[3] = {h, a.nh + kv, a.nh + a.nkv + kv};

  // ---- q, k, v: an item is four columns of both halves of a row's three heads ----
  for (int p = tid; p < b.T * HV; p += 512) {
    const int t = p / HV, i0 = (p - t * HV) * 4;
    float4 x[3][2];
#pragma unroll
    for (int n = 0; n < 3; ++n) x[n][0] = x[n][1] = make_float4(0.f, 0.f, 0.f, 0.f);
    const float* row = a.ws + (size_t)t * cols + i0;
    for (int s0 = 0; s0 < a.slabs; s0 += SL) {
      float4 y[SL][3][2];
#pragma unroll
      for (int e = 0; e < SL; ++e)
#pragma unroll
        for (int n = 0; n < 3; ++n) {
          const float* r = row + min(s0 + e, a.slabs - 1) * a.slab + head[n] * HD;
          y[e][n][0] = *reinterpret_cast<const float4*>(r);
          y[e][n][1] = *reinterpret_cast<const float4*>(r + HD / 2);
        }
#pragma unroll
      for (int e = 0; e < SL; ++e)
        if (s0 + e < a.slabs)
#pragma unroll
          for (int n = 0; n < 3; ++n)
#pragma unroll
            for (int d = 0; d < 2; ++d) {
              x[n][d].x += y[e][n][d].x; x[n][d].y += y[e][n][d].y;
              x[n][d].z += y[e][n][d].z; x[n][d].w += y[e][n][d].w;
            }
    }
    float c[4], s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) sincosf((float)t * a.inv_freq[i0 + e], &s[e], &c[e]);
    uint2 w[3][2];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
      const float lo[4] = {x[n][0].x, x[n][0].y, x[n][0].z, x[n][0].w};
      const float hi[4] = {x[n][1].x, x[n][1].y, x[n][1].z, x[n][1].w};
      uint16_t ol[4], oh[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ol[e] = from_f32<DT>(n < 2 ? lo[e] * c[e] - hi[e] * s[e] : lo[e]);
        oh[e] = from_f32<DT>(n < 2 ? lo[e] * s[e] + hi[e] * c[e] : hi[e]);
        if (n == 2) {
          vt[(i0 + e) * LV + t] = ol[e];
          vt[(i0 + HD / 2 + e) * LV + t] = oh[e];
        }
      }
      w[n][0] = make_uint2(ol[0] | (uint32_t)ol[1] << 16, ol[2] | (uint32_t)ol[3] << 16);
      w[n][1] = make_uint2(oh[0] | (uint32_t)oh[1] << 16, oh[2] | (uint32_t)oh[3] << 16);
    }
    *reinterpret_cast<uint2*>(qs + t * LQ + i0) = w[0][0];
    *reinterpret_cast<uint2*>(qs + t * LQ + i0 + HD / 2) = w[0][1];
    *reinterpret_cast<uint2*>(ks + t * LQ + i0) = w[1][0];
    *reinterpret_cast<uint2*>(ks + t * LQ + i0 + HD / 2) = w[1][1];
    if (writes) {
      uint16_t* kr = a.kc + ((size_t)kv * a.S + t) * HD + i0;
      uint16_t* vr = a.vc + ((size_t)kv * a.S + t) * HD + i0;
      *reinterpret_cast<uint2*>(kr) = w[1][0];
      *reinterpret_cast<uint2*>(kr + HD / 2) = w[1][1];
      *reinterpret_cast<uint2*>(vr) = w[2][0];
      *reinterpret_cast<uint2*>(vr + HD / 2) = w[2][1];
    }
  }
  // values past the rows meet probabilities of zero
  const int pad = 64 - b.T;
  for (int p = tid; p < HD * pad; p += 512) vt[p / pad * LV + b.T + p % pad] = 0;
  __syncthreads();

  // ---- a wave: 16 query rows, half of the value columns ----
  const int q0 = (wave & 3) * 16, qi = q0 + l15, t0 = (wave >> 2) * NT;
  if (q0 >= b.T) return;
  const int groups = q0 < 32 ? 1 : 2;   // of 32 keys, up to the last query's own
  cf32x4 sc[2][2];
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      sc[k][u] = cf32x4{0.f, 0.f, 0.f, 0.f};
      if (k >= groups) continue;
      const int key = 32 * k + 8 * (l15 >> 2) + 4 * u + (l15 & 3);
#pragma unroll
      for (int d = 0; d < NKS; ++d)
        sc[k][u] = cmfma<DT>(*reinterpret_cast<const uint4*>(ks + key * LQ + 32 * d + 8 * g),
                             *reinterpret_cast<const uint4*>(qs + qi * LQ + 32 * d + 8 * g), sc[k][u]);
    }
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool seen = k < groups && 32 * k + 8 * g + 4 * u + e <= qi;   // (a query past the rows sees some key)
        sc[k][u][e] = seen ? sc[k][u][e] * b.scale_log2 : -INFINITY;
        m = fmaxf(m, sc[k][u][e]);
      }
  m = fmaxf(m, __shfl_xor(m, 16));
  m = fmaxf(m, __shfl_xor(m, 32));
  float l = 0.f;
  uint4 pf[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    uint32_t w[4];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint16_t y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = __builtin_amdgcn_exp2f(sc[k][u][e] - m);
        l += x;
        y[e] = from_f32<DT>(x);
      }
      w[2 * u] = y[0] | (uint32_t)y[1] << 16;
      w[2 * u + 1] = y[2] | (uint32_t)y[3] << 16;
    }
    pf[k] = make_uint4(w[0], w[1], w[2], w[3]);
  }
  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  const float inv = 1.f / l;
  uint16_t* o = b.out + (size_t)qi * b.ldo + h * HD;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int d0 = 16 * (t0 + t);
    cf32x4 acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (k < groups) acc = cmfma<DT>(*reinterpret_cast<const uint4*>(vt + (d0 + l15) * LV + 32 * k + 8 * g), pf[k], acc);
    if (qi < b.T)
      *reinterpret_cast<uint2*>(o + d0 + 4 * g) =
          make_uint2(from_f32<DT>(acc[0] * inv) | (uint32_t)from_f32<DT>(acc[1] * inv) << 16,
                     from_f32<DT>(acc[2] * inv) | (uint32_t)from_f32<DT>(acc[3] * inv) << 16);
  }
}

template <int DT, int NV>
static int launch_norm(const SlabNormArgs& a, int M, int threads, hipStream_t st) {
#define CAKE_SLAB(SL) hipLaunchKernelGGL((slab_norm_kernel<DT, NV, SL>), dim3(M), dim3(threads), 0, st, a)
  if (a.slabs <= 1) CAKE_SLAB(1); else if (a.slabs == 2) CAKE_SLAB(2); else if (a.slabs <= 4) CAKE_SLAB(4);
  else CAKE_SLAB(8);
#undef CAKE_SLAB
  return (int)hipGetLastError();
}

}  // namespace cake

using namespace cake;

// x[m] += alpha (sum over slabs of ws[.][m] + bias); with w (16-bit, or f32 if w32): out[m] = norm(x[m])
// (off + w), RMS norm or (ln) layer norm; no slabs: the norm of x as it is.  ws [slabs][M][N], x [M][ldx], out [M][ldo].
CAKE_API int cake_slab_norm(int dt, const float* ws, int slabs, float* x, long long ldx, const void* bias,
                            float alpha, const void* w, int w32, float off, float eps, int ln, int M, int N,
                            void* out, long long ldo, hipStream_t st) {
  if (M < 0 || N <= 0 || N % 4 || N > 8192 || slabs < 0 || ldx < N || ldx % 4 || (slabs && !ws) || !x ||
      (w && (!out || ldo < N || ldo % 4)) ||
      (((uintptr_t)ws | (uintptr_t)x | (w32 ? (uintptr_t)w : 0)) & 15) ||
      (((uintptr_t)bias | (uintptr_t)w | (uintptr_t)out) & 7) || !(dt == kBF16 || dt == kF16))
    return (int)hipErrorInvalidValue;
  if (M == 0) return 0;
  const SlabNormArgs a{ws, x, (const uint16_t*)bias, w, out, (long long)M * N, ldx, ldo, N, slabs, w32, ln, alpha,
                       off, eps};
  const int threads = N > 2048 ? 1024 : 512;
  if (dt == kBF16) return N <= 4096 ? launch_norm<kBF16, 1>(a, M, threads, st) : launch_norm<kBF16, 2>(a, M, threads, st);
  return N <= 4096 ? launch_norm<kF16, 1>(a, M, threads, st) : launch_norm<kF16, 2>(a, M, threads, st);
}

// cake_rope_kv of rows that are sums of slabs, q to [T][ldq]
CAKE_API int cake_slab_rope(int dt, const float* ws, int slabs, void* q, int ldq, int T, int nh, int nkv, int hd,
                            const float* inv_freq, int pos0, int S, void* kc, void* vc, hipStream_t st) {
  if (T < 0 || slabs < 1 || hd <= 0 || hd % 8 || hd > 256 || ldq % 4 || nh < 1 || nkv < 1 || pos0 < 0 ||
      pos0 + T > S || ((uintptr_t)ws & 15) || (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 7) ||
      !(dt == kBF16 || dt == kF16))
    return (int)hipErrorInvalidValue;
  if (T == 0) return 0;
  const SlabRopeArgs a{ws, (uint16_t*)q, (uint16_t*)kc, (uint16_t*)vc, inv_freq,
                       (long long)T * (nh + 2 * nkv) * hd, slabs, ldq, nh, nkv, hd, pos0, S};
  const dim3 grid(T, ((nh + 2 * nkv) * (hd / 8) + 255) / 256);
#define CAKE_SLAB(DT, SL) hipLaunchKernelGGL((slab_rope_kernel<DT, SL>), grid, dim3(256), 0, st, a)
#define CAKE_SLAB_DT(DT) if (slabs == 1) CAKE_SLAB(DT, 1); else if (slabs == 2) CAKE_SLAB(DT, 2); else CAKE_SLAB(DT, 4)
  if (dt == kBF16) { CAKE_SLAB_DT(kBF16); } else { CAKE_SLAB_DT(kF16); }
#undef CAKE_SLAB_DT
#undef CAKE_SLAB
  return (int)hipGetLastError();
}

// cake_slab_rope of a prompt's first T <= 64 rows (position 0 on), and their causal attention to out [T][ldo];
// head sizes of 64 and 128
CAKE_API int cake_slab_attn(int dt, const float* ws, int slabs, void* out, long long ldo, int T, int nh, int nkv,
                            int hd, const float* inv_freq, int S, void* kc, void* vc, float scale, hipStream_t st) {
  if (T < 0 || T > 64 || slabs < 1 || !(hd == 64 || hd == 128) || nh < 1 || nkv < 1 || nh % nkv || T > S ||
      ldo < (long long)nh * hd || ldo % 4 || ((uintptr_t)ws & 15) ||
      (((uintptr_t)out | (uintptr_t)kc | (uintptr_t)vc) & 7) || !(dt == kBF16 || dt == kF16))
    return (int)hipErrorInvalidValue;
  if (T == 0) return 0;
  const SlabAttnArgs a{{ws, nullptr, (uint16_t*)kc, (uint16_t*)vc, inv_freq, (long long)T * (nh + 2 * nkv) * hd, slabs,
                        0, nh, nkv, hd, 0, S}, (uint16_t*)out, ldo, T, scale * 1.4426950408889634f};
#define CAKE_SLAB(DT, HD) \
  if (slabs <= 2) hipLaunchKernelGGL((slab_attn_kernel<DT, HD, 2>), dim3(nh), dim3(512), 0, st, a); \
  else hipLaunchKernelGGL((slab_attn_kernel<DT, HD, 4>), dim3(nh), dim3(512), 0, st, a)
  if (dt == kBF16) { if (hd == 128) { CAKE_SLAB(kBF16, 128); } else { CAKE_SLAB(kBF16, 64); } }
  else { if (hd == 128) { CAKE_SLAB(kF16, 128); } else { CAKE_SLAB(kF16, 64); } }
#undef CAKE_SLAB
  return (int)hipGetLastError();
}
