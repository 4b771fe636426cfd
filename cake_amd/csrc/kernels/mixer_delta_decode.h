// The gated delta rule (mixer_delta.hip) of one token per sequence, as a body that a launch of its own and
// the one that also streams the feed-forward's rows (mixer_beside.hip) run.
#pragma once
#include "mixer_common.h"

namespace cake {

struct DeltaArgs {
  const void* proj;       // [N][ldp] q | k | v | gate columns (storage type; decode: f32)
  long long ldp;
  const float* ab;        // [N][ldab]: a (H) then b (H)
  long long ldab;
  int N, H, G, dim, vdim, EP, taps;
  float eps;              // read-out norm
  const float* conv;      // [taps][C] f32
  const float* a_log;     // [H] f32
  const float* dt_bias;   // [H] f32
  const float* norm_w;    // [vdim] f32
  int DR;                 // dim padded to 64
  float* qn;              // [N + 15][G][DR], zeros past dim
  float* kn;              // [N + 15][G][DR]
  float* vv;              // [N + 15][H][vdim]
  float* tp;              // [NC][H][2][16][16]: T, P
  float* gm;              // [NC][H][4][16]: g_i, beta_i, G_15,i, g_15
  float* o;               // [N][H][vdim]
  float* state;
  float* ring;
  long long s_slot, r_slot;
  const int* row_pos;     // [N]
  const int* row_slot;    // [N]
  const int* row_seq0;    // [N] packed row of the sequence's first token in this step
  const SeqRow* seq;      // [B]
  const int2* chunk;      // [NC]: packed row of the first token, tokens
  const int* chunk0;      // [B]: first chunk of the sequence
  int NC;
  void* out;              // [N][ldo]
  long long ldo;
};

__device__ __forceinline__ int delta_channels(const DeltaArgs& a) {
  return 2 * a.G * a.dim + a.H * a.vdim;
}

// One token of row b, head h, 512 threads: thread = 4 columns of a few rows of S.
// proj is f32 here.  RPT rows per thread.
constexpr int kDdThreads = 512;
struct DeltaDecLds {
  __attribute__((aligned(16))) float part[kDdThreads * 4];
  float q[256], k[256], v[256], u[256];
  float red[16], sn[2];
};
template <int DT, int RPT>
__device__ __forceinline__ void mixer_delta_decode_body(const DeltaArgs& a, DeltaDecLds& s_, int h, int b) {
  using E = typename St<DT>::E;
  auto &q = s_.q, &k = s_.k, &v = s_.v, &u = s_.u;
  auto& red = s_.red;
  auto& sn = s_.sn;
  auto& part = s_.part;
  const int tid = threadIdx.x;
  const int R = a.H / a.G, gh = h / R;
  const int pos = a.row_pos[b], slot = a.row_slot[b];
  const int C = delta_channels(a);
  const int e4 = a.EP >> 2, ng = kDdThreads / e4;  // column pieces, row groups
  const int cg = tid % e4, rg = tid / e4, c = 4 * cg;
  const bool live = rg < ng;
  float* st = a.state + slot * a.s_slot + (long long)h * a.dim * a.EP;
  // the state first: its loads cover the convolution
  float4 S[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg + ng * i;
    S[i] = live && r < a.dim && pos > 0
               ? *reinterpret_cast<const float4*>(st + (long long)r * a.EP + c)
               : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  const float* pj = reinterpret_cast<const float*>(a.proj) + (long long)b * a.ldp;
  float* ring = a.ring + slot * a.r_slot;
  const int nch = 2 * a.dim + a.vdim;
  const bool own_qk = h % R == 0;
  // everything else that is read, before the first use of any: one after the other they were six round
  // trips to the memory (16 heads of 128 x 128, one row 7.9 -> 7.15 us)
  const float* ab = a.ab + (long long)b * a.ldab;
  const float a_log = a.a_log[h], a_in = ab[h] + a.dt_bias[h], b_in = ab[a.H + h];
  float norm_w = 0.f, gate = 0.f;
  if (tid < a.vdim) {
    norm_w = a.norm_w[tid];
    gate = pj[C + h * a.vdim + tid];
  }
  for (int x = tid; x < nch; x += kDdThreads) {
    const bool isv = x >= 2 * a.dim;
    const int ch = isv ? 2 * a.G * a.dim + h * a.vdim + x - 2 * a.dim
                       : x < a.dim ? gh * a.dim + x : (a.G + gh) * a.dim + x - a.dim;
    const float cur = pj[ch];
    float y = a.conv[(long long)(a.taps - 1) * C + ch] * cur;
    for (int j0 = 1; j0 < a.taps; j0 += 3) {   // three earlier inputs at a time
      float w[3], in[3];
#pragma unroll
      for (int e = 0; e < 3; ++e) {
        const int j = min(j0 + e, a.taps - 1);
        w[e] = a.conv[(long long)(a.taps - 1 - j) * C + ch];
        in[e] = ring[(long long)((pos + a.taps - j) % a.taps) * C + ch];
      }
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (j0 + e < a.taps && j0 + e <= pos) y = fmaf(w[e], in[e], y);
    }
    y = silu32(y);
    if (isv) v[x - 2 * a.dim] = y;
    else if (x < a.dim) q[x] = y;
    else k[x - a.dim] = y;
    if (isv || own_qk) ring[(long long)(pos % a.taps) * C + ch] = cur;
  }
  __syncthreads();
  {  // unit norms: wave 0 the query, wave 1 the key
    const int w = tid >> 6, lane = tid & 63;
    if (w < 2) {
      const float* x = w == 0 ? q : k;
      float ss = 0.f;
      for (int d = lane; d < a.dim; d += 64) ss += x[d] * x[d];
      ss = wave_sum(ss);
      if (lane == 0)
        sn[w] = 1.f / sqrtf(ss + 1e-6f) / (w == 0 ? sqrtf((float)a.dim) : 1.f);
    }
  }
  __syncthreads();
  const float rq = sn[0], rk = sn[1];
  const float dec = expf(-expf(a_log) * softplus32(a_in));
  const float beta = sigmoid32(b_in);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg + ng * i;
    const float kr = live && r < a.dim ? k[r] * rk : 0.f;
    S[i].x *= dec; S[i].y *= dec; S[i].z *= dec; S[i].w *= dec;
    acc.x = fmaf(kr, S[i].x, acc.x); acc.y = fmaf(kr, S[i].y, acc.y);
    acc.z = fmaf(kr, S[i].z, acc.z); acc.w = fmaf(kr, S[i].w, acc.w);
  }
  if (live) *reinterpret_cast<float4*>(part + rg * a.EP + c) = acc;
  __syncthreads();
  for (int d = tid; d < a.vdim; d += kDdThreads) {
    float s = 0.f;
    for (int g = 0; g < ng; ++g) s += part[g * a.EP + d];
    u[d] = beta * (v[d] - s);
  }
  __syncthreads();
  float uv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) uv[e] = c + e < a.vdim ? u[c + e] : 0.f;
  acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg + ng * i;
    if (live && r < a.dim) {
      const float kr = k[r] * rk, qr = q[r] * rq;
      S[i].x = fmaf(kr, uv[0], S[i].x); S[i].y = fmaf(kr, uv[1], S[i].y);
      S[i].z = fmaf(kr, uv[2], S[i].z); S[i].w = fmaf(kr, uv[3], S[i].w);
      *reinterpret_cast<float4*>(st + (long long)r * a.EP + c) = S[i];
      acc.x = fmaf(qr, S[i].x, acc.x); acc.y = fmaf(qr, S[i].y, acc.y);
      acc.z = fmaf(qr, S[i].z, acc.z); acc.w = fmaf(qr, S[i].w, acc.w);
    }
  }
  if (live) *reinterpret_cast<float4*>(part + rg * a.EP + c) = acc;
  __syncthreads();
  float ov = 0.f;  // vdim <= 256 < threads
  if (tid < a.vdim)
    for (int g = 0; g < ng; ++g) ov += part[g * a.EP + tid];
  const float rms = 1.f / sqrtf(block_sum(ov * ov, red) / (float)a.vdim + a.eps);
  if (tid < a.vdim)
    reinterpret_cast<E*>(a.out)[(long long)b * a.ldo + h * a.vdim + tid] =
        St<DT>::st(ov * rms * norm_w * silu32(gate));
}

static inline bool delta_shape_ok(int H, int G, int dim, int vdim, int EP, int taps) {
  return H > 0 && G > 0 && H % G == 0 && dim > 0 && dim <= 256 && vdim > 0 && vdim <= 256 &&
         EP >= vdim && EP % 4 == 0 && EP <= 256 && taps >= 1;
}

}  // namespace cake
