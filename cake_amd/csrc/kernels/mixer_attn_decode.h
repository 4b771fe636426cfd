// Softmax attention of one token per sequence (16- and 32-bit), as a body that a launch of its own
// (mixer_attn.hip) and the one that also streams the feed-forward's rows (mixer_beside.hip) run.
#pragma once
#include "mixer_common.h"

namespace cake {

// ---------------------------------------------------------------------------
// decode attention (one token per sequence)
// ---------------------------------------------------------------------------
struct MixDecArgs {
  const float* proj;     // [B][ldp] f32: q | k | v | gate columns
  long long ldp;
  const int* pos;        // [B]
  const int* slot;       // [B]
  const float2* cs;
  int rd2, qk_norm, sink, gated;
  float eps, scale_log2;
  void* kc;
  void* vc;
  long long k_slot, v_slot;
  void* out;             // [B][ldo]
  long long ldo;
  int H, G, dim, vdim, DP, DVP, S, nsplit;
  float* part;           // [B][ngt][nsplit][16][DVP + 2]
  unsigned int* ticket;  // [B][ngt], zero between launches
};

// rotation + norm of one head by one wave: lane handles dims 4 lane .. +3 (dim <= 256)
__device__ __forceinline__ void head_rot_norm(const float* src, int dim, int lane,
                                              const float2* cs, int rd2, int qk_norm, float eps,
                                              float* x) {
  const int d0 = 4 * lane;
#pragma unroll
  for (int e = 0; e < 4; ++e) x[e] = d0 + e < dim ? src[d0 + e] : 0.f;
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const int i = 2 * lane + p;
    if (i < rd2) {
      const float2 t = cs[i];
      const float u = x[2 * p], v = x[2 * p + 1];
      x[2 * p] = u * t.x - v * t.y;
      x[2 * p + 1] = v * t.x + u * t.y;
    }
  }
  if (qk_norm) {
    const float ss = wave_sum(x[0] * x[0] + x[1] * x[1] + x[2] * x[2] + x[3] * x[3]);
    const float r = 1.f / sqrtf(ss / (float)dim + eps);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] *= r;
  }
}

template <int DT, int CLS, int NW> struct MixDecLds {
  using E = typename St<DT>::E;
  __attribute__((aligned(16))) E qs[16 * (CLS + St<DT>::EPC)];
  __attribute__((aligned(16))) E kcur[CLS];
  __attribute__((aligned(16))) E vcur[CLS];
  float red_m[NW][16], red_l[NW][16];
  float red_o[NW][16][CLS + 1];
  int last;
};

// workgroup (gt of ngt, split sp, row b) of a decode launch, 64 NW threads
template <int DT, int CLS, bool EXACT, int NW>
__device__ __forceinline__ void mixer_attn_decode_body(const MixDecArgs& a, MixDecLds<DT, CLS, NW>& s_, int gt,
                                                       int ngt, int sp, int b) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC;
  constexpr int NKS = CLS / St<DT>::KSTEP, NVT = CLS / 16;
  constexpr bool kPrefetch = DT != kF32 && CLS <= 128;
  const int DP = EXACT ? CLS : a.DP, DVP = EXACT ? CLS : a.DVP;
  const int nks = EXACT ? NKS : DP / St<DT>::KSTEP, nvt = EXACT ? NVT : DVP / 16;
  auto& qs = s_.qs;
  auto& red_o = s_.red_o;
  auto &kcur = s_.kcur, &vcur = s_.vcur;
  auto &red_m = s_.red_m, &red_l = s_.red_l;
  int& s_last = s_.last;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int R = a.H / a.G, npg = (R + 15) / 16;      // 16-row query tiles per kv head
  const int hk = gt / npg, r0 = (gt - hk * npg) * 16;
  const int nr = min(16, R - r0);
  const int pos = a.pos[b], slot = a.slot[b];
  // key split: multiples of 128 keys, the last active one owns the new key
  const int Tk = pos + 1;
  const int kps = ((Tk + a.nsplit - 1) / a.nsplit + 127) / 128 * 128;
  const int nact = (Tk + kps - 1) / kps;
  if (sp >= nact) return;
  const bool owner = sp == nact - 1;
  const int kbeg = sp * kps, klim = min(kbeg + kps, pos);  // cached keys [kbeg, klim)
  const float* pj = a.proj + (long long)b * a.ldp;
  const float2* cs = a.cs + (long long)pos * a.rd2;
  E* kb = reinterpret_cast<E*>(a.kc) + slot * a.k_slot + (long long)hk * a.S * a.DP;
  E* vb = reinterpret_cast<E*>(a.vc) + slot * a.v_slot + (long long)hk * a.DVP * a.S;

  // the wave's first block of keys is requested ahead of the prologue.  Row i of score block u is
  // key 8 (i / 4) + 4 u + i % 4: the two blocks' accumulators of a lane group are then eight keys in
  // a row, and a value piece is one 16-byte load (as two of 8 bytes 16 positions apart the loads of
  // 256 keys took 2 us longer)
  uint4 kf[2][NKS];
  VFrag<DT> vf[NVT];
  auto load_k = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const E* kp = kb + (long long)(k0 + 8 * (l15 >> 2) + 4 * u + (l15 & 3)) * DP + g * EPC;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (EXACT || ks < nks) kf[u][ks] = *reinterpret_cast<const uint4*>(kp + ks * 4 * EPC);
    }
  };
  auto load_vs = [&](int k0) {
#pragma unroll
    for (int t = 0; t < NVT; ++t)
      if (EXACT || t < nvt) {
        const E* vp = vb + (long long)(16 * t + l15) * a.S + k0 + 8 * g;
        if constexpr (DT == kF32) {
          vf[t].lo = *reinterpret_cast<const float4*>(vp);
          vf[t].hi = *reinterpret_cast<const float4*>(vp + 4);
        } else {
          const uint4 w = *reinterpret_cast<const uint4*>(vp);
          vf[t].lo = make_uint2(w.x, w.y);
          vf[t].hi = make_uint2(w.z, w.w);
        }
      }
  };
  int k0 = kbeg + 32 * wave;
  if (kPrefetch && k0 < klim) { load_k(k0); load_vs(k0); }
  // this thread's first two gate values, first needed at the very end
  const float* gate = pj + (long long)(a.H + a.G) * a.dim + (long long)a.G * a.vdim +
                      (long long)(hk * R + r0) * a.vdim;
  float gpre[2] = {0.f, 0.f};
  if (a.gated)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if (tid + 64 * NW * i < nr * a.vdim) gpre[i] = gate[tid + 64 * NW * i];

  // rows past nr and value columns past vdim stay unwritten: they only reach accumulator
  // columns / rows that no output reads
  for (int r = wave; r < nr + (owner ? 1 : 0); r += NW) {
    const bool isk = r == nr;
    const float* src = isk ? pj + (long long)(a.H + hk) * a.dim
                           : pj + (long long)(hk * R + r0 + r) * a.dim;
    float x[4];
    head_rot_norm(src, a.dim, lane, cs, a.rd2, a.qk_norm, a.eps, x);
    E* dst = isk ? kcur : qs + r * (CLS + EPC);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (4 * lane + e < DP) dst[4 * lane + e] = St<DT>::st(x[e]);  // zeros past dim
  }
  if (owner) {
    const float* vsrc = pj + (long long)(a.H + a.G) * a.dim + (long long)hk * a.vdim;
    for (int d = tid; d < a.vdim; d += 64 * NW) {
      const E v = St<DT>::st(vsrc[d]);
      vcur[d] = v;
      if (r0 == 0) vb[(long long)d * a.S + pos] = v;
    }
  }
  __syncthreads();
  if (owner && r0 == 0)
    for (int d = tid; d < DP; d += 64 * NW) kb[(long long)pos * DP + d] = kcur[d];

  uint4 qf[NKS];
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks)
    qf[ks] = (EXACT || ks < nks)
                 ? *reinterpret_cast<const uint4*>(qs + l15 * (CLS + EPC) + (ks * 4 + g) * EPC)
                 : make_uint4(0, 0, 0, 0);
  cf32x4 o[NVT];
#pragma unroll
  for (int t = 0; t < NVT; ++t) o[t] = cf32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  if (owner && wave == 0) {  // the new key starts wave 0's softmax
    cf32x4 sc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks)
      if (EXACT || ks < nks) {
        const uint4 kk = *reinterpret_cast<const uint4*>(kcur + (ks * 4 + g) * EPC);
        sc = mm_piece<DT>(kk, qf[ks], sc);  // every A row is the new key: sc[e] = its score
      }
    m = sc[0] * a.scale_log2;
    l = g == 0 ? 1.f : 0.f;
#pragma unroll
    for (int t = 0; t < NVT; ++t)
      if (EXACT || t < nvt)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[t][e] = St<DT>::ld(vcur[16 * t + 4 * g + e]);
  }
  for (; k0 < klim; k0 += 32 * NW) {
    if constexpr (!kPrefetch) { load_k(k0); load_vs(k0); }
    cf32x4 s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = cf32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (EXACT || ks < nks) s[u] = mm_piece<DT>(kf[u][ks], qf[ks], s[u]);
    }
    const int kn = k0 + 32 * NW;
    if constexpr (kPrefetch) { if (kn < klim) load_k(kn); }
    float mx = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = k0 + 8 * g + 4 * u + e < klim;
        s[u][e] = ok ? s[u][e] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, s[u][e]);
      }
    mx = group_max(mx);
    const float mn = fmaxf(m, mx);  // finite: the block's first key is below klim
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    float rs = 0.f;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[u][e] = __builtin_amdgcn_exp2f(s[u][e] - mn);
        rs += s[u][e];
      }
    m = mn;
    l = l * alpha + rs;
    const PFrag<DT> pf = pack_p<DT>(s[0], s[1]);
#pragma unroll
    for (int t = 0; t < NVT; ++t)
      if (EXACT || t < nvt) {
        o[t] *= alpha;
        o[t] = mm_pv<DT>(vf[t], pf, o[t]);
      }
    if constexpr (kPrefetch) { if (kn < klim) load_vs(kn); }
  }

  // merge of the waves
  l = group_sum(l);
  if (g == 0) { red_m[wave][l15] = m; red_l[wave][l15] = l; }
#pragma unroll
  for (int t = 0; t < NVT; ++t)
    if (EXACT || t < nvt)
#pragma unroll
      for (int e = 0; e < 4; ++e) red_o[wave][l15][16 * t + 4 * g + e] = o[t][e];
  __syncthreads();
  const long long pstride = 16ll * (DVP + 2);
  float* part = a.part + ((long long)b * ngt + gt) * a.nsplit * pstride;
  E* out = reinterpret_cast<E*>(a.out) + (long long)b * a.ldo + (long long)(hk * R + r0) * a.vdim;
  auto finish = [&](int i, float num, float den) {  // i = r vdim + d: heads are contiguous
    float y = num / den;
    if (a.gated)
      y *= sigmoid32(i < 64 * NW ? gpre[0] : i < 128 * NW ? gpre[1] : gate[i]);
    out[i] = St<DT>::st(y);
  };
  for (int i = tid; i < nr * a.vdim; i += 64 * NW) {
    const int r = i / a.vdim, d = i - r * a.vdim;
    float M = red_m[0][r];
#pragma unroll
    for (int w = 1; w < NW; ++w) M = fmaxf(M, red_m[w][r]);
    if (nact == 1 && a.sink) M = fmaxf(M, 0.f);
    float num = 0.f, den = nact == 1 && a.sink ? __builtin_amdgcn_exp2f(-M) : 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = __builtin_amdgcn_exp2f(red_m[w][r] - M);
      num = fmaf(f, red_o[w][r][d], num);
      den = fmaf(f, red_l[w][r], den);
    }
    if (nact == 1) {
      finish(i, num, den);
    } else {
      float* pr = part + sp * pstride + (long long)r * (DVP + 2);
      // agent-scope stores: the merging workgroup may run on another XCD
      __hip_atomic_store(pr + 2 + d, num, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (d == 0) {
        __hip_atomic_store(pr, M, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(pr + 1, den, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (nact == 1) return;
  // the last split to arrive merges all of them: every wave's partials are out before the
  // workgroup's arrival counts, and both sides use agent-scope accesses
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    unsigned int* tk = a.ticket + (long long)b * ngt + gt;
    const unsigned int old =
        __hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = old == (unsigned int)(nact - 1);
    if (s_last) __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!s_last) return;
  float* wm = &red_o[0][0][0];      // [nact][16] max -> weight; the wave partials are spent
  float* wl = wm + 16 * 64;         // [nact][16] sums
  float* wd = &red_m[0][0];         // [16] denominators
  static_assert(sizeof(red_o) >= 2 * 16 * 64 * sizeof(float), "merge scratch");
  for (int i = tid; i < nr * nact; i += 64 * NW) {
    const int s = i / nr, r = i - s * nr;
    const float* pr = part + s * pstride + (long long)r * (DVP + 2);
    wm[s * 16 + r] = __hip_atomic_load(pr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    wl[s * 16 + r] = __hip_atomic_load(pr + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (tid < nr) {
    float M = a.sink ? 0.f : -INFINITY;
    for (int s = 0; s < nact; ++s) M = fmaxf(M, wm[s * 16 + tid]);
    float den = a.sink ? __builtin_amdgcn_exp2f(-M) : 0.f;
    for (int s = 0; s < nact; ++s) {
      const float f = __builtin_amdgcn_exp2f(wm[s * 16 + tid] - M);
      den = fmaf(f, wl[s * 16 + tid], den);
      wm[s * 16 + tid] = f;
    }
    wd[tid] = den;
  }
  __syncthreads();
  for (int i = tid; i < nr * a.vdim; i += 64 * NW) {
    const int r = i / a.vdim, d = i - r * a.vdim;
    const float* pr = part + (long long)r * (DVP + 2) + 2 + d;
    float num = 0.f;
    for (int s0 = 0; s0 < nact; s0 += 8) {  // eight partials in flight
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        v[j] = __hip_atomic_load(pr + min(s0 + j, nact - 1) * pstride, __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < nact) num = fmaf(wm[(s0 + j) * 16 + r], v[j], num);
    }
    finish(i, num, wd[r]);
  }
}

static inline bool mix_shape_ok(int H, int G, int dim, int vdim, int DP, int DVP, int S, int rd2) {
  return H > 0 && G > 0 && H % G == 0 && dim > 0 && vdim > 0 && DP >= dim && DP % 32 == 0 &&
         DP <= 256 && DVP >= vdim && DVP % 16 == 0 && DVP <= 256 && S > 0 && S % 64 == 0 &&
         rd2 >= 0 && 2 * rd2 <= dim;
}

// key splits of a decode launch over so many (query tile, row) pairs: no more workgroups than units
static inline int mix_dec_splits(long long groups, int nsplit) {
  while (nsplit > 1 && groups * nsplit > 256) nsplit /= 2;
  return nsplit;
}

}  // namespace cake
