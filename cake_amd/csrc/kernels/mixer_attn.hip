// Softmax attention of the hybrid designs: separate query/key and value head sizes,
// interleaved partial rotary positions, RMS-normalised queries and keys, an optional sink
// (one extra exp(0) in the denominator) and an optional sigmoid output gate.
//
// Cache of one layer run: K [slot][G][S][DP] row-major and V TRANSPOSED [slot][G][DVP][S]
// (DP = key size padded to 32, DVP = value size padded to 16, zero-filled): both products
// of both kernels then take 16-byte / 8-byte pieces of contiguous memory as their MFMA
// operands, and no kernel transposes values in LDS.
//
//   * mixer_prep: prompt rows — rotation + norm of q and k, cache write.
//   * mixer_flash (mixer_flash.h): prompt attention over a ragged batch.
//   * mixer_attn_decode: one token per sequence — rotation, norm and cache write of the new
//     key/value in the prologue, K / V^T streamed straight from memory into MFMA operands,
//     split over the keys with an in-launch merge, gate in the epilogue.
#include "mixer_flash.h"

namespace cake {

// ---------------------------------------------------------------------------
// prompt rows: q, k -> rotated, normalised
// ---------------------------------------------------------------------------
struct PrepArgs {
  const void* proj;      // [N][ldp] q | k | v | ... columns
  long long ldp;
  int N, H, G, dim, vdim, DP, DVP, S, rd2;  // rd2 = rotated pairs
  int h0;                // the first head taken: 0, or H for the keys alone
  int qk_norm;
  float eps;
  const float2* cs;      // [positions][rd2] (cos, sin)
  const int* row_pos;    // [N]
  const int* row_slot;   // [N]
  void* qn;              // [N][H][DP]
  void* kc;              // layer run's K cache
  void* vc;              // layer run's V^T cache
  long long k_slot, v_slot;  // elements per slot
};

// sum over aligned groups of `lph` lanes (a power of two): DPP inside 16-lane rows, lane swaps
// across them
__device__ __forceinline__ float lanes_sum(float v, int lph) {
  if (lph >= 2) v += dpp_f<kDppXor1>(v);
  if (lph >= 4) v += dpp_f<kDppXor2>(v);
  if (lph >= 8) v += dpp_f<kDppHalfMirror>(v);
  if (lph >= 16) v += dpp_f<kDppMirror>(v);
  if (lph >= 32) v = xor_add<16>(v);
  if (lph >= 64) v = xor_add<32>(v);
  return v;
}

// values -> V^T: a wave takes 64 rows x 8 dims, so its stores run along the positions
template <int DT>
__device__ __forceinline__ void prep_v(const PrepArgs& a, int block) {
  using E = typename St<DT>::E;
  const int nrt = (a.N + 63) / 64, rt = block % nrt;
  const int n = rt * 64 + (threadIdx.x & 63);
  const int nch = (a.vdim + 7) / 8;
  const int c = (block / nrt) * 4 + (threadIdx.x >> 6);
  if (n >= a.N || c >= a.G * nch) return;
  const int gh = c / nch, d0 = (c - gh * nch) * 8;
  const E* src = reinterpret_cast<const E*>(a.proj) + (long long)n * a.ldp +
                 (long long)(a.H + a.G) * a.dim + (long long)gh * a.vdim + d0;
  E* dst = reinterpret_cast<E*>(a.vc) + a.row_slot[n] * a.v_slot +
           ((long long)gh * a.DVP + d0) * a.S + a.row_pos[n];
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (d0 + e < a.vdim) dst[(long long)e * a.S] = src[e];
}

// Blocks [0, nvb) move the values; the others take queries and keys:
// lph lanes per (row, head), EPL consecutive dims each.  VEC: rows and heads on 2 EPL-byte
// boundaries and dim % EPL == 0 (16-bit types).
template <int DT, int EPL, bool VEC>
__global__ __launch_bounds__(256) void mixer_prep_kernel(PrepArgs a, int lph, int nvb) {
  using E = typename St<DT>::E;
  if ((int)blockIdx.x < nvb) { prep_v<DT>(a, blockIdx.x); return; }
  const int per = 256 / lph;  // (row, head) items per workgroup
  const int item = (blockIdx.x - nvb) * per + threadIdx.x / lph;
  const int l = threadIdx.x % lph, d0 = EPL * l;
  const int nh = a.H + a.G - a.h0;
  const bool live = item < a.N * nh;  // lanes past the end shadow the last item
  const int it = live ? item : a.N * nh - 1;
  const int n = it / nh, hh = it - n * nh + a.h0;
  const bool isq = hh < a.H;
  const int pos = a.row_pos[n];
  const E* src = reinterpret_cast<const E*>(a.proj) + (long long)n * a.ldp + (long long)hh * a.dim;
  float x[EPL];
  if constexpr (VEC && EPL == 8) {
    unpack8<DT == kF32 ? kBF16 : DT>(d0 < a.dim ? *reinterpret_cast<const uint4*>(src + d0)
                                                : make_uint4(0u, 0u, 0u, 0u), x);
  } else {
#pragma unroll
    for (int e = 0; e < EPL; ++e) x[e] = d0 + e < a.dim ? St<DT>::ld(src[d0 + e]) : 0.f;
  }
  const float2* cs = a.cs + (long long)pos * a.rd2;
#pragma unroll
  for (int p = 0; p < EPL / 2; ++p) {
    const int i = EPL / 2 * l + p;
    if (i < a.rd2) {
      const float2 t = cs[i];
      const float u = x[2 * p], v = x[2 * p + 1];
      x[2 * p] = u * t.x - v * t.y;
      x[2 * p + 1] = v * t.x + u * t.y;
    }
  }
  if (a.qk_norm) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < EPL; ++e) ss += x[e] * x[e];
    const float r = 1.f / sqrtf(lanes_sum(ss, lph) / (float)a.dim + a.eps);
#pragma unroll
    for (int e = 0; e < EPL; ++e) x[e] *= r;
  }
  E* dst = isq ? reinterpret_cast<E*>(a.qn) + ((long long)n * a.H + hh) * a.DP
               : reinterpret_cast<E*>(a.kc) + a.row_slot[n] * a.k_slot +
                     ((long long)(hh - a.H) * a.S + pos) * a.DP;
  if (!live || d0 >= a.DP) return;  // DP % 8 == 0; columns past dim carry zeros
  if constexpr (DT == kF32) {
#pragma unroll
    for (int e = 0; e < EPL; e += 4)
      *reinterpret_cast<float4*>(dst + d0 + e) = make_float4(x[e], x[e + 1], x[e + 2], x[e + 3]);
  } else {
    uint32_t w[EPL / 2];
#pragma unroll
    for (int e = 0; e < EPL / 2; ++e)
      w[e] = (uint32_t)St<DT>::st(x[2 * e]) | ((uint32_t)St<DT>::st(x[2 * e + 1]) << 16);
    *reinterpret_cast<uint4*>(dst + d0) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

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

template <int DT, int CLS, bool EXACT, int NW>
__global__ __launch_bounds__(64 * NW) void mixer_attn_decode_kernel(MixDecArgs a) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC;
  constexpr int NKS = CLS / St<DT>::KSTEP, NVT = CLS / 16;
  constexpr bool kPrefetch = DT != kF32 && CLS <= 128;
  const int DP = EXACT ? CLS : a.DP, DVP = EXACT ? CLS : a.DVP;
  const int nks = EXACT ? NKS : DP / St<DT>::KSTEP, nvt = EXACT ? NVT : DVP / 16;
  __shared__ __attribute__((aligned(16))) E qs[16 * (CLS + EPC)];
  __shared__ __attribute__((aligned(16))) E kcur[CLS];
  __shared__ __attribute__((aligned(16))) E vcur[CLS];
  __shared__ float red_m[NW][16], red_l[NW][16];
  __shared__ float red_o[NW][16][CLS + 1];
  __shared__ int s_last;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int R = a.H / a.G, npg = (R + 15) / 16;      // 16-row query tiles per kv head
  const int gt = blockIdx.x, hk = gt / npg, r0 = (gt - hk * npg) * 16;
  const int nr = min(16, R - r0);
  const int sp = blockIdx.y, b = blockIdx.z;
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
  const int ngt = gridDim.x;
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

}  // namespace cake

using namespace cake;

static bool mix_shape_ok(int H, int G, int dim, int vdim, int DP, int DVP, int S, int rd2) {
  return H > 0 && G > 0 && H % G == 0 && dim > 0 && vdim > 0 && DP >= dim && DP % 32 == 0 &&
         DP <= 256 && DVP >= vdim && DVP % 16 == 0 && DVP <= 256 && S > 0 && S % 64 == 0 &&
         rd2 >= 0 && 2 * rd2 <= dim;
}

// (qn null: keys and values alone)
CAKE_API int cake_mixer_prep(int dt, const void* proj, long long ldp, int N, int H, int G, int dim,
                             int vdim, int DP, int DVP, int S, int rd2, int qk_norm, float eps,
                             const void* cs, const int* row_pos, const int* row_slot, void* qn,
                             void* kc, void* vc, long long k_slot, long long v_slot,
                             hipStream_t st) {
  if (!mix_shape_ok(H, G, dim, vdim, DP, DVP, S, rd2) || N < 0) return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  const int h0 = qn ? 0 : H;
  PrepArgs a{proj, ldp, N, H, G, dim, vdim, DP, DVP, S, rd2, h0, qk_norm, eps, (const float2*)cs,
             row_pos, row_slot, qn, kc, vc, k_slot, v_slot};
  int lph = 4;
  while (8 * lph < DP) lph <<= 1;  // <= 32
  const bool vec = dt != kF32 && dim % 8 == 0 && ldp % 8 == 0 && ((uintptr_t)proj % 16) == 0;
  const long long items = (long long)N * (H + G - h0);
  const int nvb = ((N + 63) / 64) * ((G * ((vdim + 7) / 8) + 3) / 4);
  const dim3 g((unsigned)(nvb + (items + 256 / lph - 1) / (256 / lph)));
  CAKE_MIX_DT(dt, {
    if (vec) hipLaunchKernelGGL((mixer_prep_kernel<DT, 8, true>), g, dim3(256), 0, st, a, lph, nvb);
    else hipLaunchKernelGGL((mixer_prep_kernel<DT, 8, false>), g, dim3(256), 0, st, a, lph, nvb);
  });
  return (int)hipGetLastError();
}

template <int DT, int CLS, bool EXACT>
static int launch_flash_cls(const MixFlashArgs& a, dim3 grid, hipStream_t st) {
  return launch_mix_flash<DT, CLS, CLS, EXACT, false>(a, grid, st);
}

#define CAKE_MIX_CLS(FN, ...)                                                            \
  do {                                                                                   \
    const int cls = DP > DVP ? DP : DVP;                                                 \
    if (cls <= 64) return DP == 64 && DVP == 64 ? FN<DT, 64, true>(__VA_ARGS__)          \
                                                : FN<DT, 64, false>(__VA_ARGS__);        \
    if (cls <= 128) return DP == 128 && DVP == 128 ? FN<DT, 128, true>(__VA_ARGS__)      \
                                                   : FN<DT, 128, false>(__VA_ARGS__);    \
    return FN<DT, 256, false>(__VA_ARGS__);                                              \
  } while (0)

CAKE_API int cake_mixer_flash(int dt, const void* qn, const void* kc, const void* vc,
                              long long k_slot, long long v_slot, const void* seq, int B,
                              int max_len, const void* gate, long long ldg, void* out,
                              long long ldo, int H, int G, int dim, int vdim, int DP, int DVP,
                              int S, int sink, float scale, hipStream_t st) {
  if (!mix_shape_ok(H, G, dim, vdim, DP, DVP, S, 0) || B <= 0 || max_len <= 0)
    return (int)hipErrorInvalidValue;
  MixFlashArgs a{qn, kc, vc, k_slot, v_slot, (const SeqRow*)seq, gate, ldg, out, ldo,
                 H, G, DP, DVP, vdim, S, sink, scale * 1.4426950408889634f, {}};
  if (flash3_ok(dt, a, false, S, max_len, B))
    return dt == kBF16 ? launch_mix_flash3<kBF16, false>(a, max_len, B, st)
                       : launch_mix_flash3<kF16, false>(a, max_len, B, st);
  const dim3 grid((max_len + 127) / 128, H, B);
  CAKE_MIX_DT(dt, CAKE_MIX_CLS(launch_flash_cls, a, grid, st));
  return (int)hipErrorInvalidValue;
}

// Few keys: one workgroup's chain of loads (position, projections, keys, merge), so eight waves take
// 256 keys in one pass of 32 each (16 heads over 4, 256 keys, 10.6 us with four waves, 8.4).  Key
// splits only as far as the batch leaves compute units idle: 24 sequences of 8 key heads in 8 splits
// took 27 us at 300 keys and 44.5 at 1000, unsplit 10.3 and 20.3 (2000 keys 56 / 38, 4000 102 / 85);
// one sequence 1000 keys 10.4 in 8 splits, 18.2 unsplit.
template <int DT, int CLS, bool EXACT>
static int launch_mix_dec(MixDecArgs a, dim3 grid, hipStream_t st) {
  while (a.nsplit > 1 && (long long)grid.x * grid.z * a.nsplit > 256) a.nsplit /= 2;
  grid.y = a.nsplit;
  if constexpr (DT != kF32 && CLS <= 128) {
    if (a.nsplit == 1) {
      hipLaunchKernelGGL((mixer_attn_decode_kernel<DT, CLS, EXACT, 8>), grid, dim3(512), 0, st, a);
      return (int)hipGetLastError();
    }
  }
  hipLaunchKernelGGL((mixer_attn_decode_kernel<DT, CLS, EXACT, 4>), grid, dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

// f32 elements of `part` / u32 elements of `ticket` (zeroed once) for a launch
CAKE_API long long cake_mixer_attn_part(int B, int H, int G, int DVP, int nsplit) {
  const long long ngt = (long long)G * ((H / G + 15) / 16);
  return (long long)B * ngt * nsplit * 16 * (DVP + 2);
}

CAKE_API int cake_mixer_attn_decode(int dt, const float* proj, long long ldp, int B, const int* pos,
                                    const int* slot, const void* cs, int rd2, int qk_norm,
                                    int sink, int gated, float eps, float scale, void* kc, void* vc,
                                    long long k_slot, long long v_slot, void* out, long long ldo,
                                    int H, int G, int dim, int vdim, int DP, int DVP, int S,
                                    int nsplit, float* part, unsigned int* ticket, hipStream_t st) {
  if (!mix_shape_ok(H, G, dim, vdim, DP, DVP, S, rd2) || B <= 0 || nsplit < 1 || nsplit > 64)
    return (int)hipErrorInvalidValue;
  MixDecArgs a{proj, ldp, pos, slot, (const float2*)cs, rd2, qk_norm, sink, gated, eps,
               scale * 1.4426950408889634f, kc, vc, k_slot, v_slot, out, ldo, H, G, dim, vdim,
               DP, DVP, S, nsplit, part, ticket};
  const dim3 grid(G * ((H / G + 15) / 16), nsplit, B);
  CAKE_MIX_DT(dt, CAKE_MIX_CLS(launch_mix_dec, a, grid, st));
  return (int)hipErrorInvalidValue;
}
