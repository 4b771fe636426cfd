// Prompt attention of the hybrid designs over a ragged batch: S^T = K Q^T and O^T += V^T P^T (an
// accumulator of the first is the B operand of the second), 4 waves x 32 query rows, key tiles
// staged in LDS (next tile's loads in flight behind the MFMAs), gate and head concatenation in
// the epilogue.  Keys and values come from the cache (mixer_attn.hip) or, for latent attention
// (mixer_latent.hip), from the step's expansion of the latent, with the rotated key part read
// from the latent cache.
#pragma once
#include "flash3.h"
#include "mixer_common.h"

namespace cake {

// the interleaved rotation of one 16-byte piece: pairs i0 .. of the position's (cos, sin) row
template <int DT>
__device__ __forceinline__ void rotate_piece(uint4& w, const float2* cs, int i0, int rd2) {
  uint32_t v[4] = {w.x, w.y, w.z, w.w};
  if constexpr (DT == kF32) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
      if (i0 + e < rd2) {
        const float2 t = cs[i0 + e];
        const float a = __uint_as_float(v[2 * e]), b = __uint_as_float(v[2 * e + 1]);
        v[2 * e] = __float_as_uint(a * t.x - b * t.y);
        v[2 * e + 1] = __float_as_uint(b * t.x + a * t.y);
      }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (i0 + e < rd2) {
        const float2 t = cs[i0 + e];
        const float a = to_f32<DT>((uint16_t)(v[e] & 0xffffu)), b = to_f32<DT>((uint16_t)(v[e] >> 16));
        v[e] = (uint32_t)from_f32<DT>(a * t.x - b * t.y) |
               ((uint32_t)from_f32<DT>(b * t.x + a * t.y) << 16);
      }
  }
  w = make_uint4(v[0], v[1], v[2], v[3]);
}

// ---------------------------------------------------------------------------
// prompt attention
// ---------------------------------------------------------------------------
// Latent form: per-head keys and values of the step's own expansion, one rotated key part shared
// by the heads, queries rotated here.
struct LatentSrc {
  const int* koff;       // [B] first key row / value column of each sequence (multiples of 64)
  const void* rope;      // rotated key part [slot][position][ldr]
  long long rope_slot;
  int ldr;
  int dimp, rotp;        // unrotated / rotated columns of a head (multiples of 8)
  long long ldq, ldk, ldv;  // row strides of queries [N], keys [rows] and values [H DVP]
  const float2* cs;      // [positions][rd2]
  int rd2;
};

struct MixFlashArgs {
  const void* qn;        // [N][H][DP]; latent: [N][ldq], head h at h (dimp + rotp)
  const void* kc;        // latent: [key rows][ldk], head h at h dimp
  const void* vc;        // latent: [H DVP][ldv]
  long long k_slot, v_slot;
  const SeqRow* seq;     // [B]
  const void* gate;      // [N][ldg] + column 0 of the gate (null: no gate)
  long long ldg;
  void* out;             // [N][ldo]
  long long ldo;
  int H, G, DP, DVP, vdim, S, sink;
  float scale_log2;
  LatentSrc lat;
};

// KC / VC: classes of the key and value sizes (EXACT: the sizes themselves)
template <int DT, int KC> struct FlashGeo {
  // keys per tile: 32 where 64 would spill the prefetched pieces
  static constexpr int BN = DT == kF32 || KC == 192 ? 32 : 64;
  static constexpr int NBUF = KC <= 128 ? 2 : 1;     // LDS buffers
  static constexpr int WGS = KC <= 192 && (KC <= 128 || DT != kF32) ? 2 : 1;  // per CU
};

template <int DT, int KC, int VC, bool EXACT, bool LAT>
__global__ __launch_bounds__(256, (FlashGeo<DT, KC>::WGS)) void mixer_flash_kernel(MixFlashArgs a) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC;
  constexpr int NKS = KC / St<DT>::KSTEP, NVT = VC / 16;
  constexpr int BN = FlashGeo<DT, KC>::BN, NB = BN / 16;  // keys, 16-key blocks per tile
  constexpr int NPK = KC * BN / EPC / 256, NPV = VC * BN / EPC / 256;  // pieces per thread, K, V
  constexpr int NBUF = FlashGeo<DT, KC>::NBUF;
  constexpr int VLD = BN + EPC;                            // V^T row stride in LDS
  constexpr int VPR = BN / EPC;                            // pieces per V^T row
  extern __shared__ __attribute__((aligned(16))) unsigned char mixer_smem[];
  E* const sm = reinterpret_cast<E*>(mixer_smem);
  const int DP = EXACT ? KC : a.DP, DVP = EXACT ? VC : a.DVP;
  const int KLD = DP + EPC;                                // +16 bytes: no bank conflicts
  const int KPR = DP / EPC;
  const int bufe = BN * KLD + DVP * VLD;
  const int nks = EXACT ? NKS : DP / St<DT>::KSTEP, nvt = EXACT ? NVT : DVP / 16;

  const SeqRow sq = a.seq[blockIdx.z];
  const int nqt = (sq.len + 127) / 128;
  if ((int)blockIdx.x >= nqt) return;
  const int m0 = (nqt - 1 - (int)blockIdx.x) * 128;  // the longest rows first
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int h = blockIdx.y, hk = h / (a.H / a.G);
  const E *kb, *vb, *rb = nullptr;
  long long ldv = a.S;
  int npc = 0, qpc = 0;  // latent: pieces of the unrotated part, of a whole head
  if constexpr (LAT) {
    const int k0 = a.lat.koff[blockIdx.z];
    kb = reinterpret_cast<const E*>(a.kc) + k0 * a.lat.ldk + (long long)h * a.lat.dimp;
    vb = reinterpret_cast<const E*>(a.vc) + (long long)h * a.DVP * a.lat.ldv + k0;
    rb = reinterpret_cast<const E*>(a.lat.rope) + sq.slot * a.lat.rope_slot;
    ldv = a.lat.ldv;
    npc = a.lat.dimp / EPC;
    qpc = npc + a.lat.rotp / EPC;
  } else {
    kb = reinterpret_cast<const E*>(a.kc) + sq.slot * a.k_slot + (long long)hk * a.S * a.DP;
    vb = reinterpret_cast<const E*>(a.vc) + sq.slot * a.v_slot + (long long)hk * a.DVP * a.S;
  }
  const int qw = m0 + wave * 32;  // this wave's first row

  uint4 qf[2][NKS];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = min(qw + 16 * j + l15, sq.len - 1);
    if constexpr (LAT) {
      const E* qp = reinterpret_cast<const E*>(a.qn) + (sq.row0 + row) * a.lat.ldq +
                    (long long)h * (a.lat.dimp + a.lat.rotp);
      const float2* cs = a.lat.cs + (long long)(sq.pos0 + row) * a.lat.rd2;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) {
        const int p = ks * 4 + g;
        qf[j][ks] = p < qpc ? *reinterpret_cast<const uint4*>(qp + p * EPC) : make_uint4(0, 0, 0, 0);
        if (p >= npc && p < qpc) rotate_piece<DT>(qf[j][ks], cs, (p - npc) * (EPC / 2), a.lat.rd2);
      }
    } else {
      const E* qp = reinterpret_cast<const E*>(a.qn) + ((long long)(sq.row0 + row) * a.H + h) * DP;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        qf[j][ks] = (EXACT || ks < nks) ? *reinterpret_cast<const uint4*>(qp + (ks * 4 + g) * EPC)
                                        : make_uint4(0, 0, 0, 0);
    }
  }
  cf32x4 o[2][NVT];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int t = 0; t < NVT; ++t) o[j][t] = cf32x4{0.f, 0.f, 0.f, 0.f};
  // running max (log2 units) and lane-partial sum; the sink is a key of score 0 without value
  float m[2], l[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    m[j] = a.sink ? 0.f : -INFINITY;
    l[j] = a.sink && g == 0 ? 1.f : 0.f;
  }
  const int kend = min(sq.pos0 + sq.len, sq.pos0 + m0 + 128);
  const int ntiles = (kend + BN - 1) / BN;
  const int qmin = sq.pos0 + qw, qmax = qmin + 31;

  u32x4 kr[NPK], vr[NPV];
  auto gload = [&](int j) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NPK; ++i) {
      const int p = tid + 256 * i;
      if (EXACT || p < BN * KPR) {
        if constexpr (LAT) {
          const int r = p / KPR, c = p - r * KPR;
          const E* src = c < npc ? kb + (long long)(j * BN + r) * a.lat.ldk + c * EPC
                                 : rb + (long long)(j * BN + r) * a.lat.ldr + (c - npc) * EPC;
          kr[i] = c < qpc ? *reinterpret_cast<const u32x4*>(src) : u32x4{0u, 0u, 0u, 0u};
        } else {
          kr[i] = *reinterpret_cast<const u32x4*>(kb + (long long)j * BN * DP + (long long)p * EPC);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NPV; ++i) {
      const int p = tid + 256 * i;
      if (EXACT || p < DVP * VPR) {
        const int r = p / VPR, c = p - r * VPR;
        vr[i] = *reinterpret_cast<const u32x4*>(vb + (long long)r * ldv + j * BN + c * EPC);
      }
    }
  };
  auto sstore = [&](int buf) __attribute__((always_inline)) {
    E* Ks = sm + buf * bufe;
    E* Vs = Ks + BN * KLD;
#pragma unroll
    for (int i = 0; i < NPK; ++i) {
      const int p = tid + 256 * i;
      if (EXACT || p < BN * KPR) {
        const int r = p / KPR, c = p - r * KPR;
        *reinterpret_cast<u32x4*>(Ks + r * KLD + c * EPC) = kr[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NPV; ++i) {
      const int p = tid + 256 * i;
      if (EXACT || p < DVP * VPR) {
        const int r = p / VPR, c = p - r * VPR;
        *reinterpret_cast<u32x4*>(Vs + r * VLD + c * EPC) = vr[i];
      }
    }
  };

  gload(0);
  sstore(0);
  __syncthreads();
  for (int j = 0; j < ntiles; ++j) {
    const int buf = NBUF == 2 ? (j & 1) : 0;
    const bool more = j + 1 < ntiles;
    const E* Ks = sm + buf * bufe;
    const E* Vs = Ks + BN * KLD;
    const int k0 = j * BN;
    const bool active = k0 <= qmax;  // wave-uniform: some row of this wave sees the tile
    cf32x4 s[2][NB];
    if (active) {
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        s[0][b] = cf32x4{0.f, 0.f, 0.f, 0.f};
        s[1][b] = cf32x4{0.f, 0.f, 0.f, 0.f};
        const E* krow = Ks + (16 * b + l15) * KLD + g * EPC;
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) {
          if (EXACT || ks < nks) {
            const uint4 kf = *reinterpret_cast<const uint4*>(krow + ks * 4 * EPC);
            s[0][b] = mm_piece<DT>(kf, qf[0][ks], s[0][b]);
            s[1][b] = mm_piece<DT>(kf, qf[1][ks], s[1][b]);
          }
        }
      }
    }
    if (more) gload(j + 1);  // behind the QK products, in flight over the rest of the tile
    if (active) {
      const bool edge = k0 + BN - 1 > qmin;
      PFrag<DT> pf[2][NB / 2];
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        if (edge) {
          const int qpos = qmin + 16 * q + l15;
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (k0 + 16 * b + 4 * g + e > qpos) s[q][b][e] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) mx = fmaxf(mx, s[q][b][e]);
        mx = group_max(mx) * a.scale_log2;
        if (a.scale_log2 < 0.f) {  // a negative scale turns the order round
          float mn = INFINITY;
#pragma unroll
          for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (s[q][b][e] != -INFINITY) mn = fminf(mn, s[q][b][e]);
          mx = group_max(mn == INFINITY ? -INFINITY : mn * a.scale_log2);
        }
        const bool grow = mx > m[q];
        if (__builtin_amdgcn_ballot_w64(grow) != 0ull) {
          const float mn = fmaxf(m[q], mx);
          const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m[q] - mn);
          m[q] = mn;
          l[q] *= alpha;
#pragma unroll
          for (int t = 0; t < NVT; ++t)
            if (EXACT || t < nvt) o[q][t] *= alpha;
        }
        const float mc = m[q] == -INFINITY ? 0.f : m[q];
        float rs = 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float raw = s[q][b][e];
            const float p = raw == -INFINITY ? 0.f
                                             : __builtin_amdgcn_exp2f(fmaf(raw, a.scale_log2, -mc));
            s[q][b][e] = p;
            rs += p;
          }
        l[q] += rs;
#pragma unroll
        for (int b = 0; b < NB / 2; ++b) pf[q][b] = pack_p<DT>(s[q][2 * b], s[q][2 * b + 1]);
      }
#pragma unroll
      for (int b = 0; b < NB / 2; ++b)
#pragma unroll
        for (int t = 0; t < NVT; ++t)
          if (EXACT || t < nvt) {
            const VFrag<DT> vf = load_v<DT>(Vs + (16 * t + l15) * VLD + 32 * b, g);
            o[0][t] = mm_pv<DT>(vf, pf[0][b], o[0][t]);
            o[1][t] = mm_pv<DT>(vf, pf[1][b], o[1][t]);
          }
    }
    if (NBUF == 1) __syncthreads();  // every wave is past the tile before it is replaced
    if (more) sstore(NBUF == 2 ? buf ^ 1 : 0);
    __syncthreads();
  }

  // epilogue: lane (l15, g) holds O^T[16 t + 4 g + e][row l15]
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int row = qw + 16 * j + l15;
    const float lt = group_sum(l[j]);
    if (row >= sq.len) continue;
    const float inv = 1.f / lt;
    const long long n = sq.row0 + row;
    E* op = reinterpret_cast<E*>(a.out) + n * a.ldo + (long long)h * a.vdim;
    const E* gp = a.gate ? reinterpret_cast<const E*>(a.gate) + n * a.ldg + (long long)h * a.vdim
                         : nullptr;
#pragma unroll
    for (int t = 0; t < NVT; ++t)
      if (EXACT || t < nvt) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = 16 * t + 4 * g + e;
          if (d < a.vdim) {
            float y = o[j][t][e] * inv;
            if (gp) y *= sigmoid32(St<DT>::ld(gp[d]));
            op[d] = St<DT>::st(y);
          }
        }
      }
  }
}

// 16-bit types, keys of 128 columns (LAT: 128 and 64 rotated) and values of 128, on the shared
// core (flash3.h), 128 rows a workgroup, the maximum exact as in the kernel above.  Error against 64
// bits as there, 0.00210 at 2048 rows; latent 0.00203 / 0.00202 (that kernel's tiles are of 32 keys:
// twice as many find a new maximum, whose probability, 1, is not rounded).
// 32 heads over 8, us before / after: 300 rows 26.5 / 14.2, 1100 64 / 34,
// 2048 110 / 65, 24 sequences of 60 47 / 32; latent 300 27 / 16, 1100 85 / 36, 2048 154 / 71.  (64
// rows a wave: 1.05 - 1.15x faster from 3000 rows on with a deferred maximum, slower below.)
template <int DT, bool LAT>
__global__ __launch_bounds__(256, 1) void mixer_flash3_kernel(MixFlashArgs a) {
  constexpr int QS = 1, KC = LAT ? 192 : 128, KS = KC / 16;
  __shared__ __attribute__((aligned(16))) uint8_t smem[fl_lds<KC>()];
  const SeqRow sq = a.seq[blockIdx.z];
  const int nqt = (sq.len + 128 * QS - 1) / (128 * QS);
  if ((int)blockIdx.y >= nqt) return;
  const int lane = threadIdx.x & 63, l32 = lane & 31, hh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // the query heads of one key head to one XCD (8 key heads), the longest rows first
  const int x = blockIdx.x, hk = LAT ? x : x % a.G, h = LAT ? x : hk * (a.H / a.G) + x / a.G;
  const int m0 = (nqt - 1 - (int)blockIdx.y) * (128 * QS), qw = m0 + wave * (32 * QS);

  fu32x4 qf[QS][KS];
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    const int row = min(qw + 32 * qs + l32, sq.len - 1);
    const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.qn) +
        (LAT ? (sq.row0 + row) * a.lat.ldq + (long long)h * KC
             : ((long long)(sq.row0 + row) * a.H + h) * KC);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      uint4 w = *reinterpret_cast<const uint4*>(qp + (2 * ks + hh) * 8);
      if (ks >= 8)
        rotate_piece<DT>(w, a.lat.cs + (long long)(sq.pos0 + row) * a.lat.rd2,
                         (2 * (ks - 8) + hh) * 4, a.lat.rd2);
      qf[qs][ks] = __builtin_bit_cast(fu32x4, w);
    }
  }
  FlCore c{};
  c.kend = sq.pos0 + min(sq.len, m0 + 128 * QS);
  c.pos = sq.pos0 + qw;
  c.scale_log2 = a.scale_log2;
  c.sink = a.sink != 0;
  const uint16_t *kc = reinterpret_cast<const uint16_t*>(a.kc),
                 *vc = reinterpret_cast<const uint16_t*>(a.vc);
  if constexpr (LAT) {
    const int k0 = a.lat.koff[blockIdx.z];
    c.k = kc + k0 * a.lat.ldk + (long long)h * 128;
    c.k_sn = a.lat.ldk;
    c.v = vc + (long long)h * 128 * a.lat.ldv + k0;
    c.v_sn = a.lat.ldv;
    c.v_end = (unsigned)((127 * a.lat.ldv + (c.kend + 63) / 64 * 64) * 2);
    c.r = reinterpret_cast<const uint16_t*>(a.lat.rope) + sq.slot * a.lat.rope_slot;
    c.r_sn = a.lat.ldr;
    c.r_end = (unsigned)(((c.kend - 1) * c.r_sn + 64) * 2);
  } else {
    c.k = kc + sq.slot * a.k_slot + (long long)hk * a.S * 128;
    c.k_sn = 128;
    c.v = vc + sq.slot * a.v_slot + (long long)hk * 128 * a.S;
    c.v_sn = a.S;
    c.v_end = (unsigned)(256 * a.S);
  }
  c.k_end = (unsigned)(((c.kend - 1) * c.k_sn + 128) * 2);
  ff32x16 o[QS][4];
  float l[QS];
  fl_core<DT, QS, KC, true, false>(smem, c, qf, o, l);

#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    const int row = qw + 32 * qs + l32;
    if (row >= sq.len) continue;
    const float inv = 1.f / l[qs];
    const long long n = sq.row0 + row;
    uint16_t* op = reinterpret_cast<uint16_t*>(a.out) + n * a.ldo + (long long)h * 128 + 4 * hh;
    const uint16_t* gp = LAT || !a.gate ? nullptr
        : reinterpret_cast<const uint16_t*>(a.gate) + n * a.ldg + (long long)h * 128 + 4 * hh;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = o[qs][t][4 * g + e] * inv;
        if (!LAT && gp) {
          const uint2 w = *reinterpret_cast<const uint2*>(gp + 32 * t + 8 * g);
          y[0] *= sigmoid32(to_f32<DT>((uint16_t)(w.x & 0xffffu)));
          y[1] *= sigmoid32(to_f32<DT>((uint16_t)(w.x >> 16)));
          y[2] *= sigmoid32(to_f32<DT>((uint16_t)(w.y & 0xffffu)));
          y[3] *= sigmoid32(to_f32<DT>((uint16_t)(w.y >> 16)));
        }
        *reinterpret_cast<uint2*>(op + 32 * t + 8 * g) =
            make_uint2(fl_cvt<DT>(y[0], y[1]), fl_cvt<DT>(y[2], y[3]));
      }
  }
}

// Whether mixer_flash3_kernel takes a call: its head sizes, a scale that keeps the order of the
// scores, 8-byte output and gate rows, a sequence's keys and values under 2 GB (rows: its most).
// Not many sequences of a few rows: one wave of four has work then, and of the kernel above several
// workgroups share a compute unit (us, this / the other: 24 sequences of 8 rows, 16 heads 9.2 / 7.9,
// 32 heads 13.6 / 12.7, latent 14.0 / 9.2 and 20.8 / 15.3; 60 of 20 17.7 / 20.0 and 34.7 / 37.0, latent
// 30.4 / 23.3 and 59 / 45; 40 of 33 14.4 / 17.4, latent 23.7 / 26.0; 8 of 20, 256 workgroups, latent
// 8.4 / 10.4).
inline bool flash3_ok(int dt, const MixFlashArgs& a, bool lat, long long rows, int max_len, int B) {
  if (max_len <= (lat ? 32 : 12) && (long long)a.H * B > 256) return false;
  const auto al = [](const void* p, long long ld) { return (uintptr_t)p % 8 == 0 && ld % 4 == 0; };
  const long long lim = 0x7fffffffLL / 2;   // elements; the tiles requested ahead: offsets of 32 bits
  const auto rows_fit = [&](long long ld) { return rows * ld < lim && (rows + 256) * ld < 2 * lim; };
  if ((dt != kBF16 && dt != kF16) || a.DVP != 128 || a.vdim != 128 || !(a.scale_log2 > 0.f) ||
      !al(a.out, a.ldo) || (a.gate && !al(a.gate, a.ldg)))
    return false;
  if (!lat) return a.DP == 128 && 128LL * a.S < lim;
  return a.DP == 192 && a.lat.dimp == 128 && a.lat.rotp == 64 && rows_fit(a.lat.ldk) &&
         rows_fit(a.lat.ldr) && 127 * a.lat.ldv + rows + 64 < lim;
}

template <int DT, bool LAT>
int launch_mix_flash3(const MixFlashArgs& a, int max_len, int B, hipStream_t st) {
  const dim3 grid(a.H, (max_len + 127) / 128, B);
  hipLaunchKernelGGL((mixer_flash3_kernel<DT, LAT>), grid, dim3(256), 0, st, a);
  return (int)hipGetLastError();
}

template <int DT, int KC, int VC, bool EXACT, bool LAT>
int launch_mix_flash(const MixFlashArgs& a, dim3 grid, hipStream_t st) {
  using G = FlashGeo<DT, KC>;
  constexpr int EPC = St<DT>::EPC;
  const size_t lds = (size_t)G::NBUF * (G::BN * (a.DP + EPC) + (size_t)a.DVP * (G::BN + EPC)) *
                     sizeof(typename St<DT>::E);
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)mixer_flash_kernel<DT, KC, VC, EXACT, LAT>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024) != hipSuccess)
      return (int)hipErrorInvalidValue;
    raised = true;
  }
  hipLaunchKernelGGL((mixer_flash_kernel<DT, KC, VC, EXACT, LAT>), grid, dim3(256), lds, st, a);
  return (int)hipGetLastError();
}

}  // namespace cake
