// Latent attention of the hybrid designs: queries through a latent of their own, keys and values
// expanded per head from one cached latent, and one rotated key part shared by all heads.
//
// Cache of one layer run: [slot][S][LD] rows [latent c (R, padded to RP) | rotated key | 0], LD a
// multiple of 32; nothing per head is cached.
//
//   * prompts expand the latent of the live positions with two plain products (keys row-major,
//     values transposed by exchanging the operands) and run mixer_flash (mixer_flash.h) on them;
//   * one token per sequence works on the latent itself: the query is carried into the latent
//     space (latent_absorb), all heads attend over the cached rows as they are (latent_decode;
//     16 heads share every tile, values are the same LDS rows read through the transposing LDS
//     load), and the value expansion merges the key splits in its prologue (latent_out).
#include "mixer_flash.h"

namespace cake {

struct LatentProj {      // f32 projections of a row: [q latent, QP | c, RP | key part, rotp]
  const float* proj;
  long long ldp;
  int QP, R, RP, rot, LD, rd2;
  float eps;
  const float* kv_norm;  // [RP], zeros past R
  const float2* cs;      // [positions][rd2]
  const int* pos;        // [rows]
  const int* slot;
  void* cache;
  long long slot_stride;
};

// Row n by a whole workgroup of 256 threads: the latent, normalised, and the rotated key part into
// the cache; with QUERY the normalised query latent into cq.  Norm weights are padded with zeros as
// the projected columns are; the columns of a cache row between its parts stay zero.
template <int DT, bool QUERY>
__device__ __forceinline__ void latent_row(const LatentProj& a, int n, int Q, const float* q_norm,
                                           typename St<DT>::E* cq, float* red) {
  using E = typename St<DT>::E;
  constexpr int NV = QUERY ? 4 : 1;  // 4096 / 1024 columns stay in registers
  const int QP = QUERY ? a.QP : 0, end = QP + a.RP, pos = a.pos[n], slot = a.slot[n];
  const float* src = a.proj + n * a.ldp + (a.QP - QP);
  const auto weight = [&](int i) __attribute__((always_inline)) {
    return *reinterpret_cast<const float4*>(QUERY && i < QP ? q_norm + i : a.kv_norm + (i - QP));
  };
  float4 v[NV], w[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = 4 * ((int)threadIdx.x + 256 * j);
    if (i < end) {
      v[j] = *reinterpret_cast<const float4*>(src + i);
      w[j] = weight(i);
    }
  }
  float sq = 0.f, sc = 0.f;
  const auto add = [&](int i, const float4& x) __attribute__((always_inline)) {
    const int left = (QUERY && i < QP ? Q : QP + a.R) - i;
    const float y = (left > 0 ? x.x * x.x : 0.f) + (left > 1 ? x.y * x.y : 0.f) +
                    (left > 2 ? x.z * x.z : 0.f) + (left > 3 ? x.w * x.w : 0.f);
    if (QUERY && i < QP) sq += y;
    else sc += y;
  };
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = 4 * ((int)threadIdx.x + 256 * j);
    if (i < end) add(i, v[j]);
  }
  for (int i = 4 * ((int)threadIdx.x + 256 * NV); i < end; i += 1024)
    add(i, *reinterpret_cast<const float4*>(src + i));
  if constexpr (QUERY) sq = wave_sum(sq);
  sc = wave_sum(sc);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[wave] = sq;
    red[4 + wave] = sc;
  }
  __syncthreads();
  const float rq = 1.f / sqrtf((red[0] + red[1] + (red[2] + red[3])) / (float)max(Q, 1) + a.eps);
  const float rc = 1.f / sqrtf((red[4] + red[5] + (red[6] + red[7])) / (float)a.R + a.eps);
  E* dst = reinterpret_cast<E*>(a.cache) + slot * a.slot_stride + (long long)pos * a.LD;
  const auto put = [&](int i, const float4& x, const float4& g) __attribute__((always_inline)) {
    const bool q = QUERY && i < QP;
    const float r = q ? rq : rc;
    const float y[4] = {x.x * r * g.x, x.y * r * g.y, x.z * r * g.z, x.w * r * g.w};
    E* o = q ? cq + i : dst + (i - QP);
    if constexpr (DT == kF32)
      *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
    else
      *reinterpret_cast<uint2*>(o) =
          make_uint2((uint32_t)St<DT>::st(y[0]) | ((uint32_t)St<DT>::st(y[1]) << 16),
                     (uint32_t)St<DT>::st(y[2]) | ((uint32_t)St<DT>::st(y[3]) << 16));
  };
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int i = 4 * ((int)threadIdx.x + 256 * j);
    if (i < end) put(i, v[j], w[j]);
  }
  for (int i = 4 * ((int)threadIdx.x + 256 * NV); i < end; i += 1024)
    put(i, *reinterpret_cast<const float4*>(src + i), weight(i));
  const float2* cs = a.cs + (long long)pos * a.rd2;
  for (int i = threadIdx.x; i < a.rot; i += 256) {
    float y = src[end + i];
    if (i < 2 * a.rd2) {
      const float2 t = cs[i >> 1];
      const float o = src[end + (i ^ 1)];
      y = (i & 1) ? y * t.x + o * t.y : y * t.x - o * t.y;
    }
    dst[a.RP + i] = St<DT>::st(y);
  }
}

// rows [0, N): the query latent, normalised, and the cache row
template <int DT>
__global__ __launch_bounds__(256) void latent_prep_kernel(LatentProj a, int Q, const float* q_norm,
                                                          void* cq) {
  using E = typename St<DT>::E;
  __shared__ float red[8];
  const int n = blockIdx.x;
  latent_row<DT, true>(a, n, Q, q_norm, reinterpret_cast<E*>(cq) + (long long)n * a.QP, red);
}

// ---------------------------------------------------------------------------
// one token per sequence: query -> latent space (+ the token's cache row)
// ---------------------------------------------------------------------------
constexpr int kAbsRows = 32, kAbsSeqs = 8;  // latent rows / sequences per workgroup

struct AbsorbArgs {
  LatentProj p;          // proj is read by the appending workgroups only
  const float* q;        // [B][ldq] f32, head h at h (dimp + rotp): [unrotated | rotated part]
  long long ldq;
  const void* uk_t;      // [H][R][dimp]
  int B, H, dimp, rotp, append;
  void* qa;              // [B][H][LD] storage type
};

template <int DT>
__global__ __launch_bounds__(256) void latent_absorb_kernel(AbsorbArgs a) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC, NCH = 256 / EPC / 16;
  __shared__ float qs[kAbsSeqs][256];
  __shared__ float red[8];
  const int h = blockIdx.x, b0 = blockIdx.z * kAbsSeqs, nb = min(kAbsSeqs, a.B - b0);
  if (h == a.H) {  // the appending workgroups (append: one more column of the grid)
    if (blockIdx.y == 0)
      for (int b = 0; b < nb; ++b) {
        latent_row<DT, false>(a.p, b0 + b, 0, nullptr, nullptr, red);
        __syncthreads();
      }
    return;
  }
  const int tid = threadIdx.x, grp = tid >> 4, l16 = tid & 15, nch = a.dimp / EPC;
  const int R = a.p.R, LD = a.p.LD;
  uint4 w[2][NCH];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int row = min((int)blockIdx.y * kAbsRows + 16 * u + grp, R - 1);
    const uint4* src = reinterpret_cast<const uint4*>(
        reinterpret_cast<const E*>(a.uk_t) + ((long long)h * R + row) * a.dimp);
#pragma unroll
    for (int i = 0; i < NCH; ++i)
      w[u][i] = l16 + 16 * i < nch ? src[l16 + 16 * i] : make_uint4(0u, 0u, 0u, 0u);
  }
  const int hd = a.dimp + a.rotp;
  for (int i = tid; i < nb * a.dimp; i += 256) {
    const int b = i / a.dimp, d = i - b * a.dimp;
    qs[b][d] = a.q[(b0 + b) * a.ldq + (long long)h * hd + d];
  }
  if (blockIdx.y == 0) {
    // the rotated part and the padding of all sequences at once: one after the other they were a chain of round
    // trips longer than the products (13 sequences of 16 heads 9.2 us, 7.0 so)
    const int n = LD - R;
    for (int k = tid; k < nb * n; k += 256) {
      const int b = k / n, i = R + k - b * n, j = i - a.p.RP;
      const float* qr = a.q + (b0 + b) * a.ldq + (long long)h * hd + a.dimp;
      float y = j >= 0 && j < a.p.rot ? qr[j] : 0.f;
      if (j >= 0 && j < 2 * a.p.rd2) {
        const float2 t = a.p.cs[(long long)a.p.pos[b0 + b] * a.p.rd2 + (j >> 1)];
        const float o = qr[j ^ 1];
        y = (j & 1) ? y * t.x + o * t.y : y * t.x - o * t.y;
      }
      reinterpret_cast<E*>(a.qa)[((long long)(b0 + b) * a.H + h) * LD + i] = St<DT>::st(y);
    }
  }
  __syncthreads();
  for (int b = 0; b < nb; ++b) {
    E* out = reinterpret_cast<E*>(a.qa) + ((long long)(b0 + b) * a.H + h) * LD;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < NCH; ++i)
        if (l16 + 16 * i < nch) {
          const float* x = qs[b] + (l16 + 16 * i) * EPC;
          if constexpr (DT == kF32) {
            acc = fmaf(__uint_as_float(w[u][i].x), x[0], acc);
            acc = fmaf(__uint_as_float(w[u][i].y), x[1], acc);
            acc = fmaf(__uint_as_float(w[u][i].z), x[2], acc);
            acc = fmaf(__uint_as_float(w[u][i].w), x[3], acc);
          } else {
            float f[8];
            unpack8<DT>(w[u][i], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) acc = fmaf(f[e], x[e], acc);
          }
        }
      acc = row16_sum(acc);
      const int row = blockIdx.y * kAbsRows + 16 * u + grp;
      if (l16 == 0 && row < R) out[row] = St<DT>::st(acc);
    }
  }
}

// ---------------------------------------------------------------------------
// one token per sequence: attention over the cached latent rows
// ---------------------------------------------------------------------------
struct LatDecArgs {
  const void* qa;        // [B][H][LD]
  const void* cache;
  long long slot_stride;
  const int* pos;        // [B]
  const int* slot;
  int H, LD, RP, nsplit, tile;
  float scale_log2;
  float* part;           // [B][H][nsplit][RP + 4]: value sums, running max (log2), sum
};

// keys per split (whole tiles of 32 or 64 keys) and the splits that hold any
__device__ __forceinline__ int latent_split_keys(int Tk, int nsplit, int tile) {
  return ((Tk + nsplit - 1) / nsplit + tile - 1) / tile * tile;
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4* lds_s16x4;

// A operand of the value product from row-major rows: lane (l15, g) holds
// rows[8 g + i][l15], i = 0..7 (row stride ld elements)
template <int DT>
__device__ __forceinline__ uint4 load_cols(const uint16_t* rows, int ld, int l15, int g) {
  const uint16_t* p = rows + (8 * g + (l15 >> 2)) * ld + (l15 & 3) * 4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)p);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4)(p + 4 * ld));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return make_uint4(a.x, a.y, b.x, b.y);
}

// 16-byte pieces of a tile per thread
template <int DT, int RC, int BK> constexpr int lat_pieces() { return DT != kF32 && RC <= 512 && BK == 32 ? 10 : 20; }
// RC: class of the latent size, BK: keys per tile
template <int DT, int RC, int BK>
__global__ __launch_bounds__(256) void latent_decode_kernel(LatDecArgs a) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC, NB = BK / 16, NVT = RC / 64, NLD = lat_pieces<DT, RC, BK>();
  constexpr int PLD = BK + EPC;
  extern __shared__ __attribute__((aligned(16))) unsigned char mixer_smem[];
  __shared__ float red_m[4][16], red_l[4][16];
  const int LD = a.LD, KLD = LD + EPC, KPR = LD / EPC, nks = LD / St<DT>::KSTEP;
  E* const ks_ = reinterpret_cast<E*>(mixer_smem);
  E* const qs = ks_ + BK * KLD;
  E* const ps = qs + 16 * KLD;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l15 = lane & 15, g = lane >> 4;
  const int h0 = blockIdx.x * 16, nr = min(16, a.H - h0), sp = blockIdx.y, b = blockIdx.z;
  const int Tk = a.pos[b] + 1;
  const int kps = latent_split_keys(Tk, a.nsplit, a.tile);
  const int kbeg = sp * kps, kend = min(kbeg + kps, Tk);
  if (kbeg >= kend) return;
  const E* rows = reinterpret_cast<const E*>(a.cache) + a.slot[b] * a.slot_stride;

  u32x4 kr[NLD];
  auto gload = [&](int k0) __attribute__((always_inline)) {
    const u32x4* src = reinterpret_cast<const u32x4*>(rows + (long long)k0 * LD);
#pragma unroll
    for (int i = 0; i < NLD; ++i)
      if (tid + 256 * i < BK * KPR) kr[i] = src[tid + 256 * i];
  };
  // piece tid + 256 i of a tile as (row, column): one division, then steps
  const int rs = 256 / KPR, cs = 256 - rs * KPR, r_0 = tid / KPR, c_0 = tid - r_0 * KPR;
  auto step = [&](int& r, int& c) __attribute__((always_inline)) {
    r += rs;
    c += cs;
    if (c >= KPR) { c -= KPR; ++r; }
  };
  auto sstore = [&]() __attribute__((always_inline)) {
    int r = r_0, c = c_0;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      if (r < BK) *reinterpret_cast<u32x4*>(ks_ + r * KLD + c * EPC) = kr[i];
      step(r, c);
    }
  };
  gload(kbeg);
  {
    int r = r_0, c = c_0;
    const E* qb = reinterpret_cast<const E*>(a.qa) + ((long long)b * a.H + h0) * LD;
    constexpr int NLQ = (NLD * 16 + BK - 1) / BK + 1;  // pieces of 16 rows per thread
#pragma unroll
    for (int i = 0; i < NLQ; ++i) {
      if (r < 16)
        *reinterpret_cast<u32x4*>(qs + r * KLD + c * EPC) =
            *reinterpret_cast<const u32x4*>(qb + (long long)min(r, nr - 1) * LD + c * EPC);
      step(r, c);
    }
  }
  cf32x4 o[NVT];
#pragma unroll
  for (int t = 0; t < NVT; ++t) o[t] = cf32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int k0 = kbeg; k0 < kend; k0 += BK) {
    if (k0 != kbeg) __syncthreads();  // every wave is past the tile before it is replaced
    sstore();
    __syncthreads();
    if (k0 + BK < kend) gload(k0 + BK);
    cf32x4 s{0.f, 0.f, 0.f, 0.f};
    if (wave < NB) {
      const E* kp = ks_ + (16 * wave + l15) * KLD + g * EPC;
      const E* qp = qs + l15 * KLD + g * EPC;
      // six steps' operands in flight, two accumulation chains
      cf32x4 s1{0.f, 0.f, 0.f, 0.f};
      int i = 0;
      for (; i + 6 <= nks; i += 6) {
        uint4 kf[6], qf[6];
#pragma unroll
        for (int u = 0; u < 6; ++u) {
          kf[u] = *reinterpret_cast<const uint4*>(kp + 4 * (i + u) * EPC);
          qf[u] = *reinterpret_cast<const uint4*>(qp + 4 * (i + u) * EPC);
        }
#pragma unroll
        for (int u = 0; u < 6; u += 2) {
          s = mm_piece<DT>(kf[u], qf[u], s);
          s1 = mm_piece<DT>(kf[u + 1], qf[u + 1], s1);
        }
      }
      for (; i < nks; ++i)
        s = mm_piece<DT>(*reinterpret_cast<const uint4*>(kp + 4 * i * EPC),
                         *reinterpret_cast<const uint4*>(qp + 4 * i * EPC), s);
      s += s1;
      float mx = -INFINITY;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        s[e] = k0 + 16 * wave + 4 * g + e < kend ? s[e] * a.scale_log2 : -INFINITY;
        mx = fmaxf(mx, s[e]);
      }
      mx = group_max(mx);
      if (g == 0) red_m[wave][l15] = mx;
    }
    __syncthreads();
    float mn = m;
#pragma unroll
    for (int w = 0; w < NB; ++w) mn = fmaxf(mn, red_m[w][l15]);  // finite: the tile holds a key
    const float alpha = __builtin_amdgcn_exp2f(m - mn);
    m = mn;
    if (wave < NB) {
      float p[4], rs = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        p[e] = __builtin_amdgcn_exp2f(s[e] - mn);
        rs += p[e];
      }
      l = l * alpha + rs;
      E* dst = ps + l15 * PLD + 16 * wave + 4 * g;
      if constexpr (DT == kF32) {
        *reinterpret_cast<float4*>(dst) = make_float4(p[0], p[1], p[2], p[3]);
      } else {
        *reinterpret_cast<uint2*>(dst) =
            make_uint2((uint32_t)St<DT>::st(p[0]) | ((uint32_t)St<DT>::st(p[1]) << 16),
                       (uint32_t)St<DT>::st(p[2]) | ((uint32_t)St<DT>::st(p[3]) << 16));
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NVT; ++t) o[t] *= alpha;
    constexpr int STEP = DT == kF32 ? 16 : 32;
#pragma unroll
    for (int kk = 0; kk < BK / STEP; ++kk) {
      const uint4 pf =
          *reinterpret_cast<const uint4*>(ps + l15 * PLD + STEP * kk + (STEP / 4) * g);
#pragma unroll
      for (int t = 0; t < NVT; ++t) {
        const int d0 = 16 * (wave + 4 * t);
        if (d0 < a.RP) {
          const E* base = ks_ + STEP * kk * KLD + d0;
          uint4 vf;
          if constexpr (DT == kF32) {
            const E* p = base + 4 * g * KLD + l15;
            vf = make_uint4(__float_as_uint(p[0]), __float_as_uint(p[KLD]),
                            __float_as_uint(p[2 * KLD]), __float_as_uint(p[3 * KLD]));
          } else {
            vf = load_cols<DT>(base, KLD, l15, g);
          }
          o[t] = mm_piece<DT>(vf, pf, o[t]);
        }
      }
    }
  }
  l = group_sum(l);
  if (g == 0) red_l[wave][l15] = l;
  __syncthreads();
  if (l15 >= nr) return;
  const int PS = a.RP + 4;
  float* dst = a.part + (((long long)b * a.H + h0 + l15) * a.nsplit + sp) * PS;
#pragma unroll
  for (int t = 0; t < NVT; ++t) {
    const int d0 = 16 * (wave + 4 * t);
    if (d0 < a.RP)
      *reinterpret_cast<float4*>(dst + d0 + 4 * g) = make_float4(o[t][0], o[t][1], o[t][2], o[t][3]);
  }
  if (wave == 0 && g == 0) {
    dst[a.RP] = m;
    dst[a.RP + 1] = (red_l[0][l15] + red_l[1][l15]) + (red_l[2][l15] + red_l[3][l15]);
  }
}

// ---------------------------------------------------------------------------
// one token per sequence: merge of the splits, value expansion
// ---------------------------------------------------------------------------
constexpr int kOutRows = 16;  // value rows per workgroup

struct LatOutArgs {
  const float* part;
  const int* pos;
  const void* uv;        // [H][DVP][RP]
  int H, vdim, DVP, RP, nsplit, tile;
  void* out;             // [B][ldo], head h at h vdim
  long long ldo;
};

template <int DT>
__global__ __launch_bounds__(256) void latent_out_kernel(LatOutArgs a) {
  using E = typename St<DT>::E;
  constexpr int EPC = St<DT>::EPC, NCH = 1024 / EPC / 64;
  __shared__ __attribute__((aligned(16))) float ol[1024];
  __shared__ float ws[64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int h = blockIdx.y, b = blockIdx.z, nch = a.RP / EPC, PS = a.RP + 4;
  const int r0 = blockIdx.x * kOutRows + 4 * wave;
  uint4 w[4][NCH];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4* src = reinterpret_cast<const uint4*>(
        reinterpret_cast<const E*>(a.uv) + ((long long)h * a.DVP + min(r0 + i, a.DVP - 1)) * a.RP);
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      w[i][c] = lane + 64 * c < nch ? src[lane + 64 * c] : make_uint4(0u, 0u, 0u, 0u);
  }
  const int Tk = a.pos[b] + 1, kps = latent_split_keys(Tk, a.nsplit, a.tile);
  const int nact = (Tk + kps - 1) / kps;
  const float* part = a.part + ((long long)b * a.H + h) * a.nsplit * PS;
  if (wave == 0) {
    const float* ml = part + (long long)min(lane, nact - 1) * PS + a.RP;
    const float m = lane < nact ? ml[0] : -INFINITY, l = lane < nact ? ml[1] : 0.f;
    const float f = __builtin_amdgcn_exp2f(m - wave_max(m));
    const float den = wave_sum(f * l);
    ws[lane] = f / den;
  }
  __syncthreads();
  for (int r = tid; r < a.RP; r += 256) {
    float acc = 0.f;
    for (int s0 = 0; s0 < nact; s0 += 8) {  // eight partials in flight
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = part[(long long)min(s0 + j, nact - 1) * PS + r];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < nact) acc = fmaf(ws[s0 + j], v[j], acc);
    }
    ol[r] = acc;
  }
  __syncthreads();
  E* out = reinterpret_cast<E*>(a.out) + b * a.ldo + (long long)h * a.vdim;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float acc = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      if (lane + 64 * c < nch) {
        const float* x = ol + (lane + 64 * c) * EPC;
        if constexpr (DT == kF32) {
          acc = fmaf(__uint_as_float(w[i][c].x), x[0], acc);
          acc = fmaf(__uint_as_float(w[i][c].y), x[1], acc);
          acc = fmaf(__uint_as_float(w[i][c].z), x[2], acc);
          acc = fmaf(__uint_as_float(w[i][c].w), x[3], acc);
        } else {
          float f[8];
          unpack8<DT>(w[i][c], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc = fmaf(f[e], x[e], acc);
        }
      }
    acc = wave_sum(acc);
    if (lane == 0 && r0 + i < a.vdim) out[r0 + i] = St<DT>::st(acc);
  }
}

template <int DT, int RC, int BK>
static int launch_latent_decode(const LatDecArgs& a, dim3 grid, hipStream_t st) {
  constexpr int EPC = St<DT>::EPC;
  const size_t lds = ((size_t)(BK + 16) * (a.LD + EPC) + 16 * (BK + EPC)) *
                     sizeof(typename St<DT>::E);
  if (BK * (a.LD / EPC) > 256 * lat_pieces<DT, RC, BK>() || lds > 150 * 1024) return (int)hipErrorInvalidValue;
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)latent_decode_kernel<DT, RC, BK>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, 150 * 1024) != hipSuccess)
      return (int)hipErrorInvalidValue;
    raised = true;
  }
  hipLaunchKernelGGL((latent_decode_kernel<DT, RC, BK>), grid, dim3(256), lds, st, a);
  return (int)hipGetLastError();
}

}  // namespace cake

using namespace cake;

static bool latent_ok(int R, int RP, int rot, int LD, int rd2) {
  return R > 0 && RP >= R && RP % 16 == 0 && RP <= 1024 && rot >= 0 && LD >= RP + rot &&
         LD % 32 == 0 && LD <= RP + 128 + 32 && rot <= 128 && rd2 >= 0 && 2 * rd2 <= rot;
}

CAKE_API int cake_latent_prep(int dt, const float* proj, long long ldp, int N, int Q, int QP, int R,
                              int RP, int rot, int LD, int rd2, float eps, const float* q_norm,
                              const float* kv_norm, const void* cs, const int* pos, const int* slot,
                              void* cq, void* cache, long long slot_stride, hipStream_t st) {
  if (!latent_ok(R, RP, rot, LD, rd2) || N < 0 || Q < 1 || Q > QP || QP % 8 ||
      ldp < QP + RP + rot || ldp % 4 || (uintptr_t)proj % 16 || (uintptr_t)cq % 16 ||
      (uintptr_t)cache % 16 || (uintptr_t)q_norm % 16 || (uintptr_t)kv_norm % 16 || slot_stride % 8)
    return (int)hipErrorInvalidValue;
  if (N == 0) return 0;
  const LatentProj p{proj, ldp, QP, R, RP, rot, LD, rd2, eps, kv_norm, (const float2*)cs,
                     pos, slot, cache, slot_stride};
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((latent_prep_kernel<DT>), dim3(N), dim3(256), 0, st, p, Q,
                                     q_norm, cq));
  return (int)hipGetLastError();
}

// append: also write the rows' cache entries from proj (else proj may be null)
CAKE_API int cake_latent_absorb(int dt, const float* q, long long ldq, const void* uk_t, int B,
                                int H, int dimp, int rotp, int append, const float* proj,
                                long long ldp, int QP, int R, int RP, int rot, int LD, int rd2,
                                float eps, const float* kv_norm, const void* cs, const int* pos,
                                const int* slot, void* cache, long long slot_stride, void* qa,
                                hipStream_t st) {
  if (!latent_ok(R, RP, rot, LD, rd2) || B <= 0 || H <= 0 || dimp <= 0 || dimp % 8 || dimp > 256 ||
      rotp < rot || ldq < (long long)H * (dimp + rotp) ||
      (append && (proj == nullptr || ldp < QP + RP + rot || ldp % 4 || QP % 4 ||
                  (uintptr_t)proj % 16 || (uintptr_t)cache % 16 || (uintptr_t)kv_norm % 16 ||
                  slot_stride % 8)))
    return (int)hipErrorInvalidValue;
  const LatentProj p{proj, ldp, QP, R, RP, rot, LD, rd2, eps, kv_norm, (const float2*)cs,
                     pos, slot, cache, slot_stride};
  const AbsorbArgs a{p, q, ldq, uk_t, B, H, dimp, rotp, append, qa};
  const dim3 grid(H + (append ? 1 : 0), (R + kAbsRows - 1) / kAbsRows,
                  (B + kAbsSeqs - 1) / kAbsSeqs);
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((latent_absorb_kernel<DT>), grid, dim3(256), 0, st, a));
  return (int)hipGetLastError();
}

// tile: 32 or 64 keys, as cake_latent_out takes it.  A CU reads some 25 KB a us and a tile of 64 keys is 74 KB: the
// attention and value expansion of one sequence of 32 heads over 40 / 150 / 250 keys 12.2 / 12.9 / 13.3 us in up to four
// 64-key tiles, 11.0 / 12.0 / 12.3 in eight of 32; of 13 sequences 18.9 / 22.5 / 23.0, 20.0 / 23.1 / 25.3.
CAKE_API int cake_latent_decode(int dt, const void* qa, const void* cache, long long slot_stride,
                                const int* pos, const int* slot, int B, int H, int LD, int RP,
                                int nsplit, int tile, float scale, float* part, hipStream_t st) {
  if (B <= 0 || H <= 0 || LD % 32 || RP % 16 || RP <= 0 || RP > 1024 || LD < RP || nsplit < 1 ||
      nsplit > 64 || (tile != 32 && tile != 64))
    return (int)hipErrorInvalidValue;
  const LatDecArgs a{qa, cache, slot_stride, pos, slot, H, LD, RP, nsplit, tile,
                     scale * 1.4426950408889634f, part};
  const dim3 grid((H + 15) / 16, nsplit, B);
  CAKE_MIX_DT(dt, {
    constexpr bool F = DT == kF32;
    if (RP <= 256 && LD <= (F ? 384 : 640))
      return F || tile == 32 ? launch_latent_decode<DT, 256, 32>(a, grid, st)
                                    : launch_latent_decode<DT, 256, 64>(a, grid, st);
    if (RP <= 512 && LD <= 640)
      return F || tile == 32 ? launch_latent_decode<DT, 512, 32>(a, grid, st)
                                    : launch_latent_decode<DT, 512, 64>(a, grid, st);
    return launch_latent_decode<DT, 1024, F ? 16 : 32>(a, grid, st);
  });
  return (int)hipErrorInvalidValue;
}

CAKE_API int cake_latent_out(int dt, const float* part, const int* pos, const void* uv, int B,
                             int H, int vdim, int DVP, int RP, int nsplit, int tile, void* out,
                             long long ldo, hipStream_t st) {
  if (B <= 0 || H <= 0 || vdim <= 0 || DVP < vdim || RP % 16 || RP <= 0 || RP > 1024 ||
      nsplit < 1 || nsplit > 64 || (tile != 32 && tile != 64) || ldo < (long long)H * vdim)
    return (int)hipErrorInvalidValue;
  const LatOutArgs a{part, pos, uv, H, vdim, DVP, RP, nsplit, tile, out, ldo};
  const dim3 grid((vdim + kOutRows - 1) / kOutRows, H, B);
  CAKE_MIX_DT(dt, hipLaunchKernelGGL((latent_out_kernel<DT>), grid, dim3(256), 0, st, a));
  return (int)hipGetLastError();
}

// Prompt rows: q [N][ldq] (heads [dimp | rotp], not rotated yet), keys k [rows][ldk] (heads dimp
// wide) and transposed values vt [H DVP][ldv] of the live positions, sequence b at row / column
// koff[b].
CAKE_API int cake_latent_flash(int dt, const void* q, long long ldq, const void* k, long long ldk,
                               const void* vt, long long ldv, const int* koff, const void* cache,
                               long long slot_stride, int LD, int RP, const void* seq, int B,
                               int max_len, const void* cs, int rd2, int H, int dimp, int rotp,
                               int vdim, int DP, int DVP, float scale, void* out, long long ldo,
                               hipStream_t st) {
  if (B <= 0 || max_len <= 0 || H <= 0 || dimp <= 0 || dimp % 8 || rotp < 0 || rotp % 8 ||
      DP % 32 || DP < dimp + rotp || DP > 256 || DVP % 16 || DVP < vdim || DVP > 256 || vdim <= 0 ||
      ldq % 8 || ldk % 8 || ldv % 64 || LD % 32 || RP % 16 || RP + rotp > LD ||
      2 * rd2 > rotp || rd2 < 0)
    return (int)hipErrorInvalidValue;
  MixFlashArgs a{};
  a.qn = q; a.kc = k; a.vc = vt;
  a.seq = (const SeqRow*)seq;
  a.out = out; a.ldo = ldo;
  a.H = H; a.G = H; a.DP = DP; a.DVP = DVP; a.vdim = vdim;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.lat.koff = koff;
  a.lat.rope = nullptr;
  a.lat.rope_slot = slot_stride;
  a.lat.ldr = LD;
  a.lat.dimp = dimp; a.lat.rotp = rotp;
  a.lat.ldq = ldq; a.lat.ldk = ldk; a.lat.ldv = ldv;
  a.lat.cs = (const float2*)cs;
  a.lat.rd2 = rd2;
  if (dt != kF32) {
    a.lat.rope = reinterpret_cast<const uint16_t*>(cache) + RP;
    if (flash3_ok(dt, a, true, slot_stride / LD, max_len, B))
      return dt == kBF16 ? launch_mix_flash3<kBF16, true>(a, max_len, B, st)
                         : launch_mix_flash3<kF16, true>(a, max_len, B, st);
  }
  const dim3 grid((max_len + 127) / 128, H, B);
  CAKE_MIX_DT(dt, {
    a.lat.rope = reinterpret_cast<const typename St<DT>::E*>(cache) + RP;
    if (DP == 192 && DVP == 128) return launch_mix_flash<DT, 192, 128, true, true>(a, grid, st);
    if (DP <= 192 && DVP <= 128) return launch_mix_flash<DT, 192, 128, false, true>(a, grid, st);
    return launch_mix_flash<DT, 256, 256, false, true>(a, grid, st);
  });
  return (int)hipErrorInvalidValue;
}
