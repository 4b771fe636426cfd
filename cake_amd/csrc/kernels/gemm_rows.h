// Products of few rows (M <= 64): short prompts, one token of several sequences, routed experts.
// The weights are read once and little is done with each of them, so the time is their bytes (and
// a launch's fixed costs); two forms, chosen by gemm.hip rows_kind from the sizes.
//
// gemm_direct_kernel (M <= 32, weights up to some 60 MB): a workgroup owns 16 or 32 weight rows over
//   the whole of k, its eight waves taking 64-element chunks of k in turn, operands straight into
//   MFMA fragments; the waves' sums meet in LDS.  No partial sums in memory, no second launch, no
//   barrier in the loop: 4096 x 4096 at 5 / 16 rows 9.7 / 11.5 us (tile kernel with split k and its
//   finalize launch: 15-17 us), 2048 x 2048 6.1 / 7.1 us (14.6 us).  Every strip reads all of x
//   from L2, which is what ends its range.
// gemm_stream_kernel (M <= 64): 128 weight rows by 64 k (up to 16 rows of x 64 by 128) and the x tile
//   go through LDS by DMA; the steps of all strips form one sequence dealt out in equal contiguous
//   shares, at most one workgroup per CU (two): whole strips or equal parts of one where that pays, else
//   ends anywhere (gemm.hip stream_plan).  Strips that several shares cover meet in memory, the last to
//   arrive sums in share order (the result does not hang on the order).  28672 x 4096 SwiGLU at 5 / 24 /
//   45 rows 38 / 38 / 40 us (tile kernels 58-60 us), 4096 x 23552 33 / 37 / 43 us (44-46 us), 57344 x 8192
//   140 us (6.7 TB/s).  What bounds it is the memory in whole strips, in parts the parked sums; weight
//   rings of a wave's own with a barrier every four steps only ran at the same rate.  Of 128-row strips, and where sums stay in
//   slabs, four waves ask and four multiply: loads go on while a strip's sums are parked, summed and stored, and every
//   multiplying wave parks for itself (in one: 28672 x 4096 SwiGLU at 5 rows 39.9 -> 38.4 us, 6144 x 4096 in quarters at 45
//   15.0 -> 14.0, 4096 x 4096 in eighths 11.8 -> 11.1).  Strips of 64 rows whose sums meet are short and met by up to 60 shares:
//   their four waves ask and multiply in turn (at 5 rows, in two kinds: 1024 x 4096 8.2, 8.9; 256 x 11008 10.6, 12.6; 1536 x
//   8960 14.0, 15.7; 2048 x 8192 10.7, 11.3; 5120 x 5120 13.8, 13.4; 8192 x 28672 70.7, 70.5).
#pragma once
#include "gemm_kernel.h"

namespace cake {

constexpr int kRowsMinK = 512;       // k of a share at least
constexpr int kRowsTicks = 65536;    // strips of a launch at most (of 128 rows an arrival counter for each of four waves)

// the operand fragments of one 64-element chunk of k: a lane's two 16-byte pieces of each row are
// neighbours, so the two MFMA steps read whole 128-byte lines (both operands use one order of k)
template <int DT, int MT, int NT>
struct DirectChunk {
  uint4 w[NT][2], x[MT][2];

  __device__ __forceinline__ void load(const uint16_t* const* wp, const uint16_t* const* xp, int k) {
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) w[j][h] = ld_nt16(reinterpret_cast<const uint4*>(wp[j] + k) + h);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) x[i][h] = reinterpret_cast<const uint4*>(xp[i] + k)[h];
  }

  // the last, short chunk: pieces past the end are zero in both operands
  __device__ __forceinline__ void load_tail(const uint16_t* const* wp, const uint16_t* const* xp, int k,
                                            int left) {
    const uint4 z = make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = h * 8 < left;   // left: elements of the row from this lane's first piece on
#pragma unroll
      for (int j = 0; j < NT; ++j) w[j][h] = in ? reinterpret_cast<const uint4*>(wp[j] + k)[h] : z;
#pragma unroll
      for (int i = 0; i < MT; ++i) x[i][h] = in ? reinterpret_cast<const uint4*>(xp[i] + k)[h] : z;
    }
  }

  __device__ __forceinline__ void mac(cf32x4 (&acc)[NT][MT]) const {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[j][i] = cmfma<DT>(w[j][h], x[i][h], acc[j][i]);
  }
};

template <int DT, int EPI, int MT, int NT>
__global__ __launch_bounds__(512) void gemm_direct_kernel(GemmArgs g) {
  constexpr bool GATED = (EPI == kEpiSwiglu || EPI == kEpiGeglu);
  constexpr int NW = 8, D = 2;   // waves, chunks in flight of each
  constexpr int TILES = NT * MT;
  constexpr int GRP = TILES * NW <= 64 ? TILES : 64 / NW;   // tiles summed per round (<= 64 KB)
  static_assert(TILES % GRP == 0 && (!GATED || (NT == 2 && GRP % 2 == 0)), "direct tile groups");
  __shared__ float4 red[NW][GRP][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int v0 = blockIdx.x * NT * 16;

  const int r = lane & 15, kq = (lane >> 4) * 16;
  const uint16_t *wp[NT], *xp[MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wp[j] = g.b + (size_t)wrow(g, min(v0 + j * 16 + r, g.Nv - 1)) * g.ldb + kq;
#pragma unroll
  for (int i = 0; i < MT; ++i) xp[i] = g.a + (size_t)min(i * 16 + r, g.M - 1) * g.lda + kq;

  cf32x4 acc[NT][MT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[j][i] = cf32x4{0.f, 0.f, 0.f, 0.f};

  // wave w takes chunks w, w + NW, .. of the workgroup's whole ones, D of them in flight
  const int nfull = g.K / 64;
  const int mine = nfull > wave ? (nfull - wave + NW - 1) / NW : 0;
  const int k = wave * 64;
  DirectChunk<DT, MT, NT> buf[D];
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < mine) buf[d].load(wp, xp, k + d * NW * 64);
  int c = 0;
  for (; c + 2 * D <= mine; c += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      buf[d].mac(acc);
      buf[d].load(wp, xp, k + (c + D + d) * NW * 64);
    }
  }
  for (; c < mine; c += D) {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (c + d < mine) {
        buf[d].mac(acc);
        if (c + D + d < mine) buf[d].load(wp, xp, k + (c + D + d) * NW * 64);
      }
  }
  const int rest = g.K - nfull * 64;
  if (rest > 0 && wave == nfull % NW) {
    DirectChunk<DT, MT, NT> t;
    t.load_tail(wp, xp, nfull * 64, rest - kq);
    t.mac(acc);
  }

  // the waves' sums meet in LDS; item = (tile, lane): token i * 16 + (lane & 15), four weight rows
#pragma unroll
  for (int t0 = 0; t0 < TILES; t0 += GRP) {
    // tile t = i * NT + j, so the two halves of a gated pair are neighbours
#pragma unroll
    for (int t = 0; t < GRP; ++t) {
      const cf32x4 a = acc[(t0 + t) % NT][(t0 + t) / NT];
      red[wave][t][lane] = make_float4(a[0], a[1], a[2], a[3]);
    }
    __syncthreads();
    constexpr int STEP = GATED ? 2 : 1;
    for (int it = threadIdx.x; it < GRP / STEP * 64; it += NW * 64) {
      const int t = it / 64 * STEP, l = it % 64;
      float s[STEP][4];
#pragma unroll
      for (int q = 0; q < STEP; ++q) {
        float4 a = red[0][t + q][l];
#pragma unroll
        for (int w = 1; w < NW; ++w) {
          const float4 b = red[w][t + q][l];
          a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
        }
        s[q][0] = a.x; s[q][1] = a.y; s[q][2] = a.z; s[q][3] = a.w;
      }
      const int i = (t0 + t) / NT, j = (t0 + t) % NT;
      const int m = i * 16 + (l & 15);
      if (m >= g.M) continue;
      const int n = (GATED ? blockIdx.x * 16 : v0 + j * 16) + (l >> 4) * 4;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int nn = min(n + e, g.N - 1);
        float a = s[0][e] + (g.bias != nullptr ? to_f32<DT>(g.bias[nn]) : 0.f);
        if constexpr (GATED) {
          const float b = s[STEP - 1][e] + (g.bias != nullptr ? to_f32<DT>(g.bias[g.half + nn]) : 0.f);
          a = EPI == kEpiSwiglu ? silu(a) * b : a * gelu_tanh(b);
        }
        if constexpr (EPI == kEpiAdd16) a += to_f32<DT>(g.r16[(size_t)m * g.ldr + nn]);
        if constexpr (act_epi(EPI)) a = gemm_act<EPI>(a);
        y[e] = a;
      }
      if constexpr (EPI == kEpiResid32 || EPI == kEpiStore32) {
        float* o = g.r32 + (size_t)m * g.ldr + n;
        if (n + 4 <= g.N && ((g.ldr | n) & 3) == 0) {
          float4 v = EPI == kEpiResid32 ? *reinterpret_cast<float4*>(o) : make_float4(0.f, 0.f, 0.f, 0.f);
          v.x = fmaf(g.alpha, y[0], v.x); v.y = fmaf(g.alpha, y[1], v.y);
          v.z = fmaf(g.alpha, y[2], v.z); v.w = fmaf(g.alpha, y[3], v.w);
          *reinterpret_cast<float4*>(o) = v;
        } else {
          for (int e = 0; e < 4; ++e)
            if (n + e < g.N) o[e] = fmaf(g.alpha, y[e], EPI == kEpiResid32 ? o[e] : 0.f);
        }
      } else {
        uint16_t* o = g.c + (size_t)m * g.ldc + n;
        for (int e = 0; e < 4; ++e)
          if (n + e < g.N) o[e] = from_f32<DT>(y[e]);
      }
    }
    if (t0 + GRP < TILES) __syncthreads();
  }
}

// MT: 16-row tiles of x.  A stage holds 16 KB of weights: WIDE 128 rows by 64 k, else 64 by 128.
// What one workgroup of four waves can have outstanding moves 5.2 TB/s at any depth, two on a CU
// 6.1; with 64-row strips the parked sums of 512 shares are as many as those of 256 shares of 128.
// That pays while x is one tile (5 / 13 rows: 2048 x 8192 15.3 / 16.0 -> 13.6 / 13.9 us, 8192 x 8192
// 35.7 / 36.3 -> 32.1 / 32.6, 4096 x 14336 25.1 / 25.6 -> 24.1 / 25.0); at 24 rows x is read twice as
// often for it (4096 x 23552 38.7 -> 40.8).  Gated rows pair up within 32 of a wave.
template <int MT, bool WIDE> struct StreamShape {
  static constexpr int NWV = 4, RT = WIDE ? 2 : 1, KC = WIDE ? 1 : 2;   // row tiles, 64-element chunks
  static constexpr int BN = NWV * 16 * RT, KST = 64 * KC;   // weight rows of a strip, k of a step
  static constexpr int NS = WIDE ? 4 : 3, WGS = WIDE ? 256 : 512;
  static constexpr int LPR = 8 * KC, RPI = 64 / LPR;   // lanes of a row's DMA, rows of an instruction
  static constexpr int XT = 2 * MT * KC;               // x DMA instructions of a step
  static constexpr int XW = XT % 4 == 0 ? 4 : XT % 3 == 0 ? 3 : 2;   // waves that issue them
  static constexpr int XI = XT / XW;
  static constexpr int IPW = 4 + XI;
  static constexpr int STAGE = (BN + MT * 16) * 128 * KC;
  // 16-byte chunk c of row r is in slot c ^ swz(r)
  static __device__ __forceinline__ int swz(int r) { return KC == 2 ? r & 15 : (r >> 1) & 7; }
};
template <int EPI, int MT> constexpr bool stream_wide() {
  return MT > 1 || EPI == kEpiSwiglu || EPI == kEpiGeglu;
}
// four more waves ask for what these multiply
template <int EPI, int MT> constexpr bool stream_ask() { return stream_wide<EPI, MT>() || EPI == kEpiPartial; }
template <int EPI, int MT> constexpr int stream_threads() { return stream_ask<EPI, MT>() ? 512 : 256; }

// N 16-row fragments (two 32-element chunks of k) at base + STRIDE i; waits for them
template <int N, int STRIDE>
__device__ __forceinline__ void stream_read(uint32_t lo, uint32_t hi, uint4 (&a)[N][2]) {
  static_assert(N == 1 || N == 2, "fragments per read");
  if constexpr (N == 2)
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:%6\n\t"
                 "ds_read_b128 %3, %5 offset:%6\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1]), "=&v"(a[1][0]), "=&v"(a[1][1])
                 : "v"(lo), "v"(hi), "i"(STRIDE) : "memory");
  else
    asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                 : "=&v"(a[0][0]), "=&v"(a[0][1]) : "v"(lo), "v"(hi) : "memory");
}

struct StreamStrip {   // one strip of the step sequence
  const uint16_t *a, *b;
  uint16_t* c;
  float* f;   // f32 output, rows ldf apart
  long long ldf;
  int M, v0;
};

template <bool GRP, int BN>
__device__ __forceinline__ StreamStrip stream_strip(const GemmArgs& g, int s) {
  StreamStrip r{g.a, g.b, g.c, g.r32, g.ldr, g.M, s * BN};
  if constexpr (GRP) {
    const int4 t = g.groups[s / g.tiles_n];
    r.a += (size_t)t.y * g.lda;
    r.c += (size_t)t.y * g.ldc;
    r.b += (size_t)t.x * g.b_group;
    r.M = t.z;
    r.v0 = (s % g.tiles_n) * BN;
  }
  return r;
}

// epilogue of one wave's sums: acc[j][i][e] is token 16 i + (lane & 15), virtual weight row
// v0 + 16 RT wave + 16 j + 4 (lane >> 4) + e
template <int DT, int EPI, int MT, int RT>
__device__ __forceinline__ void stream_store(const GemmArgs& g, const StreamStrip& s, int wave, int lane,
                                             const cf32x4 (&acc)[RT][MT]) {
  constexpr bool GATED = (EPI == kEpiSwiglu || EPI == kEpiGeglu);
  static_assert(!GATED || RT == 2, "a gate row and its up row in one wave");
  const int vw = s.v0 + wave * (16 * RT);
#pragma unroll
  for (int j = 0; j < (GATED ? 1 : RT); ++j) {
    const int n = (GATED ? vw / 2 : vw + j * 16) + (lane >> 4) * 4;
    if (n >= g.N) continue;
    const bool full = n + 4 <= g.N;
    float b0[4], b1[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int nn = min(n + e, g.N - 1);
      b0[e] = g.bias != nullptr ? to_f32<DT>(g.bias[nn]) : 0.f;
      b1[e] = GATED && g.bias != nullptr ? to_f32<DT>(g.bias[g.half + nn]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = i * 16 + (lane & 15);
      if (m >= s.M) continue;
      float y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float a = acc[j][i][e] + b0[e];
        if constexpr (GATED) {
          const float u = acc[RT - 1][i][e] + b1[e];
          a = EPI == kEpiSwiglu ? silu(a) * u : a * gelu_tanh(u);
        }
        if constexpr (EPI == kEpiAdd16) a += to_f32<DT>(g.r16[(size_t)m * g.ldr + min(n + e, g.N - 1)]);
        if constexpr (act_epi(EPI)) a = gemm_act<EPI>(a);
        y[e] = a;
      }
      if constexpr (EPI == kEpiSections) {   // a group of four columns lies in one section
        const bool act = n >= g.n2;
        if (!act && n >= g.n1) {
          float* o = g.r32 + (size_t)m * g.ldr + (n - g.n1);
          if ((g.ldr & 3) == 0) *reinterpret_cast<float4*>(o) = make_float4(y[0], y[1], y[2], y[3]);
          else for (int e = 0; e < 4; ++e) o[e] = y[e];
          continue;
        }
        uint16_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = from_f32<DT>(act ? gemm_act<kEpiGelu>(y[e]) : y[e]);
        const long long ld = act ? g.ldc : g.ldc1;
        uint16_t* o = (act ? g.c - g.n2 : g.c1) + (size_t)m * ld + n;
        if (full && (ld & 3) == 0) *reinterpret_cast<uint2*>(o) = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
        else for (int e = 0; e < 4; ++e) if (n + e < g.N) o[e] = v[e];
      } else if constexpr (EPI == kEpiResid32 || EPI == kEpiStore32 || EPI == kEpiPartial) {
        constexpr bool ADD = EPI == kEpiResid32;
        float* o = s.f + (size_t)m * s.ldf + n;
        if (full && ((s.ldf | n) & 3) == 0) {
          float4 v = ADD ? *reinterpret_cast<float4*>(o) : make_float4(0.f, 0.f, 0.f, 0.f);
          v.x = fmaf(g.alpha, y[0], v.x); v.y = fmaf(g.alpha, y[1], v.y);
          v.z = fmaf(g.alpha, y[2], v.z); v.w = fmaf(g.alpha, y[3], v.w);
          *reinterpret_cast<float4*>(o) = v;
        } else {
          for (int e = 0; e < 4; ++e)
            if (n + e < g.N) o[e] = fmaf(g.alpha, y[e], ADD ? o[e] : 0.f);
        }
      } else {
        uint16_t* o = s.c + (size_t)m * g.ldc + n;
        uint16_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = from_f32<DT>(y[e]);
        if (full && ((g.ldc | n) & 3) == 0 && ((uintptr_t)s.c & 7) == 0)
          *reinterpret_cast<uint2*>(o) = make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
        else
          for (int e = 0; e < 4; ++e) if (n + e < g.N) o[e] = v[e];
      }
    }
  }
}

__device__ __forceinline__ void park(float* p, const cf32x4& v) {
  st_agent16(reinterpret_cast<float4*>(p), v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ cf32x4 unpark(const float* p) {
  const float4 v = ld_agent16(reinterpret_cast<const float4*>(p));
  return cf32x4{v.x, v.y, v.z, v.w};
}

template <int DT, int EPI, int MT, bool GRP>
__global__ __launch_bounds__((stream_threads<EPI, MT>()),
                             (stream_ask<EPI, MT>() ? StreamShape<MT, stream_wide<EPI, MT>()>::WGS / 128 : 2))
    void gemm_stream_kernel(GemmArgs g) {
  using S = StreamShape<MT, stream_wide<EPI, MT>()>;
  constexpr bool ASK = stream_ask<EPI, MT>();
  constexpr int NWV = S::NWV, RT = S::RT, KC = S::KC, KST = S::KST;
  __shared__ __attribute__((aligned(16))) uint8_t smem[S::NS * S::STAGE];
  __shared__ unsigned last;
  const int tid = threadIdx.x, who = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wave = who % NWV;
  const int KS = (g.K + KST - 1) / KST;
  const int strips = (GRP ? g.groups[g.tiles_m].x : 1) * g.tiles_n;
  const int total = strips * KS;
  const int per = EPI == kEpiPartial ? g.kps : max((total + (int)gridDim.x - 1) / (int)gridDim.x, g.kps);
  // neighbouring shares on one XCD (they read one strip's x and meet in its sums)
  const int nwg = gridDim.x, q8 = nwg / 8, r8 = nwg % 8, x8 = blockIdx.x % 8;
  const int wg = (x8 < r8 ? x8 * (q8 + 1) : r8 * (q8 + 1) + (x8 - r8) * q8) + blockIdx.x / 8;
  // slabs: every strip in g.pieces parts of g.kps steps (the last what is left), which do not meet
  const bool parts = EPI == kEpiPartial && g.pieces > 1;
  const int part = parts ? wg % g.pieces : 0;
  const int u0 = parts ? wg / g.pieces * KS + part * per : wg * per;
  const int u1 = parts ? min((wg / g.pieces + 1) * KS, u0 + per) : min(total, u0 + per);
  if (u0 >= u1) return;

  // ---- what is asked for: wave w the rows 16 RT w .. of the weights and its share of x ----
  const int dr = lane / S::LPR, dslot = lane % S::LPR;   // row within an instruction's, slot
  int ds = u0 / KS, dk = u0 % KS, dnext = u0;
  // shares of whole strips start 5 steps on from the share before them, equal parts of one from the strip
  // before: strips lie the same distance apart, and in step they would ask the same channels of the
  // memory at a time (28672 x 4096 in 224 whole strips 46.8 us in step, 39.6 so; 12288 x 4096 in 192
  // halves at 24 rows 28.1, 23.1; each half 5 steps on 25.5).  128-row parts that are no multiple of 4 KB apart spread by
  // themselves, and in step read x together (4096 x 14336 in 256 eighths of 3.5 KB at 24 rows 25.9, 26.7
  // turned; 8192 x 28672 at 64 rows 85.1, 86.7; of 64 rows, two on a CU, at 5 rows 88.3, 71.3 turned).
  const int seg = parts ? u1 - u0 : KS % per == 0 ? per : per % KS == 0 ? KS : 0;   // 0: other shares
  const bool turn = seg == KS || S::KC == 2 || seg * KST * 2 % 4096 == 0;
  const int seg0 = parts ? dk : seg > 0 ? dk / seg * seg : 0;
  if (seg > 0 && turn) dk = seg0 + u0 / max(per, KS) * 5 % seg;
  int left = seg;
  const uint16_t *wsrc[4], *xsrc[S::XI];
  auto aim = [&](int s) {
    const StreamStrip t = stream_strip<GRP, S::BN>(g, s);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = wave * (16 * RT) + i * S::RPI + dr;
      const int v = t.v0 + row, ch = dslot ^ S::swz(row);
      wsrc[i] = v < g.Nv ? t.b + (size_t)wrow(g, v) * g.ldb + ch * 8 : nullptr;
    }
#pragma unroll
    for (int i = 0; i < S::XI; ++i) {
      const int row = (wave % S::XW * S::XI + i) * S::RPI + dr;
      const int ch = dslot ^ S::swz(row);
      xsrc[i] = t.a + (size_t)min(row, t.M - 1) * g.lda + ch * 8;
    }
  };
  auto stage = [&](int buf) {
    uint8_t* b = smem + buf * S::STAGE;
    const bool live = dnext < u1;
    const int k = dk * KST;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = dslot ^ S::swz(wave * (16 * RT) + i * S::RPI + dr);
      const uint16_t* p = live && wsrc[i] != nullptr && k + ch * 8 < g.K ? wsrc[i] + k : g.zeros;
      __builtin_amdgcn_global_load_lds((gptr_t)p, (lptr_t)(b + (wave * 4 + i) * 1024), 16, 0, 2);
    }
    if (S::XW == NWV || wave < S::XW)
#pragma unroll
    for (int i = 0; i < S::XI; ++i) {
      const int r0 = wave * S::XI + i;
      const int ch = dslot ^ S::swz(r0 * S::RPI + dr);
      const uint16_t* p = live && k + ch * 8 < g.K ? xsrc[i] + k : g.zeros;
      glds16(p, b + (NWV * 4 + r0) * 1024);
    }
    ++dnext;
    ++dk;
    if (seg > 0) {
      if (dk == seg0 + seg) dk = seg0;
      if (--left == 0) {
        left = seg;
        ++ds;
        if (dnext < u1) aim(ds);
      }
    } else if (dk == KS) {
      dk = 0;
      ++ds;
      if (dnext < u1) aim(ds);
    }
  };
  // the step has landed; every wave has read the one before, whose stage takes the step NS - 1 ahead
  auto feed = [&](int buf) __attribute__((always_inline)) {
    if (S::XW == NWV || wave < S::XW) __builtin_amdgcn_s_waitcnt(vm_wait((S::NS - 2) * S::IPW));
    else __builtin_amdgcn_s_waitcnt(vm_wait((S::NS - 2) * 4));
    asm volatile("s_barrier" ::: "memory");
    stage(buf == 0 ? S::NS - 1 : buf - 1);
  };
  if (!ASK || who >= NWV) {
    aim(ds);
#pragma unroll
    for (int p = 0; p < S::NS - 1; ++p) stage(p);
  }
  if (ASK && who >= NWV) {
    int buf = 0;
    for (int u = u0; u < u1; ++u) {
      feed(buf);
      buf = buf + 1 == S::NS ? 0 : buf + 1;
    }
    __builtin_amdgcn_s_waitcnt(vm_wait(0));
    return;
  }
  uint32_t off[2 * KC];
#pragma unroll
  for (int h = 0; h < 2 * KC; ++h)
    off[h] = lds_off(smem) + (uint32_t)((lane & 15) * 128 * KC + ((4 * h + (lane >> 4)) ^ S::swz(lane & 15)) * 16);

  cf32x4 acc[RT][MT];
  int buf = 0, u = u0;
  while (u < u1) {
    const int s = u / KS, seg1 = min(u1, (s + 1) * KS);
#pragma unroll
    for (int j = 0; j < RT; ++j)
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[j][i] = cf32x4{0.f, 0.f, 0.f, 0.f};
    for (; u < seg1; ++u) {
      if constexpr (ASK) asm volatile("s_barrier" ::: "memory");
      else feed(buf);
      const uint32_t b = buf * S::STAGE;
      constexpr int XR = MT % 2 ? 1 : 2, T16 = 2048 * KC;   // bytes of 16 rows
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const uint32_t lo = b + off[2 * c], hi = b + off[2 * c + 1];
        uint4 w[RT][2];
        stream_read<RT, T16>(lo + wave * (RT * T16), hi + wave * (RT * T16), w);
#pragma unroll
        for (int i = 0; i < MT; i += XR) {
          uint4 x[XR][2];
          stream_read<XR, T16>(lo + (NWV * RT + i) * T16, hi + (NWV * RT + i) * T16, x);
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int p = 0; p < XR; ++p)
#pragma unroll
              for (int j = 0; j < RT; ++j) acc[j][i + p] = cmfma<DT>(w[j][h], x[p][h], acc[j][i + p]);
        }
      }
      buf = buf + 1 == S::NS ? 0 : buf + 1;
    }
    StreamStrip t = stream_strip<GRP, S::BN>(g, s);
    if constexpr (EPI == kEpiPartial) {
      t.f = g.ws + (size_t)part * g.M * g.Nv;
      t.ldf = g.Nv;
    }
    const int lo = s * KS / per, hi = ((s + 1) * KS - 1) / per;   // shares with steps of this strip
    bool mine = EPI == kEpiPartial || lo == hi;
    if (!mine) {
      auto slot = [&](int w) {   // a share's first strip, or its last
        return g.ws + ((size_t)(2 * w + (w * per / KS == s ? 0 : 1)) * NWV + wave) * (RT * MT * 256) + lane * 4;
      };
      float* p = slot(wg);
#pragma unroll
      for (int j = 0; j < RT; ++j)
#pragma unroll
        for (int i = 0; i < MT; ++i)
          if (i * 16 + (lane & 15) < t.M) park(p + (j * MT + i) * 256, acc[j][i]);
      __builtin_amdgcn_s_waitcnt(vm_wait(0));
      // (the waves of a workgroup that asks and multiplies in turn arrive as one)
      unsigned* tick = g.tick + s * NWV + (ASK ? wave : 0);
      unsigned before = 0;
      if constexpr (ASK) {
        asm volatile("" ::: "memory");
        if (lane == 0) before = __hip_atomic_fetch_add(tick, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::: "memory");
      } else {
        asm volatile("s_barrier" ::: "memory");
        if (tid == 0) last = __hip_atomic_fetch_add(tick, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        before = last;
      }
      mine = __builtin_amdgcn_readfirstlane(before) == (unsigned)(hi - lo);
      if (mine) {
        if (ASK ? lane == 0 : tid == 0) __hip_atomic_store(tick, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // in share order (the result does not hang on who came last), several shares in flight
        constexpr int UN = MT <= 2 ? 8 : 4;
        for (int w0 = lo; w0 <= hi; w0 += UN) {
          cf32x4 o[UN][RT][MT];
#pragma unroll
          for (int q = 0; q < UN; ++q) {
            const float* p = slot(min(w0 + q, hi));
#pragma unroll
            for (int j = 0; j < RT; ++j)
#pragma unroll
              for (int i = 0; i < MT; ++i)
                o[q][j][i] = i * 16 + (lane & 15) < t.M ? unpark(p + (j * MT + i) * 256) : cf32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int q = 0; q < UN; ++q)
#pragma unroll
            for (int j = 0; j < RT; ++j)
#pragma unroll
              for (int i = 0; i < MT; ++i) {
                if (q == 0 && w0 == lo) acc[j][i] = o[0][j][i];
                else if (w0 + q <= hi) acc[j][i] += o[q][j][i];
              }
        }
      }
      if constexpr (!ASK) __syncthreads();   // `last` is read
    }
    if (mine) stream_store<DT, EPI, MT, RT>(g, t, wave, lane, acc);
    // stores count with the DMA: drain them before the counted waits go on
    if (!ASK && u < u1) __builtin_amdgcn_s_waitcnt(vm_wait(0));
  }
  if constexpr (!ASK) __builtin_amdgcn_s_waitcnt(vm_wait(0));
}

template <int DT, int EPI>
int launch_stream(int mt, dim3 grid, hipStream_t st, const GemmArgs& g) {
#define CAKE_STREAM(MT)                                                                             \
  if (mt == MT) {                                                                                   \
    hipLaunchKernelGGL((gemm_stream_kernel<DT, EPI, MT, false>), grid,                              \
                       dim3(stream_threads<EPI, MT>()), 0, st, g);                                  \
    return (int)hipGetLastError();                                                                  \
  }
  CAKE_STREAM(1) CAKE_STREAM(2) CAKE_STREAM(3) CAKE_STREAM(4)
#undef CAKE_STREAM
  return (int)hipErrorInvalidValue;
}

template <int DT, int EPI>
int launch_rows(int kind, int mt, dim3 grid, hipStream_t st, const GemmArgs& g) {
  if (kind == 2) return launch_stream<DT, EPI>(mt, grid, st, g);
  constexpr bool GATED = (EPI == kEpiSwiglu || EPI == kEpiGeglu);
#define CAKE_DIRECT(KIND, MT, NT)                                                                   \
  if constexpr (!GATED || NT == 2)                                                                  \
    if (kind == KIND && mt == MT) {                                                                 \
      hipLaunchKernelGGL((gemm_direct_kernel<DT, EPI, MT, NT>), grid, dim3(512), 0, st, g);         \
      return (int)hipGetLastError();                                                                \
    }
  CAKE_DIRECT(0, 1, 1) CAKE_DIRECT(0, 2, 1) CAKE_DIRECT(1, 1, 2) CAKE_DIRECT(1, 2, 2)
#undef CAKE_DIRECT
  return (int)hipErrorInvalidValue;
}

// every epilogue of a type; grouped: rows sorted by weight group (GemmArgs::groups), tiles of at most
// 16 of them
template <int DT> struct Rows {
  static int run(int epi, int kind, int mt, dim3 grid, hipStream_t st, const GemmArgs& g) {
    switch (epi) {
#define X(E) case E: return launch_rows<DT, E>(kind, mt, grid, st, g);
      X(kEpiStore) X(kEpiResid32) X(kEpiAdd16) X(kEpiSwiglu) X(kEpiGeglu) X(kEpiStore32)
      X(kEpiSilu) X(kEpiQuick) X(kEpiGelu) X(kEpiRelu2)
#undef X
      case kEpiPartial: return launch_stream<DT, kEpiPartial>(mt, grid, st, g);
      case kEpiSections: return launch_stream<DT, kEpiSections>(mt, grid, st, g);
    }
    return (int)hipErrorInvalidValue;
  }
  static int grouped(int epi, dim3 grid, hipStream_t st, const GemmArgs& g) {
    switch (epi) {
#define X(E)                                                                                  \
  case E:                                                                                     \
    hipLaunchKernelGGL((gemm_stream_kernel<DT, E, 1, true>), grid,                            \
                       dim3(stream_threads<E, 1>()), 0, st, g);                               \
    return (int)hipGetLastError();
      X(kEpiStore) X(kEpiSilu) X(kEpiQuick) X(kEpiGelu) X(kEpiRelu2)
#undef X
    }
    return (int)hipErrorInvalidValue;
  }
};

}  // namespace cake
