// Causal attention of 128-wide heads over many rows: the part that the Llama kernel
// (flash_attn.hip) and the hybrid designs' (mixer_flash.h) share.
//
// S^T = K Q^T and O^T += V^T P^T on 32x32x16 tiles, 4 waves of 32 QS query rows, key tiles of 64;
// f32 scores, sums and output, 16-bit probabilities, maximum moved only when a tile exceeds it by
// 2^8.  What bounds it is the issue of a wave: 64 QS products of 32 cycles a tile against some
// 300 QS vector instructions of the softmax, so both are woven into one stream (a tile's softmax
// beside the next tile's score products and its own value products), one wave per SIMD with all
// 512 registers; QS 2 halves the LDS reads of a product.  Keys and values go from memory to LDS
// without registers (buffer loads with LDS destination, swizzled through their source addresses);
// row-major values are transposed by the LDS read.  One barrier per tile.
// 32 heads over 8, causal, us before (two waves a SIMD, values transposed through registers) and
// after: 777 rows 35.3 / 20.2, 1100 55 / 26, 2048 93 / 52, 6000 488 / 319 (923 TFLOP/s), 8192
// 755 / 526 (1045).
#pragma once
#include <type_traits>

#include "common.h"

namespace cake {

typedef uint32_t fu32x4 __attribute__((ext_vector_type(4)));
typedef short fs16x4 __attribute__((ext_vector_type(4)));
typedef float ff32x16 __attribute__((ext_vector_type(16)));

// The matrix instructions are written out so that the scores stay in VGPRs (the softmax reads
// them) and the output accumulators and queries in AGPRs.  What the compiler does not see then:
// 11 wait states before a VALU instruction reads a result (the products of another phase always
// lie between, or fl_settle), 2 before a product reads what a VALU instruction wrote (fl_mma_o's
// s_nop).  A register spilled beside them would be read too early: no instance may spill (build.py
// checks the compiler's remarks of each).
template <int DT>
__device__ __forceinline__ void fl_mma_s0(ff32x16& s, const uint4& k, const fu32x4& q) {
  const fu32x4 kv = __builtin_bit_cast(fu32x4, k);
  if constexpr (DT == kBF16)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s) : "v"(kv), "a"(q));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, 0" : "=&v"(s) : "v"(kv), "a"(q));
}
template <int DT>
__device__ __forceinline__ void fl_mma_s(ff32x16& s, const uint4& k, const fu32x4& q) {
  const fu32x4 kv = __builtin_bit_cast(fu32x4, k);
  if constexpr (DT == kBF16)
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s) : "v"(kv), "a"(q));
  else
    asm volatile("v_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(s) : "v"(kv), "a"(q));
}
// AG: the accumulators are in AGPRs
template <int DT, bool AG>
__device__ __forceinline__ void fl_mma_o(ff32x16& o, const uint4& v, const uint32_t (&p)[4]) {
  const fu32x4 vv = __builtin_bit_cast(fu32x4, v), pv = {p[0], p[1], p[2], p[3]};
  if constexpr (DT == kBF16 && AG)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(o) : "v"(vv), "v"(pv));
  else if constexpr (AG)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+a"(o) : "v"(vv), "v"(pv));
  else if constexpr (DT == kBF16)
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(o) : "v"(vv), "v"(pv));
  else
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_f16 %0, %1, %2, %0" : "+v"(o) : "v"(vv), "v"(pv));
}
// o's products are through
template <bool AG>
__device__ __forceinline__ void fl_settle(ff32x16& o) {
  if constexpr (AG) asm volatile("s_nop 7\n\ts_nop 7" : "+a"(o));
  else asm volatile("s_nop 7\n\ts_nop 7" : "+v"(o));
}

template <bool AG>
__device__ __forceinline__ void fl_settle(ff32x16 (&o)[4]) {
  if constexpr (AG) asm volatile("s_nop 7\n\ts_nop 7" : "+a"(o[0]), "+a"(o[1]), "+a"(o[2]), "+a"(o[3]));
  else asm volatile("s_nop 7\n\ts_nop 7" : "+v"(o[0]), "+v"(o[1]), "+v"(o[2]), "+v"(o[3]));
}

// two f32 -> packed 16-bit pair, one instruction for either type
template <int DT>
__device__ __forceinline__ uint32_t fl_cvt(float lo, float hi) {
  typedef float v2 __attribute__((ext_vector_type(2)));
  if constexpr (DT == kBF16) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2{lo, hi}), b2));
  } else {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((v2{lo, hi}), h2));
  }
}

// one KiB, 16 bytes per lane, to LDS at m0 = lds + OFF; rows past the descriptor come as zeros
template <int OFF>
__device__ __forceinline__ void fl_dma(uint32_t lds, uint32_t voff, fu32x4 d, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(lds), "v"(voff), "s"(d), "s"(soff), "i"(OFF) : "memory", "scc");
}

template <int B, int E, class F>
__device__ __forceinline__ void fl_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    fl_for<B + 1, E>(f);
  }
}

struct FlCore {
  // byte bounds are of the sequence's (head's) keys and values; rows past them read as zeros
  const uint16_t *k, *v, *r;        // keys [.][k_sn], values, rotated key part (KC 192) [.][r_sn]
  long long k_sn, v_sn, r_sn;       // VT: values [128][v_sn], else [.][v_sn]
  unsigned k_end, v_end, r_end;
  int kend, pos;                    // keys in all, position of the wave's first row
  float scale_log2;
  bool sink;                        // one more key of score 0 without a value
};

template <int KC> constexpr int fl_lds() { return 64 * 256 * 5 + (KC > 128 ? 2 * 64 * 128 : 0); }

// o[qs][t][4 g + i] = O^T[32 t + 8 g + 4 h + i][row 32 qs + lane % 32], unscaled, and the rows' sums
// DEFER: the maximum moves when a tile exceeds it by 2^8, else whenever it is exceeded (the largest
// probability is then 1 and not rounded)
template <int DT, int QS, int KC, bool VT, bool DEFER>
__device__ __forceinline__ void fl_core(uint8_t* smem, const FlCore& a,
                                        const fu32x4 (&qf)[QS][KC / 16], ff32x16 (&o)[QS][4],
                                        float (&l)[QS]) {
  constexpr int KS = KC / 16, NS = 2 * KS;  // score products per 32 keys, per tile
  constexpr int TILE = 64 * 256;            // bytes of 64 rows of 128
  constexpr int VBUF = 2 * TILE;            // two key buffers, three of values, two rotated parts
  constexpr int RBUF = 5 * TILE, RTILE = TILE / 2;
  static_assert(KC == 128 || KC == 192, "key columns");
  // without DEFER most tiles scale the output: multiplied in place in VGPRs it takes a third of
  // the instructions, and of 32 rows it fits there
  constexpr bool AG = DEFER || QS == 2;

  const int tid = threadIdx.x, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nt = (a.kend + 63) / 64;
  // Of these a wave takes the nw that some row of it sees; of the last one, with 32 rows a wave, the
  // upper 32 keys only if some row sees them (64 rows: the branch spills).  A product with
  // probability 0 would still carry a later key's infinite or NaN value into this row.
  const int seen = min(a.kend - 1, a.pos + 32 * QS - 1);
  const int nw = max(1, (seen >> 6) + 1);
  const bool upper = (seen & 63) >= 32;

  // staging of [.][128] rows: instruction i of a wave fills rows 16 i + 4 wave + lane / 16, 16-byte
  // slot lane % 16.  Slot s of a key row r holds chunk s ^ (r & 15) (a fragment read takes the same
  // chunk of 32 rows), of a value row chunk s ^ 4 (r & 3) (a transposed read takes 64 bytes of 4
  // rows).  Of [.][64] rows (rotated part, transposed values): rows 32 i + 8 wave + lane / 8, slot
  // lane % 8 with chunk slot ^ (r / 2 & 7).
  const int r4 = lane >> 4, slot = lane & 15;
  const uint32_t kvoff = (uint32_t)((wave * 4 + r4) * a.k_sn * 2) + ((slot ^ (wave * 4 + r4)) * 16);
  const uint32_t half = (uint32_t)(((lane & 7) ^ ((wave * 4 + r4) & 7)) * 16);
  const int row8 = wave * 8 + (lane >> 3);
  const uint32_t vvoff = VT ? (uint32_t)(row8 * a.v_sn * 2) + half
                            : (uint32_t)((wave * 4 + r4) * a.v_sn * 2) + ((slot ^ (r4 * 4)) * 16);
  const uint32_t rvoff = (uint32_t)(row8 * a.r_sn * 2) + half;
  const uint32_t krow16 = (uint32_t)(a.k_sn * 32), vrow16 = (uint32_t)(a.v_sn * 32),
                 rrow16 = (uint32_t)(a.r_sn * 32);
  const uint32_t lds_w = __builtin_amdgcn_readfirstlane(lds_off(smem)) + (uint32_t)wave * 1024;
  auto desc = [&](const uint16_t* p, unsigned end, int j) __attribute__((always_inline)) {
    const unsigned long long u = (unsigned long long)p;
    fu32x4 d;
    d[0] = __builtin_amdgcn_readfirstlane((unsigned)u);
    d[1] = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32) & 0xFFFFu);
    d[2] = __builtin_amdgcn_readfirstlane(j < nt ? end : 0u);   // past the last tile: no traffic
    d[3] = 0x00020000u;
    return d;
  };
  auto stage_k = [&](int j) __attribute__((always_inline)) {
    const fu32x4 d = desc(a.k, a.k_end, j);
    const uint32_t to = lds_w + (j & 1) * TILE, so = (uint32_t)j * 4 * krow16;
    fl_for<0, 4>([&](auto I) __attribute__((always_inline)) {
      fl_dma<I * 4096>(to, kvoff, d, so + I * krow16);
    });
    if constexpr (KC == 192) {
      const fu32x4 e = desc(a.r, a.r_end, j);
      const uint32_t rt = lds_w + RBUF + (j & 1) * RTILE, ro = (uint32_t)j * 4 * rrow16;
      fl_for<0, 2>([&](auto I) __attribute__((always_inline)) {
        fl_dma<I * 4096>(rt, rvoff, e, ro + I * 2 * rrow16);
      });
    }
  };
  auto stage_v = [&](int j, int buf) __attribute__((always_inline)) {
    const fu32x4 d = desc(a.v, a.v_end, j);
    const uint32_t to = lds_w + VBUF + buf * TILE;
    const uint32_t so = VT ? (uint32_t)j * 128 : (uint32_t)j * 4 * vrow16;
    fl_for<0, 4>([&](auto I) __attribute__((always_inline)) {
      fl_dma<I * 4096>(to, vvoff, d, so + (VT ? 2 * I : I) * vrow16);
    });
  };
  const auto landed = [] __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  };

  // fragment addresses.  Keys: row 32 t + l32, chunk 2 ks + h.  Values, column 32 dt + l32 of keys
  // 32 t + 16 s2 + 4 h .. and 8 on: row-major by transposing reads of 4 rows x 64 bytes a half wave
  // (lane i of 16 gets column i), transposed ones by two 8-byte reads of a row.
  const uint32_t kl = (uint32_t)l32 * 256, kx = (uint32_t)((h ^ (l32 & 15)) * 16);
  const uint32_t rl = (uint32_t)l32 * 128, rx = (uint32_t)((h ^ ((l32 >> 1) & 7)) * 16);
  uint32_t va[4];
#pragma unroll
  for (int c = 0; c < 4; ++c)
    va[c] = VBUF + (VT ? l32 * 128 + 8 * h + (uint32_t)(((2 * c) ^ ((l32 >> 1) & 7)) * 16)
                       : (4 * h + ((lane & 15) >> 2)) * 256 + 64 * (c ^ ((lane & 15) >> 2)) +
                             32 * ((lane >> 4) & 1) + 8 * (lane & 3));
  auto kfrag = [&](int buf, auto I) __attribute__((always_inline)) {  // i = KS t + ks
    constexpr int t = decltype(I)::value / KS, ks = decltype(I)::value % KS;
    if constexpr (ks < 8)
      return *reinterpret_cast<const uint4*>(smem + buf * TILE + (kl + (kx ^ (32 * ks))) + t * 8192);
    else
      return *reinterpret_cast<const uint4*>(smem + RBUF + buf * RTILE +
                                             (rl + (rx ^ (32 * (ks - 8)))) + t * 4096);
  };
  typedef __attribute__((address_space(3))) fs16x4 lds_s4;
  auto vfrag = [&](uint32_t vbuf, auto I) __attribute__((always_inline)) {  // i = 8 t + 4 s2 + dt
    constexpr int c = decltype(I)::value >> 2, dt = decltype(I)::value & 3;
    if constexpr (VT) {
      const uint2 l = *reinterpret_cast<const uint2*>(smem + (vbuf + va[c]) + dt * 4096);
      const uint2 u = *reinterpret_cast<const uint2*>(smem + ((vbuf + va[c]) ^ 16) + dt * 4096);
      return make_uint4(l.x, l.y, u.x, u.y);
    } else {
      const uint8_t* p = smem + (vbuf + va[dt]) + c * 4096;
      const fs16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
      const fs16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + 2048));
      const uint2 l = __builtin_bit_cast(uint2, lo), u = __builtin_bit_cast(uint2, hi);
      return make_uint4(l.x, l.y, u.x, u.y);
    }
  };

#pragma unroll
  for (int qs = 0; qs < QS; ++qs)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[qs][t][r] = 0.f;
      fl_settle<AG>(o[qs][t]);
    }
  float m[QS];
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    m[qs] = a.sink ? 0.f : -INFINITY;
    l[qs] = a.sink && h == 0 ? 1.f : 0.f;
  }

  constexpr int PF = 3, RG = 4;   // fragments read ahead, ring
  constexpr float kGrow = 8.f;    // log2 units
  ff32x16 sa[QS][2], sb[QS][2];
  auto score = [&](auto I, ff32x16 (&s)[QS][2], const uint4& kf) __attribute__((always_inline)) {
    constexpr int t = decltype(I)::value / KS, ks = decltype(I)::value % KS;
    fl_for<0, QS>([&](auto Q) __attribute__((always_inline)) {
      if constexpr (ks == 0) fl_mma_s0<DT>(s[Q][t], kf, qf[Q][ks]);
      else fl_mma_s<DT>(s[Q][t], kf, qf[Q][ks]);
    });
  };

  stage_k(0);
  stage_v(0, 0);
  stage_k(1);
  landed();
  uint4 kf[RG];
  fl_for<0, PF>([&](auto I) __attribute__((always_inline)) { kf[I] = kfrag(0, I); });
  fl_for<0, NS>([&](auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    if constexpr (i + PF < NS) kf[(i + PF) % RG] = kfrag(0, std::integral_constant<int, i + PF>{});
    score(I, sa, kf[i % RG]);
    __builtin_amdgcn_sched_barrier(0);
  });
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
  landed();   // every wave has read the first key tile
  stage_k(2);
  stage_v(1, 1);
  fl_for<0, PF>([&](auto I) __attribute__((always_inline)) { kf[I] = kfrag(1, I); });

  // Tile j: its softmax beside the score products of tile j + 1, its value products beside the
  // softmax's second half.  Past the middle of those everything read a tile ago is done with and
  // everything requested a tile ago has landed: the barrier, then the next requests.
  int vbuf = 0;   // buffer of tile j's values
  auto tile = [&](auto QK, int j, ff32x16 (&s)[QS][2], ff32x16 (&n)[QS][2])
                  __attribute__((always_inline)) {
    constexpr bool qk = decltype(QK)::value;
    const uint32_t vb = (uint32_t)vbuf * TILE;
    if (j * 64 + 64 > a.kend || j * 64 + 63 > a.pos) {
#pragma unroll
      for (int qs = 0; qs < QS; ++qs) {
        // last key that this row sees, from this lane's first of the tile
        const int lim = min(a.kend - 1, a.pos + 32 * qs + l32) - (j * 64 + 4 * h);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            s[qs][t][r] = 32 * t + (r & 3) + 8 * (r >> 2) > lim ? -INFINITY : s[qs][t][r];
      }
    }
    float mq[QS][4], mc[QS], rq[QS][4], al[QS];
    uint32_t pf[QS][4][4];
    uint4 vf[RG];
    bool grow = false;
    // probabilities of 2 QS scores of half t: slice c of 8
    auto probs = [&](auto T, auto Cc) __attribute__((always_inline)) {
      constexpr int t = decltype(T)::value, c = decltype(Cc)::value;
      fl_for<0, QS>([&](auto W) __attribute__((always_inline)) {
        constexpr int v = (c * QS + decltype(W)::value) * 2, qs = v / 16, r = v % 16;
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[qs][t][r], a.scale_log2, -mc[qs]));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[qs][t][r + 1], a.scale_log2, -mc[qs]));
        rq[qs][r & 3] += p0;
        rq[qs][(r & 3) + 1] += p1;
        pf[qs][2 * t + r / 8][(r % 8) / 2] = fl_cvt<DT>(p0, p1);
      });
    };
    const int kb = (j + 1) & 1;
    fl_for<0, NS>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if constexpr (qk) {
        if constexpr (i + PF < NS)
          kf[(i + PF) % RG] = kfrag(kb, std::integral_constant<int, i + PF>{});
        score(I, n, kf[i % RG]);
      }
      if constexpr (i + PF >= NS)
        vf[i + PF - NS] = vfrag(vb, std::integral_constant<int, i + PF - NS>{});
      if constexpr (i < 4) {           // row maxima: 16 scores a step (QS 2), 8 (QS 1)
#pragma unroll
        for (int e = 0; e < 8 * QS; ++e) {
          const int v = i * 8 * QS + e, qs = v / 32, t = (v / 16) % 2, r = v % 16;
          mq[qs][r & 3] = v % 32 < 4 ? s[qs][t][r] : fmaxf(mq[qs][r & 3], s[qs][t][r]);
        }
      } else if constexpr (i == 4) {
#pragma unroll
        for (int qs = 0; qs < QS; ++qs) {
          float mt = fmaxf(fmaxf(mq[qs][0], mq[qs][1]), fmaxf(mq[qs][2], mq[qs][3]));
          const int bi = __builtin_bit_cast(int, mt);
          const auto sw = __builtin_amdgcn_permlane32_swap(bi, bi, false, false);
          mt = fmaxf(__builtin_bit_cast(float, (int)sw[0]), __builtin_bit_cast(float, (int)sw[1]));
          const bool g = DEFER ? m[qs] == -INFINITY || (mt - m[qs]) * a.scale_log2 > kGrow
                               : mt > m[qs];
          const float mn = g ? fmaxf(m[qs], mt) : m[qs];
          mc[qs] = mn == -INFINITY ? 0.f : mn * a.scale_log2;
          al[qs] = g ? __builtin_amdgcn_exp2f(m[qs] * a.scale_log2 - mc[qs]) : 1.f;
          m[qs] = mn;
          grow |= g;
#pragma unroll
          for (int c = 0; c < 4; ++c) rq[qs][c] = 0.f;
        }
      } else if constexpr (i == 5) {
        if (__builtin_amdgcn_ballot_w64(grow) != 0ull) {
          fl_for<0, QS>([&](auto Q) __attribute__((always_inline)) {
            l[Q] *= al[Q];
            fl_for<0, 4>([&](auto T) __attribute__((always_inline)) {
              fl_settle<AG>(o[Q][T]);
#pragma unroll
              for (int r = 0; r < 16; ++r) o[Q][T][r] *= al[Q];
              if constexpr (AG) asm volatile("s_nop 1" : "+a"(o[Q][T]));  // back to its registers
            });
          });
        }
      } else if constexpr (i < 14) {
        probs(std::integral_constant<int, 0>{}, std::integral_constant<int, i - 6>{});
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    const auto values = [&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      if constexpr (i + PF < 16)
        vf[(i + PF) % RG] = vfrag(vb, std::integral_constant<int, i + PF>{});
      fl_for<0, QS>([&](auto Q) __attribute__((always_inline)) {
        fl_mma_o<DT, AG>(o[Q][i % 4], vf[i % RG], pf[Q][i / 4]);
      });
      if constexpr (i < 8) probs(std::integral_constant<int, 1>{}, I);
      if constexpr (i == 9 && qk) {
        landed();
        stage_k(j + 3);
        stage_v(j + 2, vbuf == 0 ? 2 : vbuf - 1);
      }
      if constexpr (qk && i + PF >= 16)
        kf[i + PF - 16] = kfrag(j & 1, std::integral_constant<int, i + PF - 16>{});
      __builtin_amdgcn_sched_barrier(0);
    };
    fl_for<0, 8>(values);
    if constexpr (qk || QS == 2) {
      fl_for<8, 16>(values);
    } else {
      // settled on either side of the branch: a register may be copied there
      fl_settle<AG>(o[0]);
      if (upper) {
        fl_for<8, 16>(values);
        fl_settle<AG>(o[0]);
      }
    }
#pragma unroll
    for (int qs = 0; qs < QS; ++qs)
      l[qs] += (rq[qs][0] + rq[qs][1]) + (rq[qs][2] + rq[qs][3]);
    vbuf = vbuf == 2 ? 0 : vbuf + 1;
    asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");  // copies at the tile's end read the results
  };
  const std::true_type more{};
  const std::false_type last{};
  int j = 0;
  for (; j + 2 < nw; j += 2) {
    tile(more, j, sa, sb);
    tile(more, j + 1, sb, sa);
  }
  if (j + 1 < nw) {
    tile(more, j, sa, sb);
    tile(last, j + 1, sb, sa);
  } else {
    tile(last, j, sa, sb);
  }
  // the barriers and requests of tiles that only later rows see (vbuf: tile i's values)
  for (int i = nw; i < nt; ++i) {
    landed();
    stage_k(i + 2);
    vbuf = vbuf == 2 ? 0 : vbuf + 1;
    stage_v(i + 1, vbuf);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // requests of tiles that are not there
#pragma unroll
  for (int qs = 0; qs < QS; ++qs) {
    l[qs] += __shfl_xor(l[qs], 32, 64);
    fl_settle<AG>(o[qs]);
  }
}

}  // namespace cake
