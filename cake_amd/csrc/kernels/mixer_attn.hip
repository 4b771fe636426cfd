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
#include "mixer_attn_decode.h"
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

template <int DT, int CLS, bool EXACT, int NW>
__global__ __launch_bounds__(64 * NW) void mixer_attn_decode_kernel(MixDecArgs a) {
  __shared__ MixDecLds<DT, CLS, NW> s;
  mixer_attn_decode_body<DT, CLS, EXACT, NW>(a, s, blockIdx.x, gridDim.x, blockIdx.y, blockIdx.z);
}

}  // namespace cake

using namespace cake;

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
  a.nsplit = mix_dec_splits((long long)grid.x * grid.z, a.nsplit);
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
