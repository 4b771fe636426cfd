// One token of a parallel layer: the mixer, and beside it the feed-forward's up rows.
//
// Both read the projections' norm and neither the other.  The mixer is a chain of round trips on one
// workgroup per head (attention 8.4 us at 230 keys, delta rule 6.8 at 16 heads of 128, whatever the rest of the
// chip does), the up rows are bytes (46 MB at a width of 2048, 9.6 us): in one launch the first workgroups run the mixer
// and the others stream the rows meanwhile, so that the mixer's time is paid by neither.  The launch in front
// is left with the mixer's own rows.  Of 16 heads: attention 10.8 us, delta rule 10.7, rows included.
#include "mixer_attn_decode.h"
#include "mixer_delta_decode.h"
#include "mixer_gemv.h"

namespace cake {

// grid: the mixer's nmix workgroups, which have the longest chain and so start first, then the rows'.
// The attention's registers (162 a lane at heads of 128) leave three waves a SIMD, so the rows have four pieces of
// each row of a pair in flight where the launch of their own has two.
template <int DT, int CLS, int NW, int NX>
__global__ __launch_bounds__(64 * NW, NW == 8 ? 2 : 3) void mixer_beside_attn_kernel(MixDecArgs a, MixInArgs u,
                                                                                     int tiles) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nmix = tiles * a.nsplit, bx = blockIdx.x;
  if (bx < nmix)
    mixer_attn_decode_body<DT, CLS, true, NW>(a, *reinterpret_cast<MixDecLds<DT, CLS, NW>*>(smem), bx % tiles,
                                              tiles, bx / tiles, 0);
  else
    mixer_in_rows<DT, 4, 4, NX, 64 * NW>(u, bx - nmix, gridDim.x - nmix, reinterpret_cast<float*>(smem));
}

template <int DT, int RPT, int NX>
__global__ __launch_bounds__(kDdThreads, 4) void mixer_beside_delta_kernel(DeltaArgs a, MixInArgs u) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int bx = blockIdx.x;
  if (bx < a.H)
    mixer_delta_decode_body<DT, RPT>(a, *reinterpret_cast<DeltaDecLds*>(smem), bx, 0);
  else
    mixer_in_rows<DT, 4, 4, NX, kDdThreads>(u, bx - a.H, gridDim.x - a.H, reinterpret_cast<float*>(smem));
}

// the widths whose rows lie in registers while the norm is taken (NormPre, prefetch of 4 x 64 pieces)
static bool beside_rows_ok(const MixInArgs& u) {
  return u.K % 8 == 0 && u.K >= 2048 && u.K <= 8192 && u.Kn >= 1 && u.Kn <= u.K && u.N > 0 && u.resid && u.norm_w &&
         u.w && u.act && u.actf >= 0 && u.actf < kMixActs;
}

// the mixer's workgroups and the rows', as many as fit on 256 units beside them at `waves` a unit
static int beside_grid(int nmix, int threads, int waves, int N) {
  const int per = threads / 64, room = 256 * waves / per - nmix, least = 64, g = ((N + 1) / 2 + per - 1) / per;
  const int most = room > least ? room : least;
  return nmix + (g < most ? g : most);
}

template <class Kern, class... Args>
static int launch_beside(Kern k, int grid, int threads, size_t lds, hipStream_t st, const Args&... args) {
  if (!allow_lds(k, lds)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL(k, dim3(grid), dim3(threads), lds, st, args...);
  return (int)hipGetLastError();
}

template <int DT, int CLS, int NW>
static int launch_beside_attn(const MixDecArgs& a, const MixInArgs& u, int tiles, hipStream_t st) {
  const size_t own = sizeof(MixDecLds<DT, CLS, NW>), xs = (size_t)u.K * 4, lds = own > xs ? own : xs;
  const int grid = beside_grid(tiles * a.nsplit, 64 * NW, 8, u.N);
  // a thread holds NX pieces of four columns of the normed row
  if (u.K <= 4096)
    return launch_beside(mixer_beside_attn_kernel<DT, CLS, NW, 16 / NW>, grid, 64 * NW, lds, st, a, u, tiles);
  return launch_beside(mixer_beside_attn_kernel<DT, CLS, NW, 32 / NW>, grid, 64 * NW, lds, st, a, u, tiles);
}

// Eight waves make the attention's chain shorter (a wave per row of the prologue, 256 keys at once), four leave
// more units to the rows where many splits run it.  Rows of 64 MB take as long as the longest chain.  16 heads of
// 128 on 4 key heads beside 46 MB, at 100 / 230 / 900 / 3000 keys: 10.7 / 10.8 / 11.8 / 13.5 us with eight waves,
// 11.5 / 12.9 / 14.3 / 17.1 with four (attention alone 6.5 / 8.4 / 9.9 / 12.9, rows alone 9.6); 32 on 8 beside 159
// MB: 27.1 / 26.6 / 28.2 / 32.2 and 26.5 / 26.5 / 27.0 / 28.4 (6.5 / 8.3 / 10.3 / 13.6, 27.8).
template <int DT, int CLS>
static int beside_attn(const MixDecArgs& a, const MixInArgs& u, int tiles, hipStream_t st) {
  return (long long)u.N * u.K * 2 < (64 << 20) ? launch_beside_attn<DT, CLS, 8>(a, u, tiles, st)
                                               : launch_beside_attn<DT, CLS, 4>(a, u, tiles, st);
}

template <int DT, int RPT>
static int beside_delta(const DeltaArgs& a, const MixInArgs& u, hipStream_t st) {
  const size_t own = sizeof(DeltaDecLds), xs = (size_t)u.K * 4, lds = own > xs ? own : xs;
  const int grid = beside_grid(a.H, kDdThreads, 16, u.N);
  if (u.K <= 4096) return launch_beside(mixer_beside_delta_kernel<DT, RPT, 2>, grid, kDdThreads, lds, st, a, u);
  return launch_beside(mixer_beside_delta_kernel<DT, RPT, 4>, grid, kDdThreads, lds, st, a, u);
}

}  // namespace cake

using namespace cake;

// cake_mixer_attn_decode of one row (heads of 64 or 128 for keys and values alike), and act [N] =
// actf(w norm(resid)) for the layer's up rows w [N][K]
CAKE_API int cake_mixer_beside_attn(int dt, const float* proj, const int* pos, const int* slot, const void* cs,
                                    int rd2, int qk_norm, int sink, int gated, float eps, float scale, void* kc,
                                    void* vc, long long k_slot, long long v_slot, void* out, int H, int G, int dim,
                                    int vdim, int DP, int DVP, int S, int nsplit, float* part, unsigned int* ticket,
                                    const float* resid, const void* norm_w, float norm_eps, float off, int ln, int Kn,
                                    const void* w, int K, int N, int actf, void* act, hipStream_t st) {
  const MixInArgs u{resid, (const uint16_t*)norm_w, (const uint16_t*)w, nullptr, nullptr, (uint16_t*)act, norm_eps,
                    off, ln, Kn, K, N, 0, actf};
  if (!mix_shape_ok(H, G, dim, vdim, DP, DVP, S, rd2) || DP != DVP || !(DP == 64 || DP == 128) || nsplit < 1 ||
      nsplit > 64 || !beside_rows_ok(u))
    return (int)hipErrorInvalidValue;
  MixDecArgs a{proj, 0, pos, slot, (const float2*)cs, rd2, qk_norm, sink, gated, eps, scale * 1.4426950408889634f,
               kc, vc, k_slot, v_slot, out, 0, H, G, dim, vdim, DP, DVP, S, nsplit, part, ticket};
  const int tiles = G * ((H / G + 15) / 16);
  if (tiles > 256) return (int)hipErrorInvalidValue;
  a.nsplit = mix_dec_splits(tiles, nsplit);
  DISPATCH_DT(dt, return DP == 128 ? beside_attn<DT, 128>(a, u, tiles, st) : beside_attn<DT, 64>(a, u, tiles, st));
}

// the same for cake_mixer_delta_decode of one row, up to eight rows of a head's state per thread
CAKE_API int cake_mixer_beside_delta(int dt, const float* proj, const float* ab, int H, int G, int dim, int vdim,
                                     int EP, int taps, float eps, const float* conv, const float* a_log,
                                     const float* dt_bias, const float* gate_w, float* state, float* ring,
                                     long long s_slot, long long r_slot, const int* pos, const int* slot, void* out,
                                     const float* resid, const void* norm_w, float norm_eps, float off, int ln,
                                     int Kn, const void* w, int K, int N, int actf, void* act, hipStream_t st) {
  const MixInArgs u{resid, (const uint16_t*)norm_w, (const uint16_t*)w, nullptr, nullptr, (uint16_t*)act, norm_eps,
                    off, ln, Kn, K, N, 0, actf};
  if (!delta_shape_ok(H, G, dim, vdim, EP, taps) || H > 256 || !beside_rows_ok(u)) return (int)hipErrorInvalidValue;
  DeltaArgs a{};
  a.proj = proj; a.ab = ab; a.N = 1; a.H = H; a.G = G; a.dim = dim; a.vdim = vdim; a.EP = EP; a.taps = taps;
  a.eps = eps; a.conv = conv; a.a_log = a_log; a.dt_bias = dt_bias; a.norm_w = gate_w; a.state = state;
  a.ring = ring; a.s_slot = s_slot; a.r_slot = r_slot; a.row_pos = pos; a.row_slot = slot; a.out = out;
  const int ng = kDdThreads / (EP / 4), rpt = (dim + ng - 1) / ng;
  if (rpt > 8) return (int)hipErrorInvalidValue;
  DISPATCH_DT(dt, return rpt <= 4 ? beside_delta<DT, 4>(a, u, st) : beside_delta<DT, 8>(a, u, st));
}
