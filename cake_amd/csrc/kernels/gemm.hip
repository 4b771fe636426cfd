// MFMA GEMM for every T > 1 linear layer: y = x W^T (+ fused epilogue).
//
// Replaces the reference's candle Linear -> cuBLAS gemm for the Llama prefill
// projections (cake-core/src/models/llama3/attention.rs:49-60 q/k/v, :120 o;
// mlp.rs:14-18 gate/up/down) and every Stable Diffusion / CLIP linear
// (candle-transformers stable_diffusion attention/FF/proj layers reached from
// cake-core/src/models/sd/{unet,vae,clip}.rs).
//
//   A = x [M][K] (activations, row stride lda), B = W [N][K] (HF weight layout,
//   row stride ldb): both operands are k-contiguous, so every MFMA fragment is
//   one 16-byte LDS read.  f32 accumulation on v_mfma_f32_16x16x32_{bf16,f16}.
//
// Structure (gfx950):
//   * Workgroup tile BM x BN x 64, 256 threads = WM x WN waves, per-wave tile
//     (BM/WM) x (BN/WN) as FM x FN 16x16 MFMA tiles.
//   * Operands staged global -> LDS by LDS-DMA (global_load_lds_dwordx4, no
//     VGPR round trip) into two buffers; the DMA of k-step t+2 is in flight
//     while step t computes.  The 128-byte rows are XOR-swizzled in 16-byte
//     slots (slot ^= (row >> 1) & 7) on the SOURCE address (the DMA writes
//     lane-linear), which makes the fragment ds_read_b128 conflict-free.
//   * Fragment reads are inline-asm ds_read_b128 with an explicit lgkmcnt wait:
//     hipcc cannot see them, so it does not drain the in-flight DMA (vmcnt(0))
//     in front of them, which it does for compiler-visible LDS reads of a
//     buffer a DMA may write.  Waits on the DMA are counted (vmcnt(N)) and the
//     barriers are raw s_barrier (MI355X guide: "Pipelining across barriers").
//   * XCD-aware grouped tile order: round-robin block -> XCD dealing is undone
//     so each XCD's blocks cover a compact group of tiles (shared A rows / W
//     rows hit that XCD's L2).
//   * Split-K (grid.y) for grids smaller than the chip: f32 partial slabs and
//     a second kernel that reduces them and applies the epilogue.
//   * Epilogues (C staged through LDS per 16-row strip, 16-32 byte vector
//     stores): plain store (+bias), f32 residual accumulate (Llama o/down
//     proj: resid += y), 16-bit add (+bias, +residual: SD proj_out), SwiGLU
//     (silu(gate) * up from the fused gate|up weight) and GEGLU
//     (h * gelu_tanh(gate), SD FeedForward).  For the gated forms the B rows
//     are read in a virtual order that interleaves 16-row blocks of the two
//     halves, so gate and up of one feature land in the same lane.
#include "gemm_kernel.h"
#include "gemm_rows.h"

#include <algorithm>
#include <cmath>

namespace cake {
// the launchers are instantiated in gemm_inst_{bf16,f16}_{a,b,c}.hip
#define CAKE_GEMM_EXTERN(DT, E) extern template int launch_gemm<DT, E>(int, dim3, hipStream_t, const GemmArgs&);
#define CAKE_GEMM_EXTERN_ALL(DT) CAKE_GEMM_EXTERN(DT, kEpiStore) CAKE_GEMM_EXTERN(DT, kEpiResid32) \
  CAKE_GEMM_EXTERN(DT, kEpiAdd16) CAKE_GEMM_EXTERN(DT, kEpiSwiglu) CAKE_GEMM_EXTERN(DT, kEpiGeglu) \
  CAKE_GEMM_EXTERN(DT, kEpiPartial) CAKE_GEMM_EXTERN(DT, kEpiStore32) CAKE_GEMM_EXTERN(DT, kEpiSilu) \
  CAKE_GEMM_EXTERN(DT, kEpiQuick) CAKE_GEMM_EXTERN(DT, kEpiGelu) CAKE_GEMM_EXTERN(DT, kEpiRelu2)
CAKE_GEMM_EXTERN_ALL(kBF16)
CAKE_GEMM_EXTERN_ALL(kF16)
#undef CAKE_GEMM_EXTERN_ALL
#undef CAKE_GEMM_EXTERN
// ... and in gemm_inst_pieces_{bf16,f16}_{a,b}.hip
#define CAKE_PIECES_EXTERN(DT, E) extern template int launch_pieces<DT, E>(int, dim3, hipStream_t, const GemmArgs&);
#define CAKE_PIECES_EXTERN_ALL(DT) CAKE_PIECES_EXTERN(DT, kEpiStore) CAKE_PIECES_EXTERN(DT, kEpiResid32) \
  CAKE_PIECES_EXTERN(DT, kEpiAdd16) CAKE_PIECES_EXTERN(DT, kEpiSwiglu) CAKE_PIECES_EXTERN(DT, kEpiGeglu) \
  CAKE_PIECES_EXTERN(DT, kEpiStore32) CAKE_PIECES_EXTERN(DT, kEpiSilu) CAKE_PIECES_EXTERN(DT, kEpiQuick) \
  CAKE_PIECES_EXTERN(DT, kEpiGelu) CAKE_PIECES_EXTERN(DT, kEpiRelu2)
CAKE_PIECES_EXTERN_ALL(kBF16)
CAKE_PIECES_EXTERN_ALL(kF16)
#undef CAKE_PIECES_EXTERN_ALL
#undef CAKE_PIECES_EXTERN
// ... and in gemm_inst_rows_{bf16,f16}.hip
#define CAKE_ROWS_EXTERN(DT)                                                                      \
  extern template struct Rows<DT>;
CAKE_ROWS_EXTERN(kBF16)
CAKE_ROWS_EXTERN(kF16)
#undef CAKE_ROWS_EXTERN
}  // namespace cake

using namespace cake;

extern "C" int cake_gemm_grouped(int dt, int epi, int cfg, const void* a, long long lda,
                                 const void* b, long long ldb, long long b_group, void* c,
                                 long long ldc, const void* tiles, int max_tiles,
                                 const void* zeros, int N, int K, hipStream_t st);

// Which capture records the stream's launches: 0 none, else an id of that capture, -1 an error.
CAKE_API long long cake_stream_capture(hipStream_t st) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  unsigned long long id = 0;
  if (hipStreamGetCaptureInfo(st, &status, &id) != hipSuccess) return -1;
  return status == hipStreamCaptureStatusNone ? 0 : (long long)(id + 1);
}

static inline void cfg_dims(int cfg, int& bm, int& bn) {
  if (cfg == kPPCfg || cfg == kRSCfg) { bm = bn = 256; return; }
  if (cfg >= k4WCfg + k4WSched && cfg <= k4WCfg128 + k4WSched) cfg -= k4WSched;   // the same tiles
  if (cfg == k4WCfg) { bm = bn = 256; return; }
  if (cfg == k4WCfg192) { bm = 256; bn = 192; return; }
  if (cfg == k4WCfg128) { bm = 128; bn = 256; return; }
#define X(id, BM, BN, WM, WN, SCHED) if (cfg == id) { bm = BM; bn = BN; return; }
  CAKE_GEMM_4W_TILES(X)
#undef X
#define X(id, BM, BN, WM, WN, NS, PR) if (cfg == id) { bm = BM; bn = BN; return; }
  CAKE_GEMM_CFGS(X)
#undef X
  bm = bn = 0;
}

CAKE_API int cake_gemm_tile(int cfg, int* bm, int* bn) {
  cfg_dims(cfg, *bm, *bn);
  return *bm > 0 ? 0 : (int)hipErrorInvalidValue;
}

// the gated epilogues pair 16-column gate / up blocks inside one wave: 32-column multiples
template <int DT>
static int dispatch_epi(int epi, int cfg, dim3 grid, hipStream_t st, const GemmArgs& g) {
  if (g.pieces > 0) {
    switch (epi) {
#define P(E) case E: return launch_pieces<DT, E>(cfg, grid, st, g);
      P(kEpiStore) P(kEpiResid32) P(kEpiAdd16) P(kEpiSwiglu) P(kEpiGeglu) P(kEpiStore32)
      P(kEpiSilu) P(kEpiQuick) P(kEpiGelu) P(kEpiRelu2)
#undef P
    }
    return (int)hipErrorInvalidValue;
  }
  switch (epi) {
    case kEpiStore: return launch_gemm<DT, kEpiStore>(cfg, grid, st, g);
    case kEpiResid32: return launch_gemm<DT, kEpiResid32>(cfg, grid, st, g);
    case kEpiAdd16: return launch_gemm<DT, kEpiAdd16>(cfg, grid, st, g);
    case kEpiSwiglu: return launch_gemm<DT, kEpiSwiglu>(cfg, grid, st, g);
    case kEpiGeglu: return launch_gemm<DT, kEpiGeglu>(cfg, grid, st, g);
    case kEpiPartial: return launch_gemm<DT, kEpiPartial>(cfg, grid, st, g);
    case kEpiStore32: return launch_gemm<DT, kEpiStore32>(cfg, grid, st, g);
    case kEpiSilu: return launch_gemm<DT, kEpiSilu>(cfg, grid, st, g);
    case kEpiQuick: return launch_gemm<DT, kEpiQuick>(cfg, grid, st, g);
    case kEpiGelu: return launch_gemm<DT, kEpiGelu>(cfg, grid, st, g);
    case kEpiRelu2: return launch_gemm<DT, kEpiRelu2>(cfg, grid, st, g);
  }
  return (int)hipErrorInvalidValue;
}

template <int DT>
static int dispatch_finalize(int epi, dim3 grid, hipStream_t st, const GemmArgs& g, int splits) {
  switch (epi) {
#define F(E) case E: hipLaunchKernelGGL((gemm_splitk_finalize<DT, E>), grid, dim3(256), 0, st, g, splits); break;
    F(kEpiStore) F(kEpiResid32) F(kEpiAdd16) F(kEpiSwiglu) F(kEpiGeglu) F(kEpiStore32)
    F(kEpiSilu) F(kEpiQuick) F(kEpiGelu) F(kEpiRelu2)
#undef F
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

// Split plan of one call: the k split actually run (whole 64-element steps per split) and, for a
// four-wave tile, its pieces instead: the tiles past the last whole wave of 256 (all of them when
// there are no more) in `splits` pieces each, or as many as one wave of 256 holds.
// cake_gemm and cake_gemm_ws_floats both decide through this one function, so a workspace sized
// by the query always covers the launch.
struct SplitPlan {
  int splits, kps, bm, bn, ntiles;
  int rest, pieces;   // tiles that run in pieces (0: none), pieces of each
};
static SplitPlan split_plan(int cfg, int splits, int M, long long Nv, int K) {
  SplitPlan p{};
  cfg_dims(cfg, p.bm, p.bn);
  if (p.bm != 0) p.ntiles = (int)(((M + p.bm - 1) / p.bm) * ((Nv + p.bn - 1) / p.bn));
  const bool four = p.bm != 0 && four_wave_cfg(cfg);
  const int rest = p.ntiles <= 256 ? p.ntiles : p.ntiles % 256;
  if (four) splits = rest > 0 ? std::max(1, std::min(splits, 256 / rest)) : 1;
  int kps = (K + splits - 1) / splits;
  kps = (kps + kGBK - 1) / kGBK * kGBK;
  p.kps = kps;
  p.splits = (K + kps - 1) / kps;
  if (four && p.splits > 1) {
    p.rest = rest;
    p.pieces = p.splits;
    p.splits = 1;
  }
  return p;
}

// f32 workspace (elements) a cake_gemm call with these arguments needs: the pieces' slabs
// (BM x BN each) or splits x M x Nv partial rows, 0 when it runs unsplit
CAKE_API long long cake_gemm_ws_floats(int cfg, int splits, int M, int N, int K, int gated) {
  if (splits < 1 || M <= 0 || N <= 0 || K <= 0) return 0;
  const long long Nv = gated ? 2LL * N : N;
  const SplitPlan p = split_plan(cfg, splits, M, Nv, K);
  if (p.pieces > 0) return (long long)p.rest * p.pieces * p.bm * p.bn;
  return p.splits > 1 ? (long long)p.splits * M * Nv : 0;
}

// ---- tile plan of a size that has no measured entry ------------------------
// t(us) = c0 + step (1 + many (whole rounds, up to 4)) (k steps of all rounds) + lone (k steps a thin
//         round loses to latency; four-wave tiles: gains), these at least mem (MB of operands)
//         + epi[class] rounds + merge [split] + fin (split: MB of slabs written and read, or pieces)
// fitted to timings on weights that no cache holds, of every tile and split: 4,200 products (width 128 ..
// 60000, k 512 .. 29000, 2 .. 6000 rows); wrong choices weighed more than wrong times.  Over these the
// plan is 1 % off the best of all on the average, 0.7 % over the widths of named models.  Fitted
// before tile 22 had its rows 8 apart and the slabs their 16-byte reads, and without the eight-wave
// tiles from 300 rows on, it was 4 %: 6000 x 57344 x 8192 SwiGLU 4250 us on 224 x 192, 3970 on 256 x 256;
// 350 x 2048 x 11776 43.4 on 128 x 128 in pieces, 34.9 on 256 x 128 in slabs; 113 x 57344 x 8192 SwiGLU,
// where all wait for the weights, 186 on 128 x 128, 169 on 128 x 256.
// An image model's products are short (k from 128) or have a 16-bit residual or GEGLU: the tile's end
// weighs as much as its k steps, so these have rows of their own, and three tiles more.
// Over 123 sizes (width 256 .. 2048, 66 .. 18432 rows) 1.5 % off the best on the average, at most 15;
// without the terms 5.5 %, at most 58 (12288 x 320 x 320 + residual 17.3 us, 11.0 so; 6144 x 5120 x
// 640 GEGLU 59.6, 50.8).
struct TileCost {
  int cfg, bm, bn, slots;                  // slots: workgroups a CU holds
  // epi: store, f32, SwiGLU, GELU, 16-bit residual, GEGLU, store of k < 512; negative epi or
  // merge: not modelled (that epilogue, that tile in splits)
  float c0, step, many, lone, mem, epi[7], merge, fin;
};
static constexpr TileCost kTileCosts[] = {
    {5, 256, 256, 1, 1.315f, 1.423f, 0.0515f, 0.1f, 0.0978f, {8.12f, 12.76f, 9.355f, 10.28f, -1.f, -1.f, -1.f}, 0.465f, 0.211f},
    {6, 256, 128, 1, 0.581f, 0.739f, 0.00913f, 0.1f, 0.0758f, {8.567f, 8.26f, 9.837f, 9.006f, -1.f, -1.f, -1.f}, 0.479f, 0.224f},
    {7, 128, 128, 1, 2.447f, 0.492f, 0.00891f, 0.1f, 0.0668f, {5.312f, 5.424f, 5.552f, 6.45f, -1.f, -1.f, -1.f}, 0.791f, 0.198f},
    {12, 64, 128, 2, 0.935f, 0.855f, -0.0328f, -0.0607f, 0.104f, {2.788f, 2.795f, 2.913f, 3.841f, -1.f, -1.f, -1.f}, 2.088f, 0.287f},
    {13, 64, 64, 2, 0.356f, 0.547f, 0.1f, 0.0549f, 0.00984f, {0.416f, 0.656f, 0.489f, 1.683f, -1.f, -1.f, -1.f}, 2.649f, 0.448f},
    {18, 64, 160, 1, 1.177f, 0.457f, 0.00266f, 0.1f, 0.0426f, {4.479f, 4.01f, -1.f, 4.044f, -1.f, -1.f, -1.f}, 1.721f, 0.209f},
    {22, 256, 256, 1, 1.152f, 1.098f, 0.0174f, 0.128f, 0.176f, {9.638f, -1.f, 10.07f, 19.8f, -1.f, -1.f, -1.f}, 13.95f, 7.829f},
    {25, 256, 256, 1, 0.661f, 1.093f, 0.0424f, 0.209f, 0.0386f, {15.45f, -1.f, 8.939f, 14.98f, -1.f, -1.f, -1.f}, 1.337f, 9.021f},
    {26, 256, 192, 1, 0.12f, 0.916f, 0.0398f, 0.127f, 0.125f, {8.747f, 12.5f, 9.162f, 13.78f, -1.f, -1.f, -1.f}, 6.793f, 3.485f},
    {27, 128, 256, 1, 0.489f, 0.657f, 0.11f, 0.169f, 0.113f, {4.901f, 7.49f, 4.916f, 11.28f, -1.f, -1.f, -1.f}, 3.05f, 3.666f},
    {28, 128, 128, 1, 0.564f, 0.443f, 0.0724f, 0.0141f, 0.119f, {3.183f, 3.551f, 3.063f, 6.329f, -1.f, -1.f, -1.f}, 1.816f, 2.725f},
    {29, 128, 192, 1, 0.158f, 0.513f, 0.11f, 0.237f, 0.18f, {6.195f, 6.798f, 5.003f, 8.104f, -1.f, -1.f, -1.f}, 6.417f, 2.032f},
    {30, 96, 256, 1, 0.562f, 0.635f, 0.043f, 0.142f, 0.149f, {3.821f, 5.301f, 3.733f, 8.382f, -1.f, -1.f, -1.f}, 3.125f, 3.253f},
    {31, 160, 256, 1, 0.797f, 0.711f, 0.0445f, 0.0764f, 0.127f, {7.909f, 11.57f, 7.589f, 13.52f, -1.f, -1.f, -1.f}, 9.75f, 3.796f},
    {32, 192, 192, 1, 1.316f, 0.62f, 0.0623f, 0.0716f, 0.127f, {7.468f, 10.46f, 6.705f, 11.87f, -1.f, -1.f, -1.f}, 4.369f, 3.521f},
    {33, 224, 192, 1, 0.846f, 0.777f, 0.0146f, -0.0934f, 0.144f, {10.04f, 12.63f, 8.565f, 13.22f, -1.f, -1.f, -1.f}, 0.812f, 3.47f},
    {34, 192, 256, 1, 1.768f, 0.979f, 0.0472f, 0.0879f, 0.126f, {6.113f, -1.f, 6.451f, 13.14f, -1.f, -1.f, -1.f}, 2.423f, 4.585f},
    {35, 224, 256, 1, 1.053f, 1.076f, 0.045f, 0.148f, 0.113f, {7.659f, -1.f, 7.822f, 13.64f, -1.f, -1.f, -1.f}, 6.25f, 4.798f},
    // between 160 and 256 rows a tile the next larger one is padding and the next smaller one a partial wave
    // more: of 2,275 products these are taken for a twelfth, 8 % faster each (SwiGLU of 777 x 28672 x 4096 172
    // us on 192 x 192, 162 on 160 x 192; 777 x 4096 x 14336 98 in three pieces of 160 x 256, 93 in two of 224 x
    // 128; 1100 x 6144 x 4096 57.6, 51.9).  Their estimates carry 1 or 2 % for the fit's own error.
    {36, 160, 192, 1, 1.492f, 0.68f, 0.019f, 0.f, 0.162f, {6.568f, 8.877f, 5.377f, 9.642f, -1.f, -1.f, -1.f}, 3.255f, 2.515f},
    {37, 160, 128, 1, 0.744f, 0.511f, 0.032f, 0.f, 0.163f, {5.184f, 7.988f, 4.123f, 7.683f, -1.f, -1.f, -1.f}, 3.312f, 3.9f},
    {38, 224, 128, 1, 0.259f, 0.64f, 0.017f, 0.f, 0.162f, {6.65f, 10.33f, 5.431f, 11.4f, -1.f, -1.f, -1.f}, 1.852f, 3.237f},
    // f32 results on the tiles of gemm_ws.h, of 180 products (2048 .. 8192 columns, k 4096 .. 28672, 100 .. 6000 rows):
    // 0.3 % off the best of all, 2.5 % faster than without them on the average, 5 to 16 % from 1300 rows on.  Of 170 others (1024
    // .. 12288 columns, k 2048 .. 28672, 700 .. 8192 rows) 3.5 % faster, at most 5 % slower (12288 x 4096 at 1665 and 2600 rows
    // 147 and 231 us on 224 x 192, 155 and 243).  22 and 25 are one kernel there; either id may be a plan's
    {22, 256, 256, 1, 7.023f, 1.101f, 0.0578f, -0.3914f, 0.1106f, {-1.f, 12.87f, -1.f, -1.f, -1.f, -1.f, -1.f}, 1.22f, 5.201f},
    {25, 256, 256, 1, 7.023f, 1.101f, 0.0578f, -0.3914f, 0.1106f, {-1.f, 12.87f, -1.f, -1.f, -1.f, -1.f, -1.f}, 1.22f, 5.201f},
    {34, 192, 256, 1, 6.121f, 0.9357f, 0.0341f, -0.3562f, 0.1039f, {-1.f, 1.538f, -1.f, -1.f, -1.f, -1.f, -1.f}, 3.788f, 5.132f},
    {35, 224, 256, 1, 6.214f, 1.06f, 0.0249f, -0.5244f, 0.0906f, {-1.f, 8.137f, -1.f, -1.f, -1.f, -1.f, -1.f}, 4.135f, 5.723f},
    // products of image models: the classes from kImageClass on
    {4, 64, 64, 4, 1.48f, 0.787f, 0.f, 0.263f, 0.f, {-1.f, -1.f, -1.f, -1.f, 3.44f, 2.92f, 3.04f}, -1.f, 0.f},
    {5, 256, 256, 1, 0.69f, 1.43f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 11.7f, 9.55f, 8.55f}, 4.16f, 0.304f},
    {6, 256, 128, 1, 0.844f, 0.802f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 7.42f, 6.68f, 6.1f}, 3.93f, 0.325f},
    {7, 128, 128, 1, 2.77f, 0.539f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 5.25f, 4.69f, 4.05f}, 3.6f, 0.382f},
    {8, 128, 128, 2, 2.27f, 1.02f, 0.f, 0.44f, 0.f, {-1.f, -1.f, -1.f, -1.f, 5.46f, 4.78f, 4.01f}, -1.f, 0.f},
    {12, 64, 128, 2, 4.62f, 0.663f, 0.f, 0.145f, 0.f, {-1.f, -1.f, -1.f, -1.f, 1.82f, 2.31f, -1.f}, 3.09f, 0.468f},
    {13, 64, 64, 2, 3.41f, 0.427f, 0.f, 0.107f, 0.f, {-1.f, -1.f, -1.f, -1.f, 2.f, 2.05f, 1.75f}, 2.83f, 0.484f},
    {14, 64, 160, 2, 1.33f, 0.779f, 0.f, 0.386f, 0.f, {-1.f, -1.f, -1.f, -1.f, 5.97f, -1.f, 3.69f}, -1.f, 0.f},
    {18, 64, 160, 1, 2.28f, 0.467f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 5.07f, -1.f, 3.2f}, 3.53f, 0.353f},
    {22, 256, 256, 1, 0.f, 1.26f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 18.1f, 11.4f, 12.f}, 13.2f, 10.2f},
    {25, 256, 256, 1, 0.f, 1.49f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 14.9f, 9.6f, 10.8f}, 20.8f, 13.2f},
    {26, 256, 192, 1, 0.f, 1.13f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 13.1f, 9.73f, 9.91f}, 16.1f, 6.33f},
    {27, 128, 256, 1, 4.43f, 0.837f, 0.f, 0.f, 0.f, {-1.f, -1.f, -1.f, -1.f, 6.33f, 4.58f, 3.86f}, 13.7f, 4.33f},
};
// 0 .. 6, as TileCost::epi; from kImageClass on the products of image models
static constexpr int kImageClass = 4;
static int cost_class(int epi, int K) {
  return epi == kEpiResid32 || epi == kEpiStore32 ? 1
         : epi == kEpiSwiglu                      ? 2
         : epi == kEpiGelu                        ? 3
         : epi == kEpiAdd16                       ? 4
         : epi == kEpiGeglu                       ? 5
         : epi == kEpiStore && K < 512            ? 6 : 0;
}
static double tile_cost(const TileCost& c, int splits, long long M, long long Nv, int K, int epi) {
  const long long ks = (K + kGBK - 1) / kGBK, t = ((M + c.bm - 1) / c.bm) * ((Nv + c.bn - 1) / c.bn);
  const int cls = cost_class(epi, K);
  if (c.epi[cls] < 0 || (splits > 1 && c.merge < 0)) return -1;   // not modelled
  double steps, rounds, whole, lone = 0, fin = 0;
  bool split = false;
  if (four_wave_cfg(c.cfg)) {
    const SplitPlan p = split_plan(c.cfg, splits, (int)M, Nv, K);
    if (splits > 1 && p.pieces != splits) return 1e30;   // it would run another split
    const long long rest = t <= 256 ? t : t % 256;
    const long long dp = (t - rest) / 256, per = p.pieces ? p.kps / kGBK : ks;
    steps = (double)(dp * ks + (rest ? per : 0));
    rounds = (double)(dp + (rest ? 1 : 0));
    whole = (double)dp;
    split = p.pieces > 0;
    fin = p.pieces;
    if (rest) lone = per * (1 - (double)rest * std::max(p.pieces, 1) / 256);
  } else {
    const long long kps = (ks + splits - 1) / splits, sp = (ks + kps - 1) / kps, n = t * sp;
    const long long full = n / (256 * c.slots), rest = n % (256 * c.slots);
    const double share = (double)((rest + 255) / 256) / c.slots;   // of a round's slots on a CU
    steps = (double)kps * (full + share);
    rounds = (double)(full + (rest ? 1 : 0));
    whole = (double)full;
    lone = rest ? (1 - share) * kps : 0;
    split = sp > 1;
    if (split) fin = (double)(sp + 1) * M * Nv * 4e-6;
  }
  const double mb = ((double)Nv * K + (double)M * K) * 2e-6;
  const bool image = cls >= kImageClass;
  const double mem = !image ? c.mem * mb : four_wave_cfg(c.cfg) ? mb / 5.2 : 0.;
  const double main = c.step * (1 + c.many * std::min(whole, 4.)) * steps + c.lone * lone;
  const double us = c.c0 + std::max(main, mem) + c.epi[cls] * rounds +
                    (split ? c.merge + c.fin * fin : 0.);
  // operands from memory; of tiles that all wait for them the one with the least work
  return image ? std::max(us, mb / 5 + 3) + 0.02 * us : us;
}

// (cfg, splits) for a product on tiles; of 64 rows and fewer captured ones, whose stream form stays out
// of graphs.  On entry *cfg, *splits: a measured plan of this very size, or cfg -1; it stands unless it
// is modelled and 10 % behind the best.  big: an operand of 2 GB or more (31-bit offsets of the
// four-wave tiles).
static double tile_plan(int M, long long Nv, int K, int epi, int big, int* cfg, int* splits) {
  const bool gated = epi == kEpiSwiglu || epi == kEpiGeglu;
  const bool image = cost_class(epi, K) >= kImageClass;
  const int ks = (K + kGBK - 1) / kGBK;
  double best = 1e30, given = -1;
  int bc = 0, bs = 1;
  for (const TileCost& c : kTileCosts) {
    const bool four = four_wave_cfg(c.cfg);
    if (c.cfg == *cfg) given = std::max(given, tile_cost(c, *splits, M, Nv, K, epi));
    if (four && (K % kGBK || big)) continue;
    if (gated && c.cfg == 18) continue;               // 80-column wave tiles
    if (!image && c.bm > 2.2 * std::max(M, 64)) continue;   // mostly padding: not in the fit
    // 256 x 256: three barriers a step for long rows of k, else two (k 8192 4.6 % faster, 11776 4.9, 14336
    // 0.8 slower, 23552 2.4; an image model's line as fitted)
    const bool three = K > (image ? 8192 : 12288);
    if (c.cfg == (three ? k4WCfg : k4WCfg + k4WSched)) continue;
    for (int sp : {1, 2, 3, 4, 6, 8, 16}) {
      if (sp > 1 && (ks / sp < 4 || (four && image && M < 200))) break;
      if (!four && (sp & (sp - 1))) continue;
      const double t = tile_cost(c, sp, M, Nv, K, epi);
      if (t >= 0 && t < best) {
        best = t;
        bc = c.cfg;
        bs = sp;
      }
    }
  }
  if (*cfg >= 0 && (given < 0 || given <= 1.1 * best)) return given < 0 ? best : given;
  *cfg = bc;
  *splits = bs;
  return best;
}
CAKE_API int cake_gemm_plan(int M, long long Nv, int K, int epi, int big, int* cfg, int* splits) {
  if (M < 1 || Nv < 1 || K < 1 || !cfg || !splits) return (int)hipErrorInvalidValue;
  tile_plan(M, Nv, K, epi, big, cfg, splits);
  return 0;
}

// counters of tick below
CAKE_API int cake_gemm_ticks() { return 2 * kPieceTiles * kPieceWaves; }

// y = epilogue(x W^T).  N = output features (gated: W has 2N rows, gate rows
// [0, N), up/gate-2 rows [N, 2N)).  splits > 1 needs ws (cake_gemm_ws_floats) and, for a four-wave
// tile, tick (cake_gemm_ticks zeros, zero again when the launch is done): both belong to one launch
// at a time, so to one stream, or to one graph.
// Requirements (host-checked in ops/gemm.py): K % 8 == 0, lda/ldb % 8 == 0,
// 16-byte aligned operand bases, gated => N % 16 == 0.
// alpha (f32 epilogues only, 1 elsewhere): r32 (+)= alpha * (x W^T + bias).
CAKE_API int cake_gemm_scaled(int dt, int epi, int cfg, int splits, const void* a, long long lda,
                              const void* b, long long ldb, void* c, long long ldc,
                              const void* bias, void* resid, long long ldr, float* ws,
                              void* tick, const void* zeros, int M, int N, int K, float alpha,
                              hipStream_t st) {
  if (alpha != 1.f && epi != kEpiResid32 && epi != kEpiStore32) return (int)hipErrorInvalidValue;
  // tiles 28 on have no 16-bit residual and no GEGLU, 64 kernels that no plan takes: whole 128 x 256 tiles
  if (cfg > k4WCfg128 + k4WSched && four_wave_cfg(cfg) && (epi == kEpiAdd16 || epi == kEpiGeglu)) {
    cfg = k4WCfg128 + k4WSched;
    splits = 1;
  }
  int bm, bn;
  cfg_dims(cfg, bm, bn);
  if (bm == 0 || M <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || splits < 1)
    return (int)hipErrorInvalidValue;
  const bool gated = (epi == kEpiSwiglu || epi == kEpiGeglu);
  if (gated && N % 16) return (int)hipErrorInvalidValue;
  const bool four = four_wave_cfg(cfg);
  if (cfg == kRSCfg || four) {  // whole 64-element k steps; 31-bit offsets
    const long long wrows = gated ? 2LL * N : N;
    if (K % kGBK || ((long long)(M - 1) * lda + K) * 2 >= 0x7fffffffLL ||
        ((wrows - 1) * ldb + K) * 2 >= 0x7fffffffLL)
      return (int)hipErrorInvalidValue;
  }
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c;
  g.bias = (const uint16_t*)bias;
  g.r32 = (epi == kEpiResid32 || epi == kEpiStore32) ? (float*)resid : nullptr;
  g.r16 = (epi == kEpiAdd16) ? (const uint16_t*)resid : nullptr;
  g.ws = ws; g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.ldr = ldr;
  g.M = M; g.N = N; g.K = K;
  g.gated = gated ? 1 : 0;
  g.alpha = alpha;
  g.half = N;
  g.Nv = gated ? 2 * N : N;
  g.tiles_m = (M + bm - 1) / bm;
  g.tiles_n = (g.Nv + bn - 1) / bn;
  const SplitPlan sp = split_plan(cfg, splits, M, g.Nv, K);
  splits = sp.splits;
  g.kps = sp.kps;
  dim3 grid(g.tiles_m * g.tiles_n, splits);
  if (sp.pieces > 0) {
    if (ws == nullptr || tick == nullptr) return (int)hipErrorInvalidValue;
    g.tick = static_cast<unsigned*>(tick);
    g.pieces = sp.pieces;
    g.dp_tiles = sp.ntiles - sp.rest;
    grid = dim3(g.dp_tiles + sp.rest * sp.pieces, 1);
  }
  const int kernel_epi = splits > 1 ? (int)kEpiPartial : epi;
  if (splits > 1 && ws == nullptr) return (int)hipErrorInvalidValue;
  int rc = (dt == kBF16) ? dispatch_epi<kBF16>(kernel_epi, cfg, grid, st, g)
         : (dt == kF16) ? dispatch_epi<kF16>(kernel_epi, cfg, grid, st, g)
                        : (int)hipErrorInvalidValue;
  if (rc != 0 || splits == 1) return rc;
  const dim3 fgrid((N + 1023) / 1024, M);
  return (dt == kBF16) ? dispatch_finalize<kBF16>(epi, fgrid, st, g, splits)
                       : dispatch_finalize<kF16>(epi, fgrid, st, g, splits);
}

CAKE_API int cake_gemm(int dt, int epi, int cfg, int splits, const void* a, long long lda,
                       const void* b, long long ldb, void* c, long long ldc, const void* bias,
                       void* resid, long long ldr, float* ws, void* tick, const void* zeros, int M,
                       int N, int K, hipStream_t st) {
  return cake_gemm_scaled(dt, epi, cfg, splits, a, lda, b, ldb, c, ldc, bias, resid, ldr, ws, tick,
                          zeros, M, N, K, 1.f, st);
}

// ---- products of few rows (gemm_rows.h) -----------------------------------
// Which form a product of M rows takes: 0 the tile kernels (cake_gemm_scaled), 1 direct, 2 stream.
// The estimates (us) are fits to timings on weights that no cache holds, 2 .. 64 rows of 80 weight
// shapes, 0.2 .. 940 MB, every form and share; wrong choices weighed more than wrong times: what they picked
// was 0.4 % off the best of all on the average, at most 16 %.  The stream form was one of four waves in turn then; its
// 128-row strips are 1 - 8 % faster since (gemm_rows.h) and not fitted again.  Of 35 narrow shapes (256 .. 3072 columns, k 2048
// .. 28672) at 2 .. 16 rows they are 1.5 % off now, at most 19 (1024 x 8960, where 64 x 64 tiles in splits are the best, 11.2
// for 13.3 us).  Both sides of the lines they draw, measured:
// 3072 x 2048 at 5 rows direct 6.7, stream 8.4; 4096 x 4096 at 5 rows 10.3, 11.5, at 16 12.4, 11.7 (tiles
// 12.1), at 24 tiles 12.4, stream 15.0; 4096 x 14336 at 24 rows stream 26.6, tiles 27.5, at 33 30.1, 27.8;
// 6144 x 4096 at 16 rows stream 14.3, tiles 15.7, at 33 18.3, 16.7; 8192 x 8192 at 24 rows stream 29.6,
// tiles 37.1; 28672 x 4096 SwiGLU at 64 rows 41.5, 51.8.  Rows of k that start amid a 128-byte line (k no
// multiple of 64) cost a second line at either end of a piece: 4096 x 10928 against 4096 x 11008, 5 rows
// direct 31.9 / 24.1, stream 21.0 / 20.1, 33 rows stream 36.1 / 30.9, tiles 26.3 / 25.2.
struct StreamPlan {
  int bn, kst, most;   // weight rows of a strip, k of a step (gemm_rows.h StreamShape), workgroups at most
  int wgs, per;        // workgroups, steps of each
  double us;
};
// The shares: as many as there are workgroups at most, of equal length wherever that ends, or whole
// strips, or equal parts of one.  The latter two park no sums, or one a share, and never wait for them
// amid a share; with fewer workgroups a CU takes up to 42 KB a us of weights, all of them 7.3 MB.
// At 24 / 45 rows, 256 shares that end anywhere against the best of the others: 28672 x 4096 SwiGLU 45.8 /
// 50.4, 38.9 / 39.9 us (224 whole strips), 19456 x 4096 37.5 / 41.4, 31.5 / 37.5 (152), 6144 x 4096 17.6 /
// 22.3, 16.3 / 19.1 (192 quarters), 12288 x 4096 24.7 / 27.1, 23.5 / 26.8 (192 halves); 10240 x 8192 35.2 /
// 38.7, 35.7 / 42.3 (160 halves).  8192 x 8192, 256 quarters: 29.6 / 30.9.
static StreamPlan stream_plan(int M, long long Nv, int K, bool gated) {
  const int mt = (M + 15) / 16;
  StreamPlan p = mt > 1 || gated ? StreamPlan{128, 64, 256, 0, 0, 1e30} : StreamPlan{64, 128, 512, 0, 0, 1e30};
  const long long strips = (Nv + p.bn - 1) / p.bn, ks = (K + p.kst - 1) / p.kst, total = strips * ks;
  const int least = kRowsMinK / p.kst;
  const double mid = K % 64 != 0 ? 1 : 0;   // rows start amid a line
  const auto take = [&](long long wgs, long long per, double us) {
    if (us < p.us) { p.wgs = (int)wgs; p.per = (int)per; p.us = us; }
  };
  for (int most = p.most; most >= 256; most /= 2) {   // ends anywhere; a strip's shares are parked and summed
    const long long per = std::max<long long>((total + most - 1) / most, least);
    const long long wgs = (total + per - 1) / per;
    const double shares = (double)ks / per, met = std::min(shares, 1.);
    if (ks % per == 0 || per % ks == 0) continue;   // below
    if (most == 512)
      take(wgs, per, 5.36 + 0.062 * M + (1.3 + 0.25 * mid) * per);
    else if (p.most == 512)
      take(wgs, per, 3.88 + 0.053 * M + 0.61 * met + 0.035 * shares + (0.594 + 0.08 * mid) * per);
    else
      take(wgs, per, (mt > 1 ? 5.37 : 6.05) +
           mt * (0.73 * met + 0.273 * shares + 0.9 * std::min(1., std::pow(4096. / K, 3))) +
           per * (0.636 - 0.0097 * mt + 0.4 * mid));
  }
  const double cu = mt == 1 ? 0.414 : mt == 2 ? 0.396 : mt == 3 ? 0.472 : 0.476;   // us of a step of a CU's own
  const auto even = [&](long long wgs, long long per, int parts) {
    const int on = (int)((wgs + 255) / 256);   // workgroups on a CU
    const double step = std::max(cu * on, wgs * 16.384e-3 / 7.33) + 0.15 * mid;
    const double sums = parts <= 1 ? 0.
                        : mt > 1           ? 2.37 + mt * (0.53 + 0.262 * parts)
                        : gated            ? 4.4
                                           : 1.34 + 0.046 * parts;
    take(wgs, per, 2.52 + 0.89 * on + per * step + sums);
  };
  for (long long c = (strips + p.most - 1) / p.most, n = 0; n < 2; ++c, ++n)
    even((strips + c - 1) / c, c * ks, 1);
  for (int s = 2; s <= 16 && strips * s <= p.most; s *= 2)
    if (ks % s == 0 && ks / s >= least) even(strips * s, ks / s, s);
  return p;
}
static double rows_best(int M, long long Nv, int K, bool gated, int* kind) {   // us of the best form
  const double kb = K * 2e-3;   // KB of one row of k
  const bool mid = K % 64 != 0;   // rows start amid a line
  const double tiles = 5.7 + Nv * kb / 5929 + 0.345e-3 * std::min(K, 8192);
  const double stream = stream_plan(M, Nv, K, gated).us;
  double direct = 1e9;
  if (M <= 32) {
    const int nt = gated || Nv > 4096 ? 2 : 1;
    const long long wgs = (Nv + 16 * nt - 1) / (16 * nt);
    // a CU's share at 30.4 (of two strips 26.4) KB a us, all weights and 0.65 of the reads of x at 5.8 MB
    const double all = (Nv + 0.65 * wgs * M) * kb / 5844;
    const double own = (double)((wgs + 255) / 256) * (16 * nt + M) * kb / (nt == 2 ? 26.4 : 30.4);
    direct = 1.91 + (mid ? 1.56 : 1.) * std::max(own, all);
  }
  *kind = direct <= stream && direct <= tiles ? 1 : stream < tiles ? 2 : 0;
  return *kind == 1 ? direct : std::min(stream, tiles);
}
static int rows_kind(int M, long long Nv, int K, bool gated) {
  int kind = 0;
  if (M <= 64 && Nv <= 64LL * kRowsTicks) rows_best(M, Nv, K, gated, &kind);
  return kind;
}
CAKE_API int cake_gemm_rows_kind(int M, long long Nv, int K, int gated) {
  return M < 1 || Nv < 1 || K < 1 ? 0 : rows_kind(M, Nv, K, gated != 0);
}

// stream form: f32 elements of ws (two parked strips per share) and counters of tick
CAKE_API long long cake_gemm_rows_ws_floats(int M) { return 256LL * 4096 * ((M + 15) / 16); }
CAKE_API int cake_gemm_rows_ticks() { return 4 * kRowsTicks; }

// cake_gemm_scaled for M <= 64 rows in the form `kind` (1 or 2).  The stream form needs ws
// (cake_gemm_rows_ws_floats) and tick (cake_gemm_rows_ticks zeros, zero again when the launch is
// done): both belong to one launch at a time, so to one stream.
CAKE_API int cake_gemm_rows(int dt, int epi, int kind, const void* a, long long lda, const void* b,
                            long long ldb, void* c, long long ldc, const void* bias, void* resid,
                            long long ldr, float* ws, void* tick, const void* zeros, int M, int N,
                            int K, float alpha, hipStream_t st) {
  if (alpha != 1.f && epi != kEpiResid32 && epi != kEpiStore32) return (int)hipErrorInvalidValue;
  const bool gated = (epi == kEpiSwiglu || epi == kEpiGeglu);
  if (M < 1 || M > 64 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || (gated && N % 16) ||
      !(kind == 1 || kind == 2) || (kind == 1 && M > 32) || (kind == 2 && (!ws || !tick || !zeros)))
    return (int)hipErrorInvalidValue;
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c;
  g.bias = (const uint16_t*)bias;
  g.r32 = (epi == kEpiResid32 || epi == kEpiStore32) ? (float*)resid : nullptr;
  g.r16 = (epi == kEpiAdd16) ? (const uint16_t*)resid : nullptr;
  g.ws = ws; g.tick = (unsigned*)tick; g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.ldr = ldr;
  g.M = M; g.N = N; g.K = K;
  g.gated = gated ? 1 : 0;
  g.alpha = alpha;
  g.half = N;
  g.Nv = gated ? 2 * N : N;
  g.tiles_m = 1;
  const int mt = (M + 15) / 16;
  int form, wgs;
  if (kind == 2) {
    const StreamPlan sp = stream_plan(M, g.Nv, K, gated);
    g.tiles_n = (g.Nv + sp.bn - 1) / sp.bn;
    if (g.tiles_n > kRowsTicks) return (int)hipErrorInvalidValue;
    g.kps = sp.per;
    form = 2;
    wgs = sp.wgs;
  } else {
    const int nt = gated || g.Nv > 4096 ? 2 : 1;   // one 16-row strip per CU, or two
    form = nt - 1;
    wgs = (g.Nv + 16 * nt - 1) / (16 * nt);
  }
  return dt == kBF16 ? Rows<kBF16>::run(epi, form, mt, dim3(wgs), st, g)
         : dt == kF16 ? Rows<kF16>::run(epi, form, mt, dim3(wgs), st, g) : (int)hipErrorInvalidValue;
}

// ---- products that leave their sums in slabs ------------------------------
// Which form such a product takes, and whether the launch that follows it gains from summing them
// (gemm_slabs.hip).  The estimates (us) are fits to timings of product and norm or rotation on weights that no
// cache holds, 2 .. 64 rows of 33 shapes, 2 .. 470 MB, every form: what they picked was 0.35 % off the best on the
// average, at most 11 % (the stream form as above).  The two launches take 0.9 of the three or two they replace at 2 .. 16 rows (4096 x
// 14336 and norm at 5 rows 26.6 -> 25.0 us), 0.87 at 24 .. 64 (at 45 rows 32.6 -> 30.2, 4096 x 4096 16.0 ->
// 13.9, 6144 x 4096 and rotation 20.3 -> 18.3, 10240 x 8192 44.4 -> 37.7, 4096 x 23552 48.5 -> 42.6).
struct SlabStream { double c0, cu, step, rate, slab, mid; };   // by 16-row tiles of x
static constexpr SlabStream kSlabStream[4] = {{3.02, 0.544, 0.518, 6.40, 1.05, 0.10},
                                              {0.52, 3.394, 0.506, 6.71, 1.15, 0.15},
                                              {1.77, 1.271, 0.587, 6.72, 1.14, 0.29},
                                              {1.69, 2.506, 0.567, 6.90, 0.82, 0.24}};
struct SlabTile { int cfg, least; double c0, step, mem, slab, wgs, mid; };   // least: rows
static constexpr SlabTile kSlabTiles[] = {{7, 49, 5.20, 0.556, 0.172, 0.688, 1.02, 0.06},
                                          {12, 1, 3.52, 1.167, 0.177, 0.380, 2.27, 0.08},
                                          {13, 1, 3.79, 0.674, 0.178, 0.464, 1.01, 0.08},
                                          {18, 1, 4.08, 0.551, 0.185, 0.462, 3.36, 0.17}};
static constexpr double kSlabGain = 2.2;
// 1 and the form in *kind, *cfg, *parts (as cake_gemm_slabs takes them); 0: the product with the epilogue
// `epi`, and what follows it as a launch of its own
CAKE_API int cake_gemm_slab_plan(int M, long long N, int K, int epi, int big, int* kind, int* cfg, int* parts) {
  if (M < 1 || N < 1 || N > 64LL * kRowsTicks || K < 1 || !kind || !cfg || !parts) return 0;
  const int k64 = (K + kGBK - 1) / kGBK;
  const double mid = K % 64 != 0 ? 1 : 0;   // rows start amid a line
  double best = 1e30;
  const auto take = [&](double us, int f, int c, int p) {
    if (us < best) { best = us; *kind = f; *cfg = c; *parts = p; }
  };
  if (M > 64) {
    // of more rows the sum of a plan's splits (eight-wave tiles) goes into what follows, which saves the launch
    // between them; other plans give way where that puts them behind: at 200 rows 4096 x 4096 28 -> 23 us,
    // 4096 x 14336 the same plan, 8192 x 8192 at 300 rows stays on four-wave pieces (slabs 2 % slower)
    int c = -1, s = 1;
    const double plain = tile_plan(M, N, K, epi, big, &c, &s);
    for (const TileCost& t : kTileCosts) {
      if (four_wave_cfg(t.cfg) || t.bm > 2.2 * M) continue;
      for (int sp : {2, 4, 8, 16}) {
        if (k64 / sp < 4) break;
        const double us = tile_cost(t, sp, M, N, K, epi);
        if (us >= 0) take(us - kSlabGain, 0, t.cfg, sp);
      }
    }
    return best < plain;
  }
  const int mt = (M + 15) / 16, bn = mt > 1 ? 128 : 64, kst = mt > 1 ? 64 : 128, most = mt > 1 ? 256 : 512;
  const int ks = (K + kst - 1) / kst;
  const long long strips = (N + bn - 1) / bn;
  const SlabStream& c = kSlabStream[mt - 1];
  for (int p : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16}) {
    const int per = (ks + p - 1) / p;
    if (p > 1 && (per * (p - 1) >= ks || ks / p < kRowsMinK / kst || strips * p > most)) continue;
    const double wgs = (double)strips * p, on = std::ceil(wgs / 256);
    take(c.c0 + c.cu * on + per * (std::max(c.step * on, wgs * 16.384e-3 / c.rate) + c.mid * mid) +
             c.slab * p * M * N * 4e-6, 2, 0, p);
  }
  for (const SlabTile& t : kSlabTiles) {
    int bm, bn2;
    cfg_dims(t.cfg, bm, bn2);
    for (int p : {2, 4, 8, 16}) {
      if (M < t.least || k64 / p < 4) break;
      const int kps = (k64 + p - 1) / p, sp = (k64 + kps - 1) / kps;
      const double n = (double)((M + bm - 1) / bm) * ((N + bn2 - 1) / bn2) * sp / 256;
      const int slots = t.cfg == 12 || t.cfg == 13 ? 2 : 1;
      const double rounds = std::ceil(n - 1e-9) / slots;   // of the chip's slots
      take(t.c0 + std::max(t.step * kps * rounds, t.mem * ((double)N * K + (double)M * K) * 2e-6) +
               t.slab * sp * M * N * 4e-6 + t.wgs * n + t.mid * mid * kps, 0, t.cfg, p);
    }
  }
  if (M <= 32) {   // as rows_kind
    const int nt = N > 4096 ? 2 : 1;
    const double kb = K * 2e-3, wgs = (double)((N + 16 * nt - 1) / (16 * nt));
    take(1.91 + 1.36 + (mid ? 1.56 : 1.) * std::max(std::ceil(wgs / 256) * (16 * nt + M) * kb / (nt == 2 ? 26.4 : 30.4),
                                                    (N + 0.65 * wgs * M) * kb / 5844), 1, 0, 1);
  }
  return 1;
}

// The product alone, as f32 slabs ws [slabs][M][N] that the launch behind it sums (gemm_slabs.hip).  kind 0:
// tiles `cfg` (no four-wave tile) with k in `parts`; 1: the direct form; 2: the stream form, every strip in
// `parts` of whole steps.  Returns the number of slabs, or minus a HIP error.
CAKE_API int cake_gemm_slabs(int dt, int kind, int cfg, int parts, const void* a, long long lda, const void* b,
                             long long ldb, float* ws, const void* zeros, int M, int N, int K, hipStream_t st) {
  if (M < 1 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || parts < 1 || !ws || !zeros ||
      !(dt == kBF16 || dt == kF16) || (kind != 0 && M > 64) || (kind == 1 && (M > 32 || parts != 1)) ||
      (kind == 0 && (parts < 2 || four_wave_cfg(cfg) || cfg == kRSCfg)) || kind < 0 || kind > 2)
    return -(int)hipErrorInvalidValue;
  if (kind == 1) {
    const int e = cake_gemm_rows(dt, kEpiStore32, 1, a, lda, b, ldb, nullptr, 0, nullptr, ws, N, nullptr, nullptr,
                                 zeros, M, N, K, 1.f, st);
    return e ? -e : 1;
  }
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b;
  g.ws = ws; g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb;
  g.M = M; g.N = g.Nv = g.half = N; g.K = K;
  if (kind == 0) {
    const SplitPlan sp = split_plan(cfg, parts, M, N, K);
    if (sp.bm == 0 || sp.splits < 2) return -(int)hipErrorInvalidValue;
    g.tiles_m = (M + sp.bm - 1) / sp.bm;
    g.tiles_n = (N + sp.bn - 1) / sp.bn;
    g.kps = sp.kps;
    const dim3 grid(g.tiles_m * g.tiles_n, sp.splits);
    const int e = dt == kBF16 ? dispatch_epi<kBF16>(kEpiPartial, cfg, grid, st, g)
                              : dispatch_epi<kF16>(kEpiPartial, cfg, grid, st, g);
    return e ? -e : sp.splits;
  }
  const int mt = (M + 15) / 16, bn = mt > 1 ? 128 : 64, kst = mt > 1 ? 64 : 128;
  const int ks = (K + kst - 1) / kst;
  g.tiles_m = 1;
  g.tiles_n = (N + bn - 1) / bn;
  g.kps = (ks + parts - 1) / parts;
  g.pieces = (ks + g.kps - 1) / g.kps;   // no part without a step
  const long long wgs = (long long)g.tiles_n * g.pieces;
  if (wgs > 0x7fffff) return -(int)hipErrorInvalidValue;
  const int e = dt == kBF16 ? Rows<kBF16>::run(kEpiPartial, 2, mt, dim3((unsigned)wgs), st, g)
                            : Rows<kF16>::run(kEpiPartial, 2, mt, dim3((unsigned)wgs), st, g);
  return e ? -e : g.pieces;
}

// Whether a layer's projections are better off as one product: up to a strip of 128 columns a unit they always
// are (13 layers, 2 .. 64 rows, 1.05 to 1.47 times as fast).  With more strips than that the one product takes two
// to a workgroup, half of which have none at 272, or shares that end amid strips, where the products by themselves
// fill the chip (34816 x 4096 of 6144 and 28672 columns at 5 / 24 / 64 rows: one 52.0 / 54.9 / 66.9 us, two 49.9 /
// 51.1 / 56.9; 43008 x 4096 of 10240 and 32768 at 24 / 64 64.6 / 77.3, 68.6 / 65.1): it is taken where the estimates put it
// a tenth ahead, which no layer that lost by it reaches (20 layers of 33 to 66 thousand columns).
CAKE_API int cake_gemm_sections_gain(int M, int n1, int n2, int N, int K) {
  if (M < 1 || M > 64 || n1 < 0 || n2 < n1 || N < n2 || N < 1 || K < 1) return 0;
  if (N <= 256 * 128) return 1;
  double apart = 0;
  int kind;
  for (const int n : {n1, n2 - n1, N - n2})
    if (n > 0) apart += rows_best(M, n, K, false, &kind);
  return 1.1 * stream_plan(M, N, K, false).us <= apart;
}

// A layer's projections in one launch of the stream form, by columns: [0, n1) to c1 (16-bit), [n1, n2) to r32,
// [n2, N) gelu to c.  n1, n2 multiples of 4; bases 16-byte aligned; ws, tick as above.
CAKE_API int cake_gemm_rows_sections(int dt, const void* a, long long lda, const void* b, long long ldb, void* c1,
                                     long long ldc1, float* r32, long long ldr, void* c, long long ldc, int n1,
                                     int n2, float* ws, void* tick, const void* zeros, int M, int N, int K,
                                     hipStream_t st) {
  if (M < 1 || M > 64 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || n1 < 0 || n2 < n1 || n2 > N ||
      n1 % 4 || n2 % 4 || (n1 > 0 && !c1) || (n2 > n1 && !r32) || (N > n2 && !c) || !ws || !tick || !zeros ||
      (((uintptr_t)c1 | (uintptr_t)r32 | (uintptr_t)c) & 15))
    return (int)hipErrorInvalidValue;
  const StreamPlan sp = stream_plan(M, N, K, false);
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c; g.c1 = (uint16_t*)c1;
  g.r32 = r32; g.ws = ws; g.tick = (unsigned*)tick; g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc; g.ldc1 = ldc1; g.ldr = ldr;
  g.M = M; g.N = g.Nv = g.half = N; g.K = K; g.n1 = n1; g.n2 = n2;
  g.tiles_m = 1;
  g.tiles_n = (N + sp.bn - 1) / sp.bn;
  if (g.tiles_n > kRowsTicks) return (int)hipErrorInvalidValue;
  g.kps = sp.per;
  return dt == kBF16 ? Rows<kBF16>::run(kEpiSections, 2, (M + 15) / 16, dim3(sp.wgs), st, g)
         : dt == kF16 ? Rows<kF16>::run(kEpiSections, 2, (M + 15) / 16, dim3(sp.wgs), st, g) : (int)hipErrorInvalidValue;
}

// cake_gemm_grouped in the stream form: tiles of at most 16 rows; ws and tick as above (ws of 16
// rows).  More strips than counters, or steps than the kernel's indexes hold (1024 experts of 4096
// columns with 1500 rows): the 64-row tile, which takes the same tile list.
CAKE_API int cake_gemm_rows_grouped(int dt, int epi, const void* a, long long lda, const void* b,
                                    long long ldb, long long b_group, void* c, long long ldc,
                                    const void* tiles, int max_tiles, float* ws, void* tick,
                                    const void* zeros, int N, int K, hipStream_t st) {
  const StreamPlan sp = stream_plan(1, N, K, false);
  const long long strips = (long long)max_tiles * ((N + sp.bn - 1) / sp.bn);
  if (max_tiles <= 0 || N <= 0 || K <= 0 || K % 8 || lda % 8 || ldb % 8 || b_group % 8 ||
      !(epi == 0 || (epi >= 7 && epi <= 10)) || !ws || !tick || !zeros)
    return (int)hipErrorInvalidValue;
  if (strips > kRowsTicks || strips * ((K + sp.kst - 1) / sp.kst) >= 0x40000000LL)
    return cake_gemm_grouped(dt, epi, 4, a, lda, b, ldb, b_group, c, ldc, tiles, max_tiles, zeros, N,
                             K, st);
  GemmArgs g{};
  g.a = (const uint16_t*)a; g.b = (const uint16_t*)b; g.c = (uint16_t*)c;
  g.ws = ws; g.tick = (unsigned*)tick; g.zeros = (const uint16_t*)zeros;
  g.lda = lda; g.ldb = ldb; g.ldc = ldc;
  g.N = N; g.K = K; g.Nv = N; g.half = N;
  g.tiles_m = max_tiles;
  g.tiles_n = (N + sp.bn - 1) / sp.bn;
  g.kps = kRowsMinK / sp.kst;
  g.groups = (const int4*)tiles;
  g.b_group = b_group;
  return dt == kBF16 ? Rows<kBF16>::grouped(epi, dim3(sp.most), st, g)
         : dt == kF16 ? Rows<kF16>::grouped(epi, dim3(sp.most), st, g) : (int)hipErrorInvalidValue;
}
