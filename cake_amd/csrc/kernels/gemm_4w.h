// Four-wave MFMA GEMM tiles (plan cfg 22-38; shapes and schedules below): the projections of
// prompts.
//
// Included by gemm_kernel.h (launch_gemm dispatches them here); same GemmArgs, tile
// order, swizzled LDS image, fragment reads and epilogues as gemm_kernel's IL path.
//
// The shape of the winning library kernel on this chip (hipBLASLt's 256x256x64 tile,
// profiles/r6_gemm_pmc_8192.txt): one wave per SIMD, 128 x 128 outputs per wave, LDS-DMA
// staging, 32 fragment reads per k-step.  At one wave per SIMD every instruction beside
// the MFMAs is paid in MFMA gaps (16 cycles, 8 of them free), so a DMA piece is three
// instructions and nothing else (k-loop stamps: profiles/r6_gemm_stamps.jsonl):
//   * buffer_load_dwordx4 ... offen lds with two per-lane byte offset VGPRs per operand (the
//     lane's row of an instruction's eight and its swizzled 16-byte chunk) and the rows'
//     offset as a loop-invariant scalar soffset;
//   * the k step in the descriptor: its base advanced and num_records shrunk per step (a
//     handful of scalar ops per step, not per piece); rows past the matrix and steps past
//     the split read through the range check as zeros (no per-issue select, no zeros
//     page); gated (SwiGLU / GEGLU) weights keep a constant row stride per group (16 gate
//     + 16 up rows), so the same form covers them;
//   * the M0 write (buffer base + the piece's offset as an immediate) and the DMA in one
//     asm statement with the MFMA it is scheduled behind, which also covers M0's wait state.
//   Needs K and the split's k range in whole 64-element steps and operands under 2 GB
//   (host-checked).
#pragma once

// Diagnostic build only (scripts/gemm_stamp.hip defines CAKE_GEMM_STAMPS and the
// g_gemm_stamps buffer): s_memtime at the k-loop's segment boundaries, summed per wave.
#ifdef CAKE_GEMM_STAMPS
#define CAKE_STAMP(v)                                                                   \
  do {                                                                                  \
    __builtin_amdgcn_sched_barrier(0);                                                  \
    asm volatile("s_memtime %0\n\ts_waitcnt lgkmcnt(0)" : "=s"(v)::"memory");           \
    __builtin_amdgcn_sched_barrier(0);                                                  \
  } while (0)
#else
#define CAKE_STAMP(v) \
  do {                \
  } while (0)
#endif

namespace cake {

constexpr int k4WCfg = 22;     // plan cfg id of the 256 x 256 tile
constexpr int k4WCfg192 = 23;  // 256 x 192 (8B q|k|v: 6144 = 32 x 192 columns, 256 tiles at
                               // 2048 tokens instead of 192)
constexpr int k4WCfg128 = 24;  // 128 x 256 (8B o / down at 2048 tokens: 256 tiles, not 128)
constexpr int k4WSched = 3;    // cfg + 3: the same tiles on three barriers (25, 26), on one (27)
constexpr int k4WLast = 38;    // 28 .. 38: the tiles of CAKE_GEMM_4W_TILES
inline bool four_wave_cfg(int cfg) { return cfg >= k4WCfg && cfg <= k4WLast; }
// op k of an alternating sequence of nr reads and nd DMAs (the longer list's tail last):
// kind 0 = read, 1 = DMA, and its index within its list
constexpr int alt_kind(int nr, int nd, int k) {
  return k < 2 * (nr < nd ? nr : nd) ? k % 2 : (nr > nd ? 0 : 1);
}
constexpr int alt_idx(int nr, int nd, int k) {
  const int mn = nr < nd ? nr : nd;
  return k < 2 * mn ? k / 2 : mn + (k - 2 * mn);
}

// LDS-DMA of one 1 KiB piece (buffer_load_dwordx4 ... offen lds) with the M0 write in the
// same statement (M0 is not preserved around inline asm); d = the buffer descriptor as an
// SGPR quad; the add sets SCC, where the compiler may keep a comparison.  amfma_dma issues an
// MFMA between the M0 write and the DMA, which covers the write's wait state (no s_nop) and
// keeps the DMA beside the MFMA it was scheduled with.
template <int OFF>
__device__ __forceinline__ void dma16(uint32_t mb, uint32_t voff, cu32x4 d, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(mb), "v"(voff), "s"(d), "s"(soff), "i"(OFF) : "memory", "scc");
}
template <int DT, int OFF>
__device__ __forceinline__ void amfma_dma(cf32x4& acc, const uint4& a, const uint4& b, uint32_t mb,
                                          uint32_t voff, cu32x4 d, uint32_t soff) {
  const cu32x4 av = __builtin_bit_cast(cu32x4, a), bv = __builtin_bit_cast(cu32x4, b);
  if constexpr (DT == kBF16)
    asm volatile("s_add_u32 m0, %3, %7\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                 "buffer_load_dwordx4 %4, %5, %6 offen lds"
                 : "+a"(acc)
                 : "v"(av), "v"(bv), "s"(mb), "v"(voff), "s"(d), "s"(soff), "i"(OFF)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %3, %7\n\tv_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\t"
                 "buffer_load_dwordx4 %4, %5, %6 offen lds"
                 : "+a"(acc)
                 : "v"(av), "v"(bv), "s"(mb), "v"(voff), "s"(d), "s"(soff), "i"(OFF)
                 : "memory", "scc");
}

// ... and with the piece's offset in a register
__device__ __forceinline__ void dma16_at(uint32_t mb, uint32_t off, uint32_t voff, cu32x4 d, uint32_t soff) {
  asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :: "s"(mb), "v"(voff), "s"(d), "s"(soff), "s"(off) : "memory", "scc");
}
template <int DT>
__device__ __forceinline__ void amfma_dma_at(cf32x4& acc, const uint4& a, const uint4& b, uint32_t mb,
                                             uint32_t off, uint32_t voff, cu32x4 d, uint32_t soff) {
  const cu32x4 av = __builtin_bit_cast(cu32x4, a), bv = __builtin_bit_cast(cu32x4, b);
  if constexpr (DT == kBF16)
    asm volatile("s_add_u32 m0, %3, %7\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0\n\t"
                 "buffer_load_dwordx4 %4, %5, %6 offen lds"
                 : "+a"(acc)
                 : "v"(av), "v"(bv), "s"(mb), "v"(voff), "s"(d), "s"(soff), "s"(off)
                 : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %3, %7\n\tv_mfma_f32_16x16x32_f16 %0, %1, %2, %0\n\t"
                 "buffer_load_dwordx4 %4, %5, %6 offen lds"
                 : "+a"(acc)
                 : "v"(av), "v"(bv), "s"(mb), "v"(voff), "s"(d), "s"(soff), "s"(off)
                 : "memory", "scc");
}

// Of a grouped product, workgroup bid's row tile and column tile (n x tiles_n of them): dealt out to the XCDs in
// runs; most groups have one or two row tiles, so two of them walk all columns and their rows are read once (eight
// read every row four times over; 64 groups of 192 rows of 4096 to 3616 columns 509 -> 483 us, back 543 -> 506)
__device__ __forceinline__ int2 grouped_place(int n, int tiles_n, int bid) {
  const int all = n * tiles_n, q = all / 8, r = all % 8, x = bid % 8;
  const int id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + bid / 8;
  const int per = 2 * tiles_n, first = id / per * 2, gm = min(2, n - first);
  return make_int2(first + id % per % gm, id % per / gm);
}

// SCHED 1: three barriers a k step (the DMAs of step t+2 issued as soon as every wave has read the
// operand region they overwrite).  SCHED 2: one barrier, for tiles of which the LDS holds three or
// four k steps.  A step of a small tile is bound by its waits, not by the matrix cores: 192 x 192 is
// 0.49 us of MFMAs and took 0.75 us alone on the chip (0.63 with one barrier), 1.13 on all CUs (0.98);
// 128 x 256 0.44, 0.72 (0.62), 1.11 (0.99).  More steps in flight alone changed neither.  Tiles of
// two steps (256 x 192 and larger) are within 3 % either way.
// GRP: grouped row tiles (GemmArgs::groups), K any multiple of 8.
// PCS: the tiles past the last whole wave in k pieces (GemmArgs::pieces); an instance of its own,
// since the sums of pieces spill twice the registers in the epilogue of whole tiles too (4096^3 with
// the residual 113.3 us with them, 109.9 without).
template <int BM, int BN, int SCHED> struct FourWave {
  static constexpr int BUF = (BM + BN) * 128;  // 64 KB at most per k-step buffer
  static constexpr int NBUF = SCHED != 2 ? 2 : 160 * 1024 / BUF > 4 ? 4 : 160 * 1024 / BUF;
};
template <int DT, int EPI, int BM, int BN, int SCHED, bool GRP, bool PCS>
__device__ __forceinline__ void gemm_4w_tile(GemmArgs g, uint8_t* smem) {
  static_assert(BM % 32 == 0 && BN % 64 == 0, "whole fragments, gated pairs within a wave");
  constexpr int WTM = BM / 2, WTN = BN / 2, FM = WTM / 16, FN = WTN / 16;
  constexpr int BUF = FourWave<BM, BN, SCHED>::BUF, NBUF = FourWave<BM, BN, SCHED>::NBUF;
  static_assert(SCHED != 2 || NBUF > 2, "one barrier a step: three steps in the LDS");
  constexpr int IPW = (BM + BN) / 32;   // DMA wave-instructions per wave per k-step
  constexpr int NA = BM / 32;           // of which A
  static_assert(IPW == FM + FN, "the second half alternates one DMA with one fragment read");
  constexpr int STG_LD = WTN + 4, STG = 16 * STG_LD * 4;
  static_assert(8 * STG <= NBUF * BUF - 16, "epilogue staging (2 slices per wave) fits the operand buffers");

  const int tid = threadIdx.x, lane = tid & 63;
#ifdef CAKE_GEMM_STAMPS
  unsigned long long st_[8] = {0, 0, 0, 0, 0, 0, 0, 0}, t_entry;
  CAKE_STAMP(t_entry);
#endif
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wc = wave & 1;

  // ---- XCD-aware grouped tile order (as gemm_kernel) ---------------------
  // Pieces (PCS): workgroups [0, dp_tiles) run whole tiles, the rest run the remaining tiles
  // in equal k pieces — the last partial wave of a grid at a fraction of its length (8B gate|up
  // at 2048 tokens: 896 tiles = 3 full waves + 128 tiles in halves), or every tile in pieces
  // when there are too few.  Equal pieces of all tiles walk k side by side and share their
  // operands in L2, so an XCD takes neighbouring tiles of one piece (with the pieces of a tile side
  // by side it read most of both operands: 1100 x 4096 x 23552 in 224 x 192 tiles 203 us, 191 so);
  // one line of k steps cut into 256 equal shares (a tile's pieces at any k)
  // balanced better and ran at half the rate, every workgroup reading for itself.
  if constexpr (GRP) g.tiles_m = g.groups[g.tiles_m].x;
  const int ntiles = g.tiles_m * g.tiles_n;
  if (GRP && (int)blockIdx.x >= ntiles) return;
  int id, piece = 0;
  int kb = 0, ke = g.K;
  {
    const int dp = PCS ? g.dp_tiles : ntiles;   // (a multiple of 8 where pieces follow)
    const bool whole = !PCS || (int)blockIdx.x < dp;
    const int n = whole ? dp : (int)gridDim.x - dp, bid = whole ? blockIdx.x : blockIdx.x - dp;
    const int q = n / 8, r = n % 8, x = bid % 8, i = bid / 8;
    id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i;
    if (PCS && !whole) {   // the first pieces of all these tiles, then the second ones, ..
      const int rest = n / g.pieces;
      piece = id / rest;
      id = dp + id % rest;
      kb = piece * g.kps;
      ke = min(g.K, kb + g.kps);
    }
  }
  const int pieces = PCS && (int)blockIdx.x >= g.dp_tiles ? g.pieces : 1;
  constexpr int GROUP = 8;
  const int per_group = GROUP * g.tiles_n;
  const int first_m = (id / per_group) * GROUP;
  const int gm = min(GROUP, g.tiles_m - first_m);
  const int2 at = GRP ? grouped_place(g.tiles_m, g.tiles_n, blockIdx.x)
                      : make_int2(first_m + (id % per_group) % gm, (id % per_group) / gm);
  const int tm = at.x;
  const int m0 = GRP ? 0 : tm * BM;
  const int n0 = at.y * BN;
  int group = 0;
  if constexpr (GRP) {
    const int4 t = g.groups[tm];
    group = t.x;
    g.a += (size_t)t.y * g.lda;
    g.c += (size_t)t.y * g.ldc;
    g.b += (size_t)t.x * g.b_group + (size_t)n0 * g.ldb;
    g.M = min(t.z, BM);
  }
  const int nk = GRP ? (ke - kb + kGBK - 1) / kGBK : (ke - kb) / kGBK;

  // ---- DMA: an instruction fills 8 LDS rows, lane l row l/8, slot l%8 of it holding source chunk
  // (l%8) ^ ((row >> 1) & 7).  A wave's instructions take rows side by side, 8 NA of A and 8 NB of B:
  // with the waves' rows 8 apart (one 32-row group an instruction) the rows in flight at a time met on
  // few channels of the memory where k is an odd multiple of 1024 or so (8 x 32 tiles of 128 x 256, k
  // 5120 95 -> 77 us, 23552 364 -> 340, 28672 460 -> 402; 256 x 256 148 -> 130, 624 -> 588, 805 -> 699)
  // SCHED 0 takes weight rows of 4096, 8192, .. the other way, since there the rows that waves have side by
  // side are the ones that meet: 6000 x 28672 x 4096 SwiGLU 1063 us side by side, 1047 8 rows apart,
  // plain 1094, 1062; 2048 x 16384 x 2048 103.9, 104.8.  (SCHED 1 is even there.)
  constexpr int NB = IPW - NA;
  constexpr bool EITHER = SCHED == 0 && !GRP;
  const bool apart = EITHER && g.ldb >= 4096 && (g.ldb & (g.ldb - 1)) == 0;
  const int l8 = lane >> 3;
  const int rA = wave * (apart ? 8 : NA * 8) + l8, rB = wave * (apart ? 8 : NB * 8) + l8;
  const int chunk_a = (lane & 7) ^ ((rA >> 1) & 7), chunk_b = (lane & 7) ^ ((rB >> 1) & 7);
  // (grouped: weights from this tile's first row on, so that a tile, not a weight, is under 2 GB)
  const long long brows = GRP ? min(BN, g.Nv - n0) : g.gated ? 2LL * g.half : (long long)g.Nv;
  const int nrec_a = (int)(((long long)(g.M - 1) * g.lda + g.K) * 2);
  const int nrec_b = (int)(((brows - 1) * g.ldb + g.K) * 2);
  // scalar byte offsets of each instruction's rows: loop-invariant SGPRs.  Gated: virtual rows 32 b ..
  // are 16 gate rows from 16 b on and the 16 up rows beside them
  const uint32_t gstride_a = (uint32_t)((apart ? 32LL : 8LL) * g.lda * 2);
  uint32_t soff_b[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int q = apart ? 4 * j + wave : wave * NB + j;
    const long long row = !g.gated ? (apart ? 32 : 8) * j : q / 4 * 16 + q % 2 * 8 + (q % 4 < 2 ? 0 : g.half);
    soff_b[j] = __builtin_amdgcn_readfirstlane((uint32_t)(row * g.ldb * 2));
  }
  const long long brow0 = GRP ? rB : g.gated ? n0 / 2 + l8 : n0 + rB;
  // byte offsets of this lane, of the even and the odd instructions (rows 8 on: the chunk's bit 2)
  const int odd = apart ? 0 : 4;
  const auto voff = [](long long row, long long ld, int chunk) { return (uint32_t)((row * ld + chunk * 8) * 2); };
  const uint32_t voff_a[2] = {voff(m0 + rA, g.lda, chunk_a), voff(m0 + rA, g.lda, chunk_a ^ odd)};
  const uint32_t voff_b[2] = {voff(brow0, g.ldb, chunk_b), voff(brow0, g.ldb, chunk_b ^ odd)};
  // The k step lives in the descriptors: base advanced to the step's first column and
  // num_records shrunk by as much (a step past the split's end: 0 records, every lane out
  // of range -> zeros, no memory traffic).  Per DMA that leaves the M0 write and the DMA
  // itself in the MFMA stream, the rest is a handful of scalar ops per k-step.
  // descriptor words: base (48 bits, stride 0), num_records, flags (raw, offen)
  auto desc_at = [&](const uint16_t* base, int nrec, int step) __attribute__((always_inline)) {
    const int k0 = kb + step * kGBK;
    const unsigned long long p = (unsigned long long)(base + k0);
    cu32x4 d;
    d[0] = __builtin_amdgcn_readfirstlane((unsigned)p);
    d[1] = __builtin_amdgcn_readfirstlane((unsigned)(p >> 32) & 0xFFFFu);
    d[2] = __builtin_amdgcn_readfirstlane(step < nk ? (unsigned)(nrec - 2 * k0) : 0u);
    d[3] = 0x00020000u;
    return d;
  };
  auto src_a = [&](int step) __attribute__((always_inline)) { return desc_at(g.a, nrec_a, step); };
  auto src_b = [&](int step) __attribute__((always_inline)) { return desc_at(g.b, nrec_b, step); };
  const uint32_t m0_a = __builtin_amdgcn_readfirstlane(lds_off(smem) + (uint32_t)wave * (apart ? 1024 : NA * 1024));
  const uint32_t m0_b = __builtin_amdgcn_readfirstlane(lds_off(smem) + BM * 128u + (uint32_t)wave * (apart ? 1024 : NB * 1024));
  const uint32_t piece_b = apart ? 4096 : 1024;   // LDS bytes from an instruction's rows to the next one's
  // M0 = buffer base + piece_b per piece (an immediate where it is always 1 KiB) / voffset / soffset
  // of DMA I (A pieces for I < NA) into buffer buf
  auto dma_mb = [&](int buf, int i) __attribute__((always_inline)) {
    return (i < NA ? m0_a : m0_b) + (uint32_t)(buf * BUF);
  };
  // GRP: the last step of a K that is no multiple of 64 reads its missing chunks out of range
  // (the descriptors only bound the matrix, a row's end lies inside it)
  uint32_t cur_a[2] = {voff_a[0], voff_a[1]}, cur_b[2] = {voff_b[0], voff_b[1]};
  auto tail_step = [&](int step) __attribute__((always_inline)) {
    if constexpr (GRP) {
#pragma unroll
      for (int o = 0; o < 2; ++o) {
        cur_a[o] = step * kGBK + (chunk_a ^ 4 * o) * 8 < g.K ? voff_a[o] : 0x80000000u;
        cur_b[o] = step * kGBK + (chunk_b ^ 4 * o) * 8 < g.K ? voff_b[o] : 0x80000000u;
      }
    }
  };
  auto dma_voff = [&](int i) __attribute__((always_inline)) {
    return i < NA ? cur_a[i % 2] : cur_b[(i - NA) % 2];
  };
  auto dma_soff = [&](int i) __attribute__((always_inline)) {
    return i < NA ? (uint32_t)i * gstride_a : soff_b[i < NA ? 0 : i - NA];
  };
  auto stage_one = [&](const cu32x4& sa, const cu32x4& sb, int buf, auto I)
                       __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    constexpr int n = i < NA ? i : i - NA;
    if constexpr (EITHER) dma16_at(dma_mb(buf, i), n * piece_b, dma_voff(i), i < NA ? sa : sb, dma_soff(i));
    else dma16<n * 1024>(dma_mb(buf, i), dma_voff(i), i < NA ? sa : sb, dma_soff(i));
  };
  // MFMA with DMA I fused behind it
  auto mfma_dma = [&](cf32x4& c, const uint4& a, const uint4& b, const cu32x4& sa,
                      const cu32x4& sb, int buf, auto I) __attribute__((always_inline)) {
    constexpr int i = decltype(I)::value;
    constexpr int n = i < NA ? i : i - NA;
    if constexpr (EITHER)
      amfma_dma_at<DT>(c, a, b, dma_mb(buf, i), n * piece_b, dma_voff(i), i < NA ? sa : sb, dma_soff(i));
    else
      amfma_dma<DT, n * 1024>(c, a, b, dma_mb(buf, i), dma_voff(i), i < NA ? sa : sb, dma_soff(i));
  };
  auto stage = [&](int step, int buf) {
    const cu32x4 sa = src_a(step), sb = src_b(step);
    tail_step(step);
    static_for<0, IPW>([&](auto I) __attribute__((always_inline)) { stage_one(sa, sb, buf, I); });
  };

  cf32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) azero(acc[i][j]);
  // ---- fragment addresses (as gemm_kernel) ----------------------------------
  const int swz = (lane & 15) >> 1;
  const uint32_t lrow = (uint32_t)(lane & 15) * 128;
  const uint32_t off0 = (uint32_t)(((lane >> 4) ^ swz) * 16);
  const uint32_t off1 = (uint32_t)(((4 + (lane >> 4)) ^ swz) * 16);
  const uint32_t lds0 = lds_off(smem);
  const uint32_t a_base = lds0 + (uint32_t)(wr * WTM) * 128 + lrow;
  const uint32_t b_base = lds0 + (uint32_t)(BM + wc * WTN) * 128 + lrow;
  constexpr int NM = FM * FN, NR = FM + FN;
  uint4 af0[FM], bf0[FN], af1[FM], bf1[FN];

  if constexpr (SCHED == 1) {
    // Three barriers per k-step; a step's operand regions are restaged as soon as every
    // wave has read them, so the DMAs spread over two thirds of the step:
    //   phase 1 (k 0..31 MFMAs of t): [B k 32..63 reads] lgkm+barrier (B of t free)
    //     [A k 32..63 reads + B DMAs of t+2] lgkm+barrier (A of t free) [A DMAs]
    //   phase 2 (k 32..63 MFMAs of t): [A DMAs] vmcnt(this step's) + barrier
    //     (t+1 landed) [k 0..31 reads of t+1] lgkm
    // Each wait + barrier follows an MFMA issue, so the pipe runs while the waves align.
    // (placements measured: barriers at NM/8 and NM/2, or all A DMAs before phase 2 with its
    // barrier at MFMA 1, ran within 3 % / 3-6 % slower, profiles/r6_gemm_three_barrier_ab.txt)
    constexpr int Q1 = NM / 4, Q2 = (NM * 5) / 8, P1 = NM / 4;
    constexpr int NA1 = NA / 2;  // A DMAs in phase 1's tail, the rest in phase 2's head
    static_assert(Q1 >= FN / 2 && Q2 - Q1 - 1 >= (FM + NB) / 2, "op density");
    stage(0, 0);
    stage(1, 1);
    __builtin_amdgcn_s_waitcnt(vm_wait(IPW));
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < FM; ++i) af0[i] = ds_read16(a_base + i * 16 * 128 + off0);
#pragma unroll
    for (int j = 0; j < FN; ++j) bf0[j] = ds_read16(b_base + j * 16 * 128 + off0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    int buf = 0;
    for (int t = 0; t < nk; ++t) {
      const uint32_t ab = a_base + buf * BUF, bb = b_base + buf * BUF;
      const int nbuf = buf ^ 1;
      const uint32_t na = a_base + nbuf * BUF, nb = b_base + nbuf * BUF;
      const cu32x4 sa = src_a(t + 2), sb = src_b(t + 2);
      tail_step(t + 2);
      // ops k of n spread over MFMAs [lo, hi): op k after MFMA lo + floor(k (hi-lo) / n)
      static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
        constexpr int m = decltype(mi)::value;
        // the first op placed after this MFMA, when it is a DMA, goes in the MFMA's statement
        constexpr int L2 = Q2 - Q1 - 1, n2 = FM + NB, m2 = m - Q1 - 1;
        constexpr int L3 = NM - Q2 - 1, m3 = m - Q2 - 1;
        constexpr int k2 = (m2 * n2 + L2 - 1) / L2, k2e = ((m2 + 1) * n2 + L2 - 1) / L2;
        constexpr int k3 = (m3 * NA1 + L3 - 1) / L3, k3e = ((m3 + 1) * NA1 + L3 - 1) / L3;
        constexpr int fd = (m > Q1 && m < Q2 && k2 < k2e && alt_kind(FM, NB, k2) == 1)
                               ? NA + alt_idx(FM, NB, k2)
                               : (m > Q2 && k3 < k3e) ? k3 : -1;
        if constexpr (fd >= 0) mfma_dma(acc[m / FN][m % FN], af0[m / FN], bf0[m % FN], sa, sb, buf, std::integral_constant<int, fd>{});
        else amfma_v<DT>(acc[m / FN][m % FN], af0[m / FN], bf0[m % FN]);
        if constexpr (m < Q1) {
          static_for<(m * FN + Q1 - 1) / Q1, ((m + 1) * FN + Q1 - 1) / Q1>([&](auto ji)
                                                                    __attribute__((always_inline)) {
            constexpr int j = decltype(ji)::value;
            bf1[j] = ds_read16_off<j * 16 * 128>(bb + off1);
          });
        } else if constexpr (m == Q1 || m == Q2) {
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        } else if constexpr (m < Q2) {
          static_for<k2 + (fd >= 0 ? 1 : 0), k2e>([&](auto ki) __attribute__((always_inline)) {
            constexpr int k = decltype(ki)::value;  // reads and DMAs alternate
            if constexpr (alt_kind(FM, NB, k) == 0)
              af1[alt_idx(FM, NB, k)] = ds_read16_off<alt_idx(FM, NB, k) * 16 * 128>(ab + off1);
            else
              stage_one(sa, sb, buf, std::integral_constant<int, NA + alt_idx(FM, NB, k)>{});
          });
        } else {
          static_for<k3 + (fd >= 0 ? 1 : 0), k3e>([&](auto ki) __attribute__((always_inline)) {
            stage_one(sa, sb, buf, ki);
          });
        }
      });
      static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
        constexpr int m = decltype(mi)::value;
        constexpr int n1 = NA - NA1;
        constexpr int k1 = (m * n1 + P1 - 1) / P1, k1e = ((m + 1) * n1 + P1 - 1) / P1;
        constexpr int fd = (m < P1 && k1 < k1e) ? NA1 + k1 : -1;
        if constexpr (fd >= 0) mfma_dma(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN], sa, sb, buf, std::integral_constant<int, fd>{});
        else amfma_v<DT>(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN]);
        if constexpr (m < P1) {
          static_for<k1 + (fd >= 0 ? 1 : 0), k1e>([&](auto ki) __attribute__((always_inline)) {
            stage_one(sa, sb, buf, std::integral_constant<int, NA1 + decltype(ki)::value>{});
          });
        } else if constexpr (m == P1) {
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_waitcnt(vm_wait(IPW));  // step t+1's DMAs landed
          asm volatile("s_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        } else {
          constexpr int L = NM - P1 - 1, mm = m - P1 - 1;
          static_for<(mm * NR + L - 1) / L, ((mm + 1) * NR + L - 1) / L>([&](auto ri)
                                                                   __attribute__((always_inline)) {
            constexpr int r = decltype(ri)::value;
            if constexpr (r < FM) af0[r] = ds_read16_off<r * 16 * 128>(na + off0);
            else bf0[r - FM] = ds_read16_off<(r - FM) * 16 * 128>(nb + off0);
          });
        }
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      // the last MFMAs' results settle before the loop is left: a spill may read them first thing
      // (on every step: asked for on the last one only, the branch cost whole tiles that leave the
      // clock up to 9 %, 2048 x 4096 x 14336 281 us against 257)
      asm volatile("s_nop 7" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      buf = nbuf;
    }
  } else if constexpr (SCHED == 2) {
    // One barrier a k step, early in its second half: by then every wave has read all of step t (its
    // buffer takes step t + NBUF) and waits for its own DMAs of step t+1.
    //   first half: MFMAs of k 0..31, reads of k 32..63
    //   second half: MFMAs of k 32..63, after the P-th of them vmcnt + barrier, then reads of
    //     k 0..31 of t+1
    // The reads end LAT MFMAs before their half does (their latency); the DMAs of a step are spread
    // from barrier to barrier, ND2 of them before the next step begins.
    constexpr int P = 2, LAT = 7;
    constexpr int R1 = NM - LAT, W2 = NM - P - 1, R2 = W2 - LAT;   // MFMAs that reads, DMAs follow
    constexpr int ND2 = IPW / 2, ND1 = IPW - ND2;
    static_assert(R2 >= NR / 2 && W2 >= ND2, "op density");
    static_for<0, NBUF - 1>([&](auto i) __attribute__((always_inline)) { stage(i, i); });
    {  // the first part of the last buffered step, as the loop leaves it
      const cu32x4 sa = src_a(NBUF - 1), sb = src_b(NBUF - 1);
      tail_step(NBUF - 1);
      static_for<0, ND2>([&](auto I) __attribute__((always_inline)) { stage_one(sa, sb, NBUF - 1, I); });
    }
    __builtin_amdgcn_s_waitcnt(vm_wait((NBUF - 2) * IPW + ND2));
    asm volatile("s_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < FM; ++i) af0[i] = ds_read16(a_base + i * 16 * 128 + off0);
#pragma unroll
    for (int j = 0; j < FN; ++j) bf0[j] = ds_read16(b_base + j * 16 * 128 + off0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    int buf = 0;
    cu32x4 sa = src_a(NBUF - 1), sb = src_b(NBUF - 1);
    for (int t = 0; t < nk; ++t) {
      const uint32_t ab = a_base + buf * BUF, bb = b_base + buf * BUF;
      const int nbuf = buf + 1 == NBUF ? 0 : buf + 1, pbuf = buf == 0 ? NBUF - 1 : buf - 1;
      const uint32_t na = a_base + nbuf * BUF, nb = b_base + nbuf * BUF;
      tail_step(t + NBUF - 1);
      static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
        constexpr int m = decltype(mi)::value;
        constexpr int d0 = (m * ND1 + NM - 1) / NM, d1 = ((m + 1) * ND1 + NM - 1) / NM;
        if constexpr (d0 < d1) mfma_dma(acc[m / FN][m % FN], af0[m / FN], bf0[m % FN], sa, sb, pbuf, std::integral_constant<int, ND2 + d0>{});
        else amfma_v<DT>(acc[m / FN][m % FN], af0[m / FN], bf0[m % FN]);
        if constexpr (m < R1)
          static_for<(m * NR + R1 - 1) / R1, ((m + 1) * NR + R1 - 1) / R1>([&](auto ri) __attribute__((always_inline)) {
            constexpr int r = decltype(ri)::value;
            if constexpr (r < FN) bf1[r] = ds_read16_off<r * 16 * 128>(bb + off1);
            else af1[r - FN] = ds_read16_off<(r - FN) * 16 * 128>(ab + off1);
          });
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      sa = src_a(t + NBUF);
      sb = src_b(t + NBUF);
      tail_step(t + NBUF);
      static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
        constexpr int m = decltype(mi)::value, mm = m - P - 1;
        constexpr int d0 = mm < 0 ? 0 : (mm * ND2 + W2 - 1) / W2, d1 = mm < 0 ? 0 : ((mm + 1) * ND2 + W2 - 1) / W2;
        if constexpr (d0 < d1) mfma_dma(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN], sa, sb, buf, std::integral_constant<int, d0>{});
        else amfma_v<DT>(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN]);
        if constexpr (m == P) {
          __builtin_amdgcn_sched_barrier(0);
          __builtin_amdgcn_s_waitcnt(vm_wait((NBUF - 2) * IPW));
          asm volatile("s_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        } else if constexpr (mm >= 0 && mm < R2)
          static_for<(mm * NR + R2 - 1) / R2, ((mm + 1) * NR + R2 - 1) / R2>([&](auto ri) __attribute__((always_inline)) {
            constexpr int r = decltype(ri)::value;
            if constexpr (r < FN) bf0[r] = ds_read16_off<r * 16 * 128>(nb + off0);
            else af0[r - FN] = ds_read16_off<(r - FN) * 16 * 128>(na + off0);
          });
      });
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      asm volatile("s_nop 7" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      buf = nbuf;
    }
  } else {

  // The interleaved two-stage schedule of gemm_kernel (IL, NS = 2):
  //   [kk1 reads of t | kk0 MFMAs of t] wait | vmcnt(DMA t+1) barrier
  //   [DMA t+2 into t's buffer + kk0 reads of t+1 | kk1 MFMAs of t] wait
  // Every step issues all 16 DMAs (past the split's end: out of the descriptors' range,
  // zeros) so the counted waits hold.
  constexpr int NL = IPW + NR;
  stage(0, 0);
  __builtin_amdgcn_s_waitcnt(vm_wait(0));
  asm volatile("s_barrier" ::: "memory");
  stage(1, 1);
#pragma unroll
  for (int i = 0; i < FM; ++i) af0[i] = ds_read16(a_base + i * 16 * 128 + off0);
#pragma unroll
  for (int j = 0; j < FN; ++j) bf0[j] = ds_read16(b_base + j * 16 * 128 + off0);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  int buf = 0;
  unsigned long long tp = 0, t1 = 0, t2 = 0, t3 = 0;
  CAKE_STAMP(tp);
#ifdef CAKE_GEMM_STAMPS
  st_[4] = tp - t_entry;  // prologue: tile decode, descriptors, first two steps' DMAs
#endif
  for (int t = 0; t < nk; ++t) {
    const uint32_t ab = a_base + buf * BUF, bb = b_base + buf * BUF;
    static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
      constexpr int m = decltype(mi)::value;
      amfma_v<DT>(acc[m / FN][m % FN], af0[m / FN], bf0[m % FN]);
      static_for<(m * NR + NM - 1) / NM, ((m + 1) * NR + NM - 1) / NM>([&](auto ri)
                                                                    __attribute__((always_inline)) {
        constexpr int r = decltype(ri)::value;
        if constexpr (r < FM) af1[r] = ds_read16_off<r * 16 * 128>(ab + off1);
        else bf1[r - FM] = ds_read16_off<(r - FM) * 16 * 128>(bb + off1);
      });
    });
    CAKE_STAMP(t1);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const int nbuf = buf ^ 1;
    __builtin_amdgcn_s_waitcnt(vm_wait(0));  // DMA of step t+1 landed
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    CAKE_STAMP(t2);
    const uint32_t na = a_base + nbuf * BUF, nb = b_base + nbuf * BUF;
    const cu32x4 sa = src_a(t + 2), sb = src_b(t + 2);
    tail_step(t + 2);
    static_for<0, NM>([&](auto mi) __attribute__((always_inline)) {
      constexpr int m = decltype(mi)::value;
      constexpr int l0 = (m * NL + NM - 1) / NM, l1 = ((m + 1) * NL + NM - 1) / NM;
      constexpr bool fuse = l0 < l1 && l0 % 2 == 0 && l0 / 2 < IPW;
      if constexpr (fuse) mfma_dma(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN], sa, sb, buf, std::integral_constant<int, l0 / 2>{});
      else amfma_v<DT>(acc[m / FN][m % FN], af1[m / FN], bf1[m % FN]);
      static_for<l0 + (fuse ? 1 : 0), l1>([&](auto li) __attribute__((always_inline)) {
        constexpr int l = decltype(li)::value;
        if constexpr (l % 2 == 0 && l / 2 < IPW) {  // DMAs and reads alternate
          stage_one(sa, sb, buf, std::integral_constant<int, l / 2>{});
        } else {
          constexpr int r = (l - 1) / 2;
          if constexpr (r < FM) af0[r] = ds_read16_off<r * 16 * 128>(na + off0);
          else bf0[r - FM] = ds_read16_off<(r - FM) * 16 * 128>(nb + off0);
        }
      });
    });
    CAKE_STAMP(t3);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    asm volatile("s_nop 7" ::: "memory");  // (as above)
    __builtin_amdgcn_sched_barrier(0);
    buf = nbuf;
#ifdef CAKE_GEMM_STAMPS
    unsigned long long t4;
    CAKE_STAMP(t4);
    st_[0] += t1 - tp; st_[1] += t2 - t1; st_[2] += t3 - t2; st_[3] += t4 - t3;
    tp = t4;
#endif
  }
#ifdef CAKE_GEMM_STAMPS
  st_[5] = tp;  // loop end; the epilogue's length is taken at the kernel's end
#endif
  (void)tp; (void)t1; (void)t2; (void)t3;

  }

  // ---- epilogue (as gemm_kernel) -----------------------------------------
#pragma unroll
  for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[FM - 1][j]));
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int j = 0; j < FN; ++j) asm volatile("" : "+a"(acc[FM - 1][j]));
  __builtin_amdgcn_s_waitcnt(vm_wait(0));
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  Pieces add{};
  if (pieces > 1) {
    // Counters per tile (agent scope).  Every piece but the last to arrive stores its
    // accumulators to its slab ([i][j][thread] float4, coalesced; agent scope, so no fence has to
    // write an XCD's L2 back), counts itself ready once they are there and is done; the last
    // waits for the others (they are past their arrival, so they are running: no residency
    // assumption), sums the pieces while it stages the strips, and clears the counters for the
    // next launch.  Two pieces are summed in either
    // order; of more the last parks its own too, and all are summed in piece order: the same
    // bits whichever arrives last.
    const int tile = id - g.dp_tiles;
    unsigned* tk = g.tick + tile;
    unsigned* fl = g.tick + kPieceTiles + tile;
    volatile uint32_t* bc = reinterpret_cast<volatile uint32_t*>(smem + NBUF * BUF - 16);
    if (tid == 0) bc[0] = __hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const bool last = bc[0] == (uint32_t)(pieces - 1);
    constexpr uint32_t SLAB = BM * BN * 4;
    add = Pieces{g.ws + (size_t)tile * pieces * (BM * BN), pieces * SLAB, (uint32_t)tid * 16u,
                 pieces > 2 ? 0u : (1 - piece) * SLAB, SLAB, pieces};
    if (!last || pieces > 2) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) add.store(piece * SLAB + (i * FN + j) * 4096u, acc[i][j]);
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
    }
    if (!last) {
      if (tid == 0) __hip_atomic_fetch_add(fl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return;
    }
    if (tid == 0) {
      while (__hip_atomic_load(fl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != (unsigned)(pieces - 1))
        __builtin_amdgcn_s_sleep(2);
      __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(fl, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
  float* stg = reinterpret_cast<float*>(smem + wave * STG);
  const int row_m0 = m0 + wr * WTM;
  const int vcol0 = n0 + wc * WTN;
  if constexpr (EpiW<DT, EPI, FN>::OK) {
    EpiW<DT, EPI, FN> ops;
    ops.load_bias(g, vcol0, lane);
    ops.template load_res<0>(g, row_m0, vcol0, lane);
#ifdef CAKE_GEMM_STAMPS
    unsigned long long ts0, ts1;
    CAKE_STAMP(ts0);
    st_[7] = ts0 - st_[5];  // loop end -> first strip
#endif
    // two staging slices per wave: strip i+1 is staged while strip i is read out (one
    // LDS wait per strip; a wave's LDS accesses complete in order, so restaging a slice
    // after the reads of the strip before it needs no wait)
    float* sg0 = reinterpret_cast<float*>(smem + (wave * 2) * STG);
    float* sg1 = reinterpret_cast<float*>(smem + (wave * 2 + 1) * STG);
    stage_strip_w<FN>(acc[0], sg0, lane, add);
    static_for<0, FM>([&](auto ii) __attribute__((always_inline)) {
      constexpr int i = decltype(ii)::value;
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
      if constexpr (i + 1 < FM) {
        stage_strip_w<FN>(acc[i + 1], (i & 1) ? sg0 : sg1, lane, add.strip(i + 1, FN));
        ops.template load_res<(i + 1) & 1>(g, row_m0 + (i + 1) * 16, vcol0, lane);
      }
      readout_strip_w<DT, EPI, FN, i & 1>(g, (i & 1) ? sg1 : sg0, row_m0 + i * 16, vcol0, 0,
                                          lane, ops);
    });
#ifdef CAKE_GEMM_STAMPS
    CAKE_STAMP(ts1);
    st_[6] = ts1 - ts0;  // the strips (staging + read-out + store issue)
#endif
  } else {  // 96-column wave tiles (256 x 192): 4 lanes per row
    EpiOps<DT, EPI, FN> ops;
    ops.load_bias(g, vcol0, lane);
    ops.template load_res<0>(g, row_m0 + (lane >> 2), vcol0, lane);
    static_for<0, FM>([&](auto ii) __attribute__((always_inline)) {
      constexpr int i = decltype(ii)::value;
      if constexpr (i + 1 < FM)
        ops.template load_res<(i + 1) & 1>(g, row_m0 + (i + 1) * 16 + (lane >> 2), vcol0, lane);
      epi_strip<DT, EPI, FN, i & 1>(g, acc[i], stg, row_m0 + i * 16, vcol0, 0, lane, ops,
                                    add.strip(i, FN));
    });
  }
#ifdef CAKE_GEMM_STAMPS
  {
    unsigned long long t_end;
#ifndef CAKE_STAMP_NODRAIN
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the tile's stores issued and done
#endif
    CAKE_STAMP(t_end);
    st_[5] = t_end - st_[5];
    if (lane == 0)
      for (int i = 0; i < 8; ++i) g_gemm_stamps[((size_t)blockIdx.x * 4 + wave) * 8 + i] = st_[i];
  }
#endif
}

template <int DT, int EPI, int BM, int BN, int SCHED = 0, bool PCS = false>
__global__ __launch_bounds__(256) void gemm_4w_kernel(GemmArgs g) {
  using F = FourWave<BM, BN, SCHED>;
  __shared__ __attribute__((aligned(16))) uint8_t smem[F::NBUF * F::BUF];
  gemm_4w_tile<DT, EPI, BM, BN, SCHED, false, PCS>(g, smem);
}

}  // namespace cake
