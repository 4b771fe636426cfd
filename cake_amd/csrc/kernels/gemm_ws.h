// Tiles whose operands are asked for by waves of their own.
//
// Included by gemm_kernel.h; same GemmArgs, LDS image and epilogues as gemm_4w.h.
//
// Twelve waves, three on each SIMD: eight compute (2 x 4 of a tile, two a SIMD, so that one's LDS reads hide behind the
// other's MFMAs), four ask for operands (LDS-DMA).  A CU seems to have some 20 KB of loads under way, whatever it asks
// for (an estimate from such kernels' times, no counter shows it): a step would take its bytes times their latency (330
// clocks from the L2, 1600 from the memory) / 20 KB, 1620 clocks on 192 x 192 where the MFMAs are 1152, and a wave that asks for more stands still at that instruction with everything behind
// it.  So large tiles, whose bytes the MFMAs cover, and the standing still left to waves that do nothing else (64 experts
// 4096 x 3648 at 150 rows: MFMAs alone 190 us, weights alone 300, one after the other 425 on the four waves of gemm_4w.h,
// 358 here).  192 x 256 is 144 KB of LDS and 168 registers a wave, 96 of them sums.
//
// One workgroup a CU walks over its tiles, and the asking waves run ahead across the ends of tiles: a workgroup of its own
// for each tile waits 5.5 us (its launch, the tile list, the first operands) beside 70 - 80 us of steps.  The epilogue
// stages its strips in the weights' buffer of the tile's last step, which is asked for one step later than else.
#pragma once

namespace cake {

// Steps of 64 k: of the weights, which come from the memory, three in the LDS, of x, which mostly comes from the L2, two
// or three.
template <int BM, int BN> struct WsTile {
  static constexpr int WM = 2, WN = 4, NC = WM * WN, THREADS = 64 * (NC + 4);
  static constexpr int ABUF = BM * 128, BBUF = BN * 128;
  static constexpr int AB = 3 * (ABUF + BBUF) <= 160 * 1024 ? 3 : 2;
  static constexpr int LEFT = 160 * 1024 - AB * ABUF - 3 * BBUF;
  // a wave's staging of a strip, rows four columns apart where there is room; FIT waves' in a step's buffer, the
  // others' behind all
  static constexpr int slices(int ld) { return BBUF / (64 * ld) < NC ? BBUF / (64 * ld) : NC; }
  static constexpr int PAD = (NC - slices(BN / WN + 4)) * 64 * (BN / WN + 4) <= LEFT ? 4 : 0;
  static constexpr int SLD = BN / WN + PAD, STG = 64 * SLD, FIT = slices(SLD);
  static constexpr int LDS = AB * ABUF + 3 * BBUF + (NC - FIT) * STG;
  static_assert(NC == kPieceWaves, "counters");
  static_assert(LDS <= 160 * 1024 && BM % 32 == 0 && BM >= 128 && BN % 64 == 0, "LDS");
};

// a tile, or one of a tile's k pieces
struct WsItem {
  const uint16_t *a, *b;   // its first row, its first column's weights
  uint16_t* c;
  int rows;                // of a, from a on
  int wrows;               // of b, from b on
  int m0, n0;              // of c
  int kb, nk;              // first k, steps
  int rot;                 // the step that it begins with
  int piece, rest;         // of a tile in pieces: which of them, the tile's place among such (-1: whole)
  bool once;               // its weights are read by this tile alone: they pass the L2 by, where x stays
};

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }
template <class T> __device__ __forceinline__ T* uni(T* p) {
  const unsigned long long x = (unsigned long long)p;
  return (T*)((unsigned long long)(unsigned)uni((int)(unsigned)(x >> 32)) << 32 | (unsigned)uni((int)(unsigned)x));
}

template <bool GRP, int BM, int BN>
__device__ __forceinline__ WsItem ws_item(const GemmArgs& g, int tiles_m, int bid, int items) {
  WsItem t{};
  t.rest = -1;
  t.kb = 0;
  int ke = g.K;
  if constexpr (GRP) {
    int2 at = grouped_place(tiles_m, g.tiles_n, bid);
    at.x = uni(at.x);
    at.y = uni(at.y);
    const int4 e = g.groups[at.x];
    const int group = uni(e.x), row = uni(e.y);
    t.a = g.a + (size_t)row * g.lda;
    t.c = g.c + (size_t)row * g.ldc;
    t.rows = min(uni(e.z), BM);
    t.m0 = 0;
    t.n0 = at.y * BN;
    t.b = g.b + (size_t)group * g.b_group + (size_t)t.n0 * g.ldb;
    t.wrows = min(BN, g.Nv - t.n0);
    const int before = at.x > 0 ? uni(g.groups[at.x - 1].x) : -1;
    const int behind = at.x + 1 < tiles_m ? uni(g.groups[at.x + 1].x) : -1;
    t.once = before != group && behind != group;
    // every tile begins at a k of its own: rows of 4 KB, 8 KB, .. meet on few channels of the memory while all are at the
    // same k (64 experts 2048 -> 1984 at 105 rows 130 us, 100 so; 16 of 4096 -> 4096 123, 90; 64 of 4096 -> 3648 391, 334)
    t.rot = uni((group * 7 + at.y) % ((g.K + kGBK - 1) / kGBK));
  } else {
    // the order of gemm_4w.h: an XCD's items side by side, pieces behind whole tiles
    const int dp = g.pieces > 0 ? g.dp_tiles : items;
    const bool whole = bid < dp;
    const int n = whole ? dp : items - dp, i = whole ? bid : bid - dp;
    const int q = n / 8, r = n % 8, x = i % 8;
    int id = (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i / 8;
    if (!whole) {
      const int rest = n / g.pieces;
      t.piece = uni(id / rest);
      t.rest = id - t.piece * rest;
      id = dp + t.rest;
      t.kb = t.piece * g.kps;
      ke = min(g.K, t.kb + g.kps);
    }
    constexpr int GROUP = 8;
    const int per = GROUP * g.tiles_n, blk = uni(id / per), in = id - blk * per;
    const int first = blk * GROUP, gm = min(GROUP, g.tiles_m - first), col = uni(in / gm);
    t.m0 = (first + in - col * gm) * BM;
    t.n0 = col * BN;
    t.a = g.a + (size_t)t.m0 * g.lda;
    t.c = g.c;
    t.rows = g.M - t.m0;
    const int w0 = g.gated ? t.n0 / 2 : t.n0;
    t.b = g.b + (size_t)w0 * g.ldb;
    t.wrows = (g.gated ? 2 * g.half : g.Nv) - w0;
    t.once = g.tiles_m == 1;
  }
  t.nk = (ke - t.kb + kGBK - 1) / kGBK;
  t.a = uni(t.a);
  t.b = uni(t.b);
  t.c = uni(t.c);
  return t;
}

// LDS-DMA of 1 KB (dma16 of gemm_4w.h); NT: past what the L2 keeps
template <int OFF, bool NT>
__device__ __forceinline__ void ws_dma(uint32_t mb, uint32_t voff, cu32x4 d, uint32_t soff) {
  if constexpr (NT)
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 :: "s"(mb), "v"(voff), "s"(d), "s"(soff), "i"(OFF) : "memory", "scc");
  else
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :: "s"(mb), "v"(voff), "s"(d), "s"(soff), "i"(OFF) : "memory", "scc");
}

// the sums stay in their VGPRs (left to itself the compiler moves them from one MFMA to the next)
template <int DT>
__device__ __forceinline__ void vmfma(cf32x4& acc, const uint4& a, const uint4& b) {
  const cu32x4 av = __builtin_bit_cast(cu32x4, a), bv = __builtin_bit_cast(cu32x4, b);
  if constexpr (DT == kBF16)
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(av), "v"(bv));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(av), "v"(bv));
}

// The waves that ask.  Before step f's barrier all of step f + 1 has landed; behind it the buffers of step f are free: x of
// step f + 2 and weights of f + 3 are asked for, the latter, where f is a tile's last step, behind the next barrier.
template <int BM, int BN, bool GRP>
__device__ __forceinline__ void ws_ask(const GemmArgs& g, int tiles_m, int items, uint8_t* smem, int wave, int lane) {
  using T = WsTile<BM, BN>;
  constexpr int IPW = (BM + BN) / 32, NA = BM / 32, NB = IPW - NA;
  const int l8 = lane >> 3, rA = wave * NA * 8 + l8, rB = wave * NB * 8 + l8;
  const int chunk_a = (lane & 7) ^ ((rA >> 1) & 7), chunk_b = (lane & 7) ^ ((rB >> 1) & 7);
  const auto voff = [](long long row, long long ld, int chunk) { return (uint32_t)((row * ld + chunk * 8) * 2); };
  const uint32_t voff_a[2] = {voff(rA, g.lda, chunk_a), voff(rA, g.lda, chunk_a ^ 4)};
  const uint32_t voff_b[2] = {voff(g.gated ? l8 : rB, g.ldb, chunk_b), voff(g.gated ? l8 : rB, g.ldb, chunk_b ^ 4)};
  const uint32_t stride_a = (uint32_t)(16LL * g.lda);
  uint32_t soff_b[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int q = wave * NB + j;
    const long long row = !g.gated ? 8 * j : q / 4 * 16 + q % 2 * 8 + (q % 4 < 2 ? 0 : g.half);
    soff_b[j] = __builtin_amdgcn_readfirstlane((uint32_t)(row * g.ldb * 2));
  }
  const uint32_t m0_a = __builtin_amdgcn_readfirstlane(lds_off(smem) + (uint32_t)wave * (NA * 1024));
  const uint32_t m0_b = __builtin_amdgcn_readfirstlane(lds_off(smem) + (uint32_t)(T::AB * T::ABUF) + (uint32_t)wave * (NB * 1024));

  // a walk over the steps of this workgroup's items
  struct Walk {
    WsItem t;
    int bid, step, slot;
    bool live;
  };
  Walk xa{ws_item<GRP, BM, BN>(g, tiles_m, blockIdx.x, items), (int)blockIdx.x, 0, 0, true}, xb = xa;
  const auto k_of = [&](const Walk& w) __attribute__((always_inline)) {
    const int s = w.step + w.t.rot;
    return w.t.kb + (s < w.t.nk ? s : s - w.t.nk) * kGBK;
  };
  const auto desc = [&](const Walk& w, const uint16_t* base, int rows, long long ld) __attribute__((always_inline)) {
    const int k0 = k_of(w);
    const unsigned long long p = (unsigned long long)(base + k0);
    cu32x4 d;
    d[0] = uni((int)(unsigned)p);
    d[1] = uni((int)((unsigned)(p >> 32) & 0xFFFFu));
    d[2] = uni((int)(w.live ? (unsigned)(((long long)(rows - 1) * ld + g.K - k0) * 2) : 0u));
    d[3] = 0x00020000u;
    return d;
  };
  const auto next = [&](Walk& w, int slots) __attribute__((always_inline)) {
    w.slot = w.slot + 1 == slots ? 0 : w.slot + 1;
    if (w.live && ++w.step == w.t.nk) {
      w.step = 0;
      w.bid += gridDim.x;
      w.live = w.bid < items;
      if (w.live) w.t = ws_item<GRP, BM, BN>(g, tiles_m, w.bid, items);
    }
  };
  // (the last step of a K that is no multiple of 64 reads its missing chunks out of range)
  const auto ask_a = [&]() __attribute__((always_inline)) {
    const cu32x4 d = desc(xa, xa.t.a, min(xa.t.rows, BM), g.lda);
    const int k0 = k_of(xa);
    uint32_t v[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) v[o] = k0 + (chunk_a ^ 4 * o) * 8 < g.K ? voff_a[o] : 0x80000000u;
    const uint32_t m = m0_a + xa.slot * T::ABUF;
    static_for<0, NA>([&](auto I) __attribute__((always_inline)) {
      constexpr int i = decltype(I)::value;
      ws_dma<i * 1024, false>(m, v[i % 2], d, (uint32_t)i * stride_a);
    });
    next(xa, T::AB);
  };
  const auto ask_b = [&]() __attribute__((always_inline)) {
    const cu32x4 d = desc(xb, xb.t.b, xb.t.wrows, g.ldb);
    const int k0 = k_of(xb);
    uint32_t v[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) v[o] = k0 + (chunk_b ^ 4 * o) * 8 < g.K ? voff_b[o] : 0x80000000u;
    const uint32_t m = m0_b + xb.slot * T::BBUF;
    if (xb.t.once)
      static_for<0, NB>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        ws_dma<i * 1024, true>(m, v[i % 2], d, soff_b[i]);
      });
    else
      static_for<0, NB>([&](auto I) __attribute__((always_inline)) {
        constexpr int i = decltype(I)::value;
        ws_dma<i * 1024, false>(m, v[i % 2], d, soff_b[i]);
      });
    next(xb, 3);
  };
#pragma unroll 1
  for (int i = 0; i < 3; ++i) {
    if (i < T::AB) ask_a();
    ask_b();
  }
  __builtin_amdgcn_s_waitcnt(vm_wait((T::AB - 1) * NA + 2 * NB));
  asm volatile("s_barrier" ::: "memory");
  bool late = false;   // the weights' buffer is still the last epilogue's
#pragma unroll 1
  for (int b = blockIdx.x; b < items; b += gridDim.x) {
    const int nk = GRP ? (g.K + kGBK - 1) / kGBK : ws_item<GRP, BM, BN>(g, tiles_m, b, items).nk;
#pragma unroll 1
    for (int s = 0; s < nk; ++s) {
      // younger than step f + 1: of two buffers of x the weights of f + 2, of three all of it
      if (late) __builtin_amdgcn_s_waitcnt(vm_wait((T::AB - 2) * NA));
      else __builtin_amdgcn_s_waitcnt(vm_wait((T::AB - 2) * NA + NB));
      asm volatile("s_barrier" ::: "memory");
      const bool last = s + 1 == nk;
      if (late) ask_b();   // (the older step first, as the waits count)
      ask_a();
      if (!last) ask_b();
      late = last;
    }
  }
  __builtin_amdgcn_s_waitcnt(vm_wait(0));
}

template <int DT, int EPI, int BM, int BN, bool GRP>
__device__ __forceinline__ void ws_compute(GemmArgs g, int tiles_m, int items, uint8_t* smem, int wave, int lane) {
  using T = WsTile<BM, BN>;
  constexpr int WTM = BM / T::WM, WTN = BN / T::WN, FM = WTM / 16, FN = WTN / 16;
  // fragments of x in flight (a row of tiles uses one FN times); both halves' weights, or one half's where the sums leave
  // no room for more
  constexpr int R = FM * FN < 32 ? 4 : 3, ROWS = 2 * FM, BAR = ROWS - 3;   // (rows of both half steps; the barrier's)
  constexpr bool BOTH = 4 * (FM * FN + 2 * FN + R) <= 152;
  const int wr = wave / T::WN, wc = wave % T::WN;
  const int swz = (lane & 15) >> 1, lrow = (lane & 15) * 128;
  const int off[2] = {((lane >> 4) ^ swz) * 16, ((4 + (lane >> 4)) ^ swz) * 16};
  const uint8_t* const a_base = smem + wr * WTM * 128 + lrow;
  const uint8_t* const b_base = smem + T::AB * T::ABUF + wc * WTN * 128 + lrow;
  int sa = 0, sb = 0;   // buffers of the step at work
  const auto lda_ = [&](int i, int h) __attribute__((always_inline)) {
    return *reinterpret_cast<const uint4*>(a_base + sa * T::ABUF + i * 2048 + off[h]);
  };
  const auto ldb_ = [&](int j, int h) __attribute__((always_inline)) {
    return *reinterpret_cast<const uint4*>(b_base + sb * T::BBUF + j * 2048 + off[h]);
  };
  uint4 af[R], bf[2][FN];
  asm volatile("s_barrier" ::: "memory");
#pragma unroll 1
  for (int bid = blockIdx.x; bid < items; bid += gridDim.x) {
    const WsItem it = ws_item<GRP, BM, BN>(g, tiles_m, bid, items);
    cf32x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        acc[i][j] = cf32x4{0.f, 0.f, 0.f, 0.f};
        asm volatile("" : "+v"(acc[i][j]));
      }
    asm volatile("s_nop 3" ::: "memory");   // a VALU's write and an MFMA's read
    // (not kept through the epilogue)
#pragma unroll
    for (int j = 0; j < FN; ++j) bf[0][j] = ldb_(j, 0);
#pragma unroll
    for (int i = 0; i < R; ++i) af[i] = lda_(i, 0);
    int prev = 0;
#pragma unroll 1
    for (int s = 0; s < it.nk; ++s) {
      static_for<0, ROWS>([&](auto ri) __attribute__((always_inline)) {
        constexpr int row = decltype(ri)::value, h = row / FM, i = row % FM;
        if constexpr (row == BAR) {   // the step is read, the next one there
          asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
          prev = sb;
          sa = sa + 1 == T::AB ? 0 : sa + 1;
          sb = sb == 2 ? 0 : sb + 1;
          if constexpr (BOTH)
#pragma unroll
            for (int j = 0; j < FN; ++j) bf[0][j] = ldb_(j, 0);
          static_for<0, R>([&](auto qi) __attribute__((always_inline)) {   // registers that are free by now
            constexpr int q = decltype(qi)::value, user = (ROWS - 1 - q) / R * R + q;
            if constexpr (user < BAR) af[q] = lda_(q, 0);
          });
        }
        if constexpr (BOTH && row == 0)
#pragma unroll
          for (int j = 0; j < FN; ++j) bf[1][j] = ldb_(j, 1);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          vmfma<DT>(acc[i][j], af[row % R], bf[BOTH ? h : 0][j]);
          if constexpr (!BOTH && i == FM - 1) bf[0][j] = ldb_(j, 1 - h);
        }
        // the register's next row, of this step or, behind the barrier, of the next
        if constexpr (row + R < ROWS) af[row % R] = lda_((row + R) % FM, (row + R) / FM);
        else if constexpr (row >= BAR) af[row % R] = lda_(row % R, 0);
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    // the last MFMAs' results settle
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(acc[i][j]));
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) asm volatile("" : "+v"(acc[i][j]));
    Pieces add{};
    if (!GRP && it.rest >= 0 && g.pieces > 1) {
      // a wave's share of the tile's sums, with counters of its own (a barrier would wait for the asking waves); else
      // as in gemm_4w.h: parked but for the last to arrive, who waits for waves that are past their arrival
      const int n = g.pieces;
      constexpr uint32_t SLAB = BM * BN * 4;
      unsigned* tk = g.tick + it.rest * T::NC + wave;
      unsigned* fl = tk + kPieceWaves * kPieceTiles;
      unsigned got = 0;
      if (lane == 0) got = __hip_atomic_fetch_add(tk, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const bool lastp = __builtin_amdgcn_readfirstlane(got) == (unsigned)(n - 1);
      add = Pieces{g.ws + (size_t)it.rest * n * (BM * BN), n * SLAB, (uint32_t)(wave * (FM * FN * 1024) + lane * 16),
                   n > 2 ? 0u : (1 - it.piece) * SLAB, SLAB, n, 1024u};
      if (!lastp || n > 2) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) add.store(it.piece * SLAB + (i * FN + j) * 1024u, acc[i][j]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      if (!lastp) {
        if (lane == 0) __hip_atomic_fetch_add(fl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        continue;
      }
      while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(fl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) !=
             (unsigned)(n - 1))
        __builtin_amdgcn_s_sleep(2);
      if (lane == 0) {
        __hip_atomic_store(tk, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(fl, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    float* stg = reinterpret_cast<float*>(smem + T::AB * T::ABUF + (wave < T::FIT ? prev * T::BBUF + wave * T::STG
                                                                                : 3 * T::BBUF + (wave - T::FIT) * T::STG));
    GemmArgs e = g;
    e.c = it.c;
    if constexpr (GRP) e.M = it.rows;
    int row_m0 = it.m0 + wr * WTM, vcol0 = it.n0 + wc * WTN, el = lane;
    asm volatile("" : "+s"(row_m0), "+s"(vcol0), "+v"(el));   // (no address of the strips is kept through the steps)
    static_assert(EpiW<DT, EPI, FN>::OK, "whole chunks of a row");
    EpiW<DT, EPI, FN> ops;
    ops.load_bias(e, vcol0, el);
    ops.template load_res<0>(e, row_m0, vcol0, el);
    static_for<0, FM>([&](auto ii) __attribute__((always_inline)) {
      constexpr int i = decltype(ii)::value;
      if constexpr (i + 1 < FM) ops.template load_res<(i + 1) & 1>(e, row_m0 + (i + 1) * 16, vcol0, el);
      stage_strip_w<FN, T::SLD>(acc[i], stg, el, add.strip(i, FN));
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
      readout_strip_w<DT, EPI, FN, i & 1, T::SLD>(e, stg, row_m0 + i * 16, vcol0, 0, el, ops);
      __builtin_amdgcn_wave_barrier();
    });
  }
}

template <int DT, int EPI, int BM, int BN, bool GRP>
__device__ __forceinline__ void ws_tiles(GemmArgs g, uint8_t* smem) {
  if constexpr (GRP) g.tiles_n = (g.N + BN - 1) / BN;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int tiles_m = GRP ? __builtin_amdgcn_readfirstlane(g.groups[g.tiles_m].x) : g.tiles_m;
  const int tiles = tiles_m * g.tiles_n;
  const int items = !GRP && g.pieces > 0 ? g.dp_tiles + (tiles - g.dp_tiles) * g.pieces : tiles;
  if ((int)blockIdx.x >= items) return;
  constexpr int NC = WsTile<BM, BN>::NC;
  if (wave >= NC) ws_ask<BM, BN, GRP>(g, tiles_m, items, smem, wave - NC, lane);
  else ws_compute<DT, EPI, BM, BN, GRP>(g, tiles_m, items, smem, wave, lane);
}

template <int DT, int EPI, int BM, int BN>
__global__ __launch_bounds__((WsTile<BM, BN>::THREADS)) void gemm_ws_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint8_t smem[WsTile<BM, BN>::LDS];
  ws_tiles<DT, EPI, BM, BN, false>(g, smem);
}

}  // namespace cake
