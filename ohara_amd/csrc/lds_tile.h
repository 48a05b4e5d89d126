// The tiled product of the many-row kernels (gemm_tile.hip, moe.hip): activations x packed weights on MFMA, both operands
// through LDS.
//
// A workgroup owns a tile of TM activation rows x TS packed 16-row weight strips; its WM x WN waves own FM x FN
// fragments of v_mfma_f32_16x16x32_bf16 each (weights = A operand, activations = B operand, as in the skinny kernels, so
// the epilogues are shared).  K is walked in order, KH MFMA steps of 32 at a time.  Both operands of a step travel straight
// from global memory into LDS (global_load_lds, 16 bytes a lane: no registers held in flight, NST - 1 steps ahead) and
// every wave reads its fragments from there:
//   * a packed weight tile (strip, k-step) is 1 KiB in lane order: one load, and a conflict-free 16-byte read;
//   * a load of activations is 1 KiB of whole row segments of 64 KH bytes; the 16-byte pieces of a row are permuted by the
//     row's number on their way in (each lane chooses its global address, the LDS side is always in lane order), which
//     is what makes the fragment reads of sixteen rows conflict-free without padding (SQ_LDS_BANK_CONFLICT 0; with 256-byte
//     segments and the low three bits of the row alone it was two cycles a read, 4 being what one takes).
// One barrier per step: it says that the step's loads have arrived (every wave waits for its own first) and that the slot
// of the step before is free for the next loads.
//
// LA = 0: a k-step's fragments are read, then multiplied; the other waves of the CU fill the gap.  LA = 1, for the tiles with one or
// two products a wave and activation fragment whose step is a chain: the fragments of the next group of products are read before
// the present group's, across the barrier too.  us a call, 0 / 1, from a graph over one set of operands: 32 x 32 tiles, 96 rows
// 768 x 3072 10.1 / 8.8; 64 x 128, 192 rows 11264 x 2048 22.5 / 21.9; but 64 x 64, 192 rows 2048 x 5632 28.2 / 30.2; 128 x 192, 8192 rows
// 768 x 768 and 3072 (a mean) 37.0 / 39.5.
// What K leaves for a last step that is not full has its own code behind the loop: inside, its selects cost every step
// (128 x 128, 4001 rows: 74.3 / 67.7).
#pragma once
#include "common.h"

#include <type_traits>

namespace {

// 16 bytes per lane from sbase + voff to LDS byte lds + 16 * lane.  (Assembly: behind the builtin the compiler waits for
// every such load in flight before any LDS read, which would undo the ring.  No vector register is written; the waits
// are wait_loads below; M0 holds nothing of the compiler's: none of the kernels that use this has another instruction that reads it.)
__device__ __forceinline__ void load_lds16(uint32_t lds, const void* sbase, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(sbase) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_loads() {  // until at most N of this wave's loads are in flight
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int WM_, int WN_, int FM_, int FN_, int KH_, int NST_, int LA_>
struct Tile {
  static constexpr bool HALVES = false;
  static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_, KH = KH_, NST = NST_, LA = LA_;
  static constexpr int NW = WM * WN;                       // waves
  static constexpr int TM = WM * FM * 16, TS = WN * FN;    // rows, strips
  static constexpr int RPL = 16 / KH;                      // activation rows of a 1 KiB load
  static constexpr int XL = TM / RPL, WL = TS * KH;        // 1 KiB loads of a step
  static constexpr int XPW = XL / NW, LPW = (XL + WL) / NW;  // of one wave
  static constexpr int STAGE = (XL + WL) * 1024, LDS = NST * STAGE;
  static_assert(XL % NW == 0 && WL % NW == 0, "loads split evenly over the waves");
  static_assert((KH == 2 || KH == 4) && LDS <= 160 * 1024, "");
};

// A tile whose waves work in two halves (halves_product): PU k-steps of 32 a phase, the activations in a ring of XS slots of 64 columns,
// the weights in one of WS slots of a phase.
template <int WM_, int WN_, int FM_, int FN_, int PU_, int XS_, int WS_>
struct HalvesTile {
  static constexpr bool HALVES = true;
  static constexpr int WM = WM_, WN = WN_, FM = FM_, FN = FN_, KH = 2, PU = PU_, XS = XS_, WS = WS_, LA = 0;
  static constexpr int NW = WM * WN, TM = WM * FM * 16, TS = WN * FN;
  static constexpr int RPL = 8, XL = TM / RPL, WL = TS * PU, XPW = XL / NW, WPW = WL / NW;
  static constexpr int XPP = XPW * PU / 2;                 // activation loads of a wave in a phase
  static constexpr int XSLOT = XL * 1024, WSLOT = WL * 1024, LDS = XS * XSLOT + WS * WSLOT;
  static_assert(XL % NW == 0 && WL % NW == 0 && XPW * PU % 2 == 0 && NW == 8, "loads split evenly over the waves and phases; two waves a SIMD");
  static_assert((PU == 1 && WS == XS + 1) || (PU == 2 && WS == XS), "both rings as far ahead");
  static_assert(LDS <= 160 * 1024, "");
};

// Where a lane finds the activations it loads: a byte offset for each of its wave's loads (the caller gives the element offset
// of the row), and the 16-byte piece of the row that is this lane's.
template <class C, bool ALIGNED>
struct XOffsets {
  typedef typename std::conditional<ALIGNED, uint32_t, uint64_t>::type type;
  type off[C::XPW];
  int piece[C::XPW];
  static __device__ __forceinline__ int row(int i, int wave, int lane) { return (wave + i * C::NW) * C::RPL + lane / (4 * C::KH); }
  __device__ __forceinline__ void set(int i, int wave, int lane, type row_elements) {
    piece[i] = (lane ^ row(i, wave, lane)) & (4 * C::KH - 1);
    off[i] = (row_elements + piece[i] * 8) * 2;
  }
};

// acc[u][t]: strip u x row block t of this wave.  ALIGNED: activation rows start on 16 bytes (false: through registers, any).
// K is a multiple of 8; what the last step reads past it are the row's last piece, which the packed weights' zeros meet as a zero, and the
// strip's last tile, which nothing multiplies (times zero an infinite weight would be a NaN).
__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The product by two halves of the waves, four each, one wave a SIMD: while one half reads its fragments of a phase from LDS and asks for
// loads, the other multiplies; a barrier, and they change places.  So a SIMD's matrix pipe has products from one of its two waves and the
// reads of the other travel under them (before, all eight read first and then all multiplied).  K a phase: 32 where that is 32 products a
// wave, 64 where it would be 12 or 16 (a phase costs a barrier).  Without its loads the walk takes 478 of 728 us (8192^3, zeros), without its
// reads 758: what a CU takes in is the bound.  So the activations go by 64 columns, whole 128-byte lines (loads alone: 59 GB/s a CU in
// 64-byte pieces, 90 in lines; the walk 728 / 571), the weights by phases, both as far ahead as LDS allows.
// Which slot is free: a phase's loads go into the slots of the phase (activations: the step) before, which the other half has read in the
// phase between.  What has landed: a wave waits for its own loads of the next phase before the barrier in front of it.
// Bits: those of tile_product.  K >= 64.
template <class C>
__device__ __forceinline__ void halves_product(f32x4 (&acc)[C::FN][C::FM], const char* xb, const XOffsets<C, true>& x, const uint4* wp, int strip0,
                                               int nstrips, int K, int wave, int lane, unsigned char* smem, int strip_steps) {
  constexpr int FM = C::FM, FN = C::FN, NW = C::NW, PU = C::PU, PH = 2 / PU, XS = C::XS, WS = C::WS, WPW = C::WPW, XPP = C::XPP;
  const int wm = wave / C::WN, wn = wave % C::WN, m = lane & 15, g = lane >> 4;
  const int KS = (K + 31) >> 5, SS = strip_steps ? strip_steps : KS;
  const int nfull = K >> 6, tail = K & 63;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem, ldsw = lds0 + XS * C::XSLOT;
  const uint32_t lane16 = lane * 16;
  const char* wb[WPW];
#pragma unroll
  for (int i = 0; i < WPW; ++i)
    wb[i] = reinterpret_cast<const char*>(wp) + (size_t)min(strip0 + (wave + i * NW) / PU, nstrips - 1) * SS * 1024;
  // Past the last step the last full one is loaded again, unused: the loads in flight stay the same number.
  auto load_x = [&](int s, uint32_t slot, int i) {
    const uint32_t dst = lds0 + slot + (wave + i * NW) * 1024;
    if (tail && s == nfull) load_lds16(dst, xb + (size_t)s * 128, x.off[i] - (uint32_t)max(0, s * 64 + x.piece[i] * 8 - (K - 8)) * 2);
    else load_lds16(dst, xb + (size_t)min(s, nfull - 1) * 128, x.off[i]);
  };
  auto load_w = [&](int p, uint32_t slot, int i) {
    const int t = wave + i * NW;
    load_lds16(ldsw + slot + t * 1024, wb[i] + (size_t)min(p * PU + t % PU, KS - 1) * 1024, lane16);
  };
#pragma unroll
  for (int u = 0; u < FN; ++u)
#pragma unroll
    for (int t = 0; t < FM; ++t) acc[u][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const uint32_t xrd = lds0 + (wm * FM * 16 + m) * 128, wrd = ldsw + wn * FN * PU * 1024 + lane16;
  auto x_frag = [&](uint32_t slot, int jj, int t) { return lds16_at(xrd + slot + t * 2048 + (uint32_t)((4 * jj + g) ^ (m & 7)) * 16); };
  auto w_frag = [&](uint32_t slot, int j, int u) { return lds16_at(wrd + slot + (u * PU + j) * 1024); };
  // As many phases' loads ahead as the rings hold, in the order of the phases.
#pragma unroll
  for (int i = 0; i < C::XPW; ++i) load_x(0, 0, i);
#pragma unroll
  for (int p = 0; p < WS - 1; ++p) {
    if (p > 0) {
#pragma unroll
      for (int i = 0; i < XPP; ++i) {
        const int l = (p - 1) * XPP + i;  // of the activations' loads behind the first step's
        load_x(1 + l / C::XPW, (1 + l / C::XPW) * C::XSLOT, l % C::XPW);
      }
    }
#pragma unroll
    for (int i = 0; i < WPW; ++i) load_w(p, p * C::WSLOT, i);
  }
  wait_loads<(WS - 2) * (WPW + XPP)>();
  __builtin_amdgcn_s_barrier();
  const bool late = wave >= NW / 2;
  if (late) __builtin_amdgcn_s_barrier();
  uint32_t xo = 0, xi = (XS - 1) * C::XSLOT, wo = 0, wi = (WS - 1) * C::WSLOT;
  auto step = [&](int s, auto whole) {  // whole: it asks for whole steps (past the last one, for that)
#pragma unroll
    for (int h = 0; h < PH; ++h) {
      uint4 xf[PU][FM], wf[PU][FN];
#pragma unroll
      for (int j = 0; j < PU; ++j) {
#pragma unroll
        for (int u = 0; u < FN; ++u) wf[j][u] = w_frag(wo, j, u);
#pragma unroll
        for (int t = 0; t < FM; ++t) xf[j][t] = x_frag(xo, h * PU + j, t);
      }
      // Into the slots of the phase (the step) before: the other half has read them, a barrier ago.
      const int p = s * PH + h + WS - 1;
#pragma unroll
      for (int i = 0; i < XPP; ++i) {
        if (decltype(whole)::value) load_lds16(lds0 + xi + (wave + (h * XPP + i) * NW) * 1024, xb + (size_t)min(s + XS - 1, nfull - 1) * 128, x.off[h * XPP + i]);
        else load_x(s + XS - 1, xi, h * XPP + i);
      }
#pragma unroll
      for (int i = 0; i < WPW; ++i) {
        const int t = wave + i * NW;
        if (decltype(whole)::value) load_lds16(ldsw + wi + t * 1024, wb[i] + (size_t)(min(p, nfull * PH - 1) * PU + t % PU) * 1024, lane16);
        else load_w(p, wi, i);
      }
      wait_loads<(WS - 2) * (WPW + XPP)>();  // the next phase's have landed
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < PU; ++j)
#pragma unroll
        for (int t = 0; t < FM; ++t)
#pragma unroll
          for (int u = 0; u < FN; ++u) acc[u][t] = mfma16(wf[j][u], xf[j][t], acc[u][t]);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      wo = wo + C::WSLOT == WS * C::WSLOT ? 0 : wo + C::WSLOT;
      wi = wi + C::WSLOT == WS * C::WSLOT ? 0 : wi + C::WSLOT;
    }
    xo = xo + C::XSLOT == XS * C::XSLOT ? 0 : xo + C::XSLOT;
    xi = xi + C::XSLOT == XS * C::XSLOT ? 0 : xi + C::XSLOT;
  };
  int s = 0;
  for (const int n = tail ? nfull - XS + 1 : nfull; s < n; ++s) step(s, std::true_type());
  for (; s < nfull; ++s) step(s, std::false_type());
  if (!late) __builtin_amdgcn_s_barrier();
  wait_loads<0>();
  if (tail) {
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      if (64 * nfull + 32 * jj >= K) break;  // (uniform) as behind tile_product's loop
      const bool in = 64 * nfull + 32 * jj + 8 * g < K;
      const uint32_t slot = PU == 2 || !jj ? wo : wo + C::WSLOT == WS * C::WSLOT ? 0 : wo + C::WSLOT;
      uint4 wt[FN];
#pragma unroll
      for (int u = 0; u < FN; ++u) wt[u] = w_frag(slot, PU == 2 ? jj : 0, u);
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const uint4 xt = in ? x_frag(xo, jj, t) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < FN; ++u) acc[u][t] = mfma16(wt[u], xt, acc[u][t]);
      }
    }
  }
}

// The same walk over tile after tile, for depths of whole steps: the loads run ahead of the products by the same number of phases throughout, out
// of a tile into the one that follows, so that between two tiles there are only the barriers that bring the halves together.
template <class C>
struct HalvesStream {
  static constexpr int FM = C::FM, FN = C::FN, NW = C::NW, PU = C::PU, PH = 2 / PU, XS = C::XS, WS = C::WS, WPW = C::WPW, XPP = C::XPP;
  const char* xb;            // where the loads are: the tile's rows, this lane's offsets from there, strips
  uint32_t xoff[C::XPW];
  const char* wb[WPW];
  const uint4* wp;
  int nsteps, nstrips, wave;
  uint32_t lds0, ldsw, lane16, xrd, wrd, xkey;
  uint32_t xo, xi, wo, wi;   // slots: read from, asked for

  __device__ __forceinline__ HalvesStream(const uint4* wp_, int K, int nstrips_, int wave_, int lane, unsigned char* smem)
      : wp(wp_), nsteps(K >> 6), nstrips(nstrips_), wave(wave_) {
    const int m = lane & 15, g = lane >> 4;
    lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;
    ldsw = lds0 + XS * C::XSLOT;
    lane16 = lane * 16;
    xrd = lds0 + (wave / C::WN * FM * 16 + m) * 128;
    wrd = ldsw + wave % C::WN * FN * PU * 1024 + lane16;
    xkey = g ^ (m & 7);
    xo = wo = 0;
    xi = (XS - 1) * C::XSLOT;
    wi = (WS - 1) * C::WSLOT;
  }
  __device__ __forceinline__ void strips(int strip0) {
#pragma unroll
    for (int i = 0; i < WPW; ++i)
      wb[i] = reinterpret_cast<const char*>(wp) + (size_t)min(strip0 + (wave + i * NW) / PU, nstrips - 1) * nsteps * 2048;
  }
  __device__ __forceinline__ void load_x(int s, uint32_t slot, int i) const { load_lds16(lds0 + slot + (wave + i * NW) * 1024, xb + (size_t)s * 128, xoff[i]); }
  __device__ __forceinline__ void load_w(int p, uint32_t slot, int i) const {
    const int t = wave + i * NW;
    load_lds16(ldsw + slot + t * 1024, wb[i] + (size_t)(p * PU + t % PU) * 1024, lane16);
  }
  // The first tile's first phases, as many as the rings hold (its rows are set).
  __device__ __forceinline__ void begin(int strip0) {
    strips(strip0);
#pragma unroll
    for (int i = 0; i < C::XPW; ++i) load_x(0, 0, i);
#pragma unroll
    for (int p = 0; p < WS - 1; ++p) {
      if (p > 0) {
#pragma unroll
        for (int i = 0; i < XPP; ++i) {
          const int l = (p - 1) * XPP + i;
          load_x(1 + l / C::XPW, (1 + l / C::XPW) * C::XSLOT, l % C::XPW);
        }
      }
#pragma unroll
      for (int i = 0; i < WPW; ++i) load_w(p, p * C::WSLOT, i);
    }
    wait_loads<(WS - 2) * (WPW + XPP)>();
    __builtin_amdgcn_s_barrier();
  }
  // E < 0: a step whose loads are this tile's; else the E-th of the last XS - 1, whose activations (and, from phase 0 on, weights) are the next tile's.
  // FIRST: a tile's first step, which nothing is added to; where `stored`, at least STORES stores of this wave lie between its loads and those before,
  // so many more may be on their way (they finish in order).
  template <int E, bool FIRST, int STORES>
  __device__ __forceinline__ void step(f32x4 (&acc)[FN][FM], int s, int next_strip0, bool stored) {
#pragma unroll
    for (int h = 0; h < PH; ++h) {
      uint4 xf[PU][FM], wf[PU][FN];
#pragma unroll
      for (int j = 0; j < PU; ++j) {
#pragma unroll
        for (int u = 0; u < FN; ++u) wf[j][u] = lds16_at(wrd + wo + (u * PU + j) * 1024);
#pragma unroll
        for (int t = 0; t < FM; ++t) xf[j][t] = lds16_at(xrd + xo + t * 2048 + (xkey ^ (4 * (h * PU + j))) * 16);
      }
      // Into the slots of the phase (the step) before: the other half has read them, a barrier ago.
#pragma unroll
      for (int i = 0; i < XPP; ++i) load_x(E < 0 ? s + XS - 1 : E, xi, h * XPP + i);
      const int over = (E - (XS - 1)) * PH + h + WS - 1;  // phases past this tile's last one
      if (E >= 0 && over == 0) strips(next_strip0);
#pragma unroll
      for (int i = 0; i < WPW; ++i) load_w(E < 0 || over < 0 ? s * PH + h + WS - 1 : over, wi, i);
      // the next phase's have landed (WS - 2 phases, the first step, wait for loads in front of the stores)
      static_assert(!FIRST || PH == WS - 2, "");
      if (FIRST && STORES && stored) wait_loads<(WS - 2) * (WPW + XPP) + STORES>();
      else wait_loads<(WS - 2) * (WPW + XPP)>();
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < PU; ++j)
#pragma unroll
        for (int t = 0; t < FM; ++t)
#pragma unroll
          for (int u = 0; u < FN; ++u) acc[u][t] = mfma16(wf[j][u], xf[j][t], FIRST && h == 0 && j == 0 ? (f32x4){0.f, 0.f, 0.f, 0.f} : acc[u][t]);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      wo = wo + C::WSLOT == WS * C::WSLOT ? 0 : wo + C::WSLOT;
      wi = wi + C::WSLOT == WS * C::WSLOT ? 0 : wi + C::WSLOT;
    }
    xo = xo + C::XSLOT == XS * C::XSLOT ? 0 : xo + C::XSLOT;
    xi = xi + C::XSLOT == XS * C::XSLOT ? 0 : xi + C::XSLOT;
  }
  // One tile; rows_of_next() sets the next one's rows.  Its first phase has landed on entry, and the next one's on return.
  template <int STORES, class F>
  __device__ __forceinline__ void walk(f32x4 (&acc)[FN][FM], int next_strip0, bool stored, F rows_of_next) {
    static_assert(XS == 3, "two steps at a tile's end");
    const bool late = wave >= NW / 2;
    if (late) __builtin_amdgcn_s_barrier();
    step<-1, true, STORES>(acc, 0, 0, stored);
    for (int s = 1; s < nsteps - 2; ++s) step<-1, false, 0>(acc, s, 0, false);
    rows_of_next();
    step<0, false, 0>(acc, nsteps - 2, next_strip0, false);
    step<1, false, 0>(acc, nsteps - 1, next_strip0, false);
    if (!late) __builtin_amdgcn_s_barrier();
  }
};

template <class C, bool ALIGNED>
__device__ __forceinline__ void tile_product(f32x4 (&acc)[C::FN][C::FM], const char* xb, const XOffsets<C, ALIGNED>& x, const uint4* wp,
                                             int strip0, int nstrips, int K, int wave, int lane, unsigned char* smem, int strip_steps = 0) {
  if constexpr (C::HALVES) {
    static_assert(ALIGNED, "");
    halves_product<C>(acc, xb, x, wp, strip0, nstrips, K, wave, lane, smem, strip_steps);
  } else {
  constexpr int FM = C::FM, FN = C::FN, KH = C::KH, NST = C::NST, NW = C::NW, XL = C::XL, WL = C::WL, LPW = C::LPW;
  constexpr int STAGE = C::STAGE, KB = 32 * KH;
  const int wm = wave / C::WN, wn = wave % C::WN;
  const int m = lane & 15, g = lane >> 4;
  const int KS = (K + 31) >> 5, nsteps = (KS + KH - 1) / KH;
  const bool tail = K % KB != 0;                           // the last step is not full
  const int SS = strip_steps ? strip_steps : KS;           // k-steps from strip to strip (more than KS: a part of the depth)
  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;
  const char* wb = reinterpret_cast<const char*>(wp);
  const uint32_t lane16 = lane * 16;
  auto issue = [&](int s, uint32_t slot) {
    const char* xs = xb + (size_t)s * (2 * KB);
    const bool last = tail && s == nsteps - 1;
#pragma unroll
    for (int i = 0; i < C::XPW; ++i) {
      const uint32_t dst = slot + (wave + i * NW) * 1024;
      const uint32_t back = last ? (uint32_t)max(0, s * KB + x.piece[i] * 8 - (K - 8)) * 2 : 0u;
      if (ALIGNED) {
        load_lds16(dst, xs, x.off[i] - back);
      } else {
        const uint4 v = ldg16(xs + x.off[i] - back);
        *(OHARA_LDS u32x4*)(uintptr_t)(dst + lane16) = (u32x4){v.x, v.y, v.z, v.w};
      }
    }
#pragma unroll
    for (int i = 0; i < WL / NW; ++i) {
      const int t = wave + i * NW;  // strip t / KH, k-step t % KH; past the end: the last one, never used
      const int strip = min(strip0 + t / KH, nstrips - 1), j = min(KH * s + t % KH, KS - 1);
      load_lds16(slot + (XL + t) * 1024, wb + ((size_t)strip * SS + j) * 1024, lane16);
    }
  };
#pragma unroll
  for (int u = 0; u < FN; ++u)
#pragma unroll
    for (int t = 0; t < FM; ++t) acc[u][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const uint32_t xrd = lds0 + (wm * FM * 16 + m) * (64 * KH);
  const uint32_t wrd = lds0 + (XL + wn * FN * KH) * 1024 + lane16;
  auto x_frag = [&](uint32_t slot, int jj, int t) {
    return lds16_at(xrd + slot + t * (1024 * KH) + (uint32_t)((4 * jj + g) ^ (m & (4 * KH - 1))) * 16);
  };
  auto w_frag = [&](uint32_t slot, int jj, int u) { return lds16_at(wrd + slot + (u * KH + jj) * 1024); };
  auto arrive = [&](bool all, auto left) {  // the loads of the next step have landed, everyone's
    if (!ALIGNED) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else if (all) wait_loads<0>();
    else wait_loads<decltype(left)::value>();
    __builtin_amdgcn_s_barrier();
  };
  constexpr int LA = C::LA, G = KH * FM;
  constexpr int AHEAD = LA ? NST : NST - 1;  // steps whose loads are in flight
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (s < nsteps) issue(s, lds0 + s * STAGE);
  uint32_t so = 0;
  const int nfull = nsteps - (tail ? 1 : 0);
  if constexpr (LA == 0) {
    uint32_t si = (NST - 1) * STAGE;
    for (int s = 0; s < nsteps; ++s) {
      arrive(NST == 2 || s + NST - 2 >= nsteps, std::integral_constant<int, (NST - 2) * LPW>());
      if (s + NST - 1 < nsteps) issue(s + NST - 1, lds0 + si);
      if (s == nfull) break;
#pragma unroll
      for (int jj = 0; jj < KH; ++jj) {
        uint4 xf[FM], wf[FN];
#pragma unroll
        for (int u = 0; u < FN; ++u) wf[u] = w_frag(so, jj, u);
#pragma unroll
        for (int t = 0; t < FM; ++t) xf[t] = x_frag(so, jj, t);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < FM; ++t)
#pragma unroll
          for (int u = 0; u < FN; ++u) acc[u][t] = mfma16(wf[u], xf[t], acc[u][t]);
        __builtin_amdgcn_sched_barrier(0);
      }
      so = so + STAGE == NST * STAGE ? 0 : so + STAGE;
      si = si + STAGE == NST * STAGE ? 0 : si + STAGE;
    }
  } else {
    // A group is the products of one activation fragment.  Its fragments are read LA groups before, across the steps: the barrier
    // stands LA groups before the end of a step, behind the last read of its slot.
    constexpr int R = LA + 1, W = 2;
    static_assert(G % R == 0 && KH % W == 0 && LA <= FM, "fragments stay where the unrolled groups expect them");
    uint4 xf[R], wf[W][FN];
    auto fetch = [&](uint32_t slot, int i) {
      if (i % FM == 0) {
#pragma unroll
        for (int u = 0; u < FN; ++u) wf[i / FM % W][u] = w_frag(slot, i / FM, u);
      }
      xf[i % R] = x_frag(slot, i / FM, i % FM);
    };
    arrive(NST > nsteps, std::integral_constant<int, (NST - 1) * LPW>());
#pragma unroll
    for (int i = 0; i < LA; ++i) fetch(0, i);
    for (int s = 0; s < nfull; ++s) {
      const uint32_t next = so + STAGE == NST * STAGE ? 0 : so + STAGE;
#pragma unroll
      for (int i = 0; i < G; ++i) {
        if (i == G - LA) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          arrive(s + NST > nsteps, std::integral_constant<int, (NST - 2) * LPW>());
          if (s + NST < nsteps) issue(s + NST, lds0 + so);
        }
        if (i + LA < G) fetch(so, i + LA);
        else fetch(next, i + LA - G);  // (behind the last step: what the slot holds, unused)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < FN; ++u) acc[u][i % FM] = mfma16(wf[i / FM % W][u], xf[i % R], acc[u][i % FM]);
        __builtin_amdgcn_sched_barrier(0);
      }
      so = next;
    }
  }
  if (tail) {
#pragma unroll
    for (int jj = 0; jj < KH; ++jj) {
      if (KB * nfull + 32 * jj >= K) break;  // (uniform) k-steps past the end: what stands in for them is not multiplied, not even by zero
      const bool in = KB * nfull + 32 * jj + 8 * g < K;
      uint4 wt[FN];
#pragma unroll
      for (int u = 0; u < FN; ++u) wt[u] = w_frag(so, jj, u);
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const uint4 xt = in ? x_frag(so, jj, t) : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < FN; ++u) acc[u][t] = mfma16(wt[u], xt, acc[u][t]);
      }
    }
  }
  }
}

}  // namespace
