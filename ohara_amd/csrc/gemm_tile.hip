// Tiled MFMA GEMM for the batched (prefill) projections: y = epi(x W^T) with many rows.
//
// The walk over K is tile_product (lds_tile.h); the sums do not depend on the tile, but on the parts of the depth they are made of.
//
// What bounds it: in the large tiles, whose waves work in two halves (lds_tile.h), the chip's clock under the products (8192 x 8192 x 8192 on
// zeros 571 us, on random data 715 = 1.54 PFLOP/s; with all waves reading, then all multiplying, and 64 KB in flight 745 and 863), at K of 768
// a tile's start and epilogue (9 of 25 us a round); in small ones the chain barrier - read - multiply of a step (0.14 to 0.36 us).  us a call, that
// walk over K / halves, sets of random operands in turn: 256 x 256: 8192 rows 6144 x 768 with SwiGLU 82 / 75, 4001 rows 11264 x 2048 with
// SwiGLU 179 / 149, 11200 rows 459 / 387, 704 rows 17920 x 2560 77 / 59;  the best of the tiles before / of all: 8192 rows 768 x 3072 with a
// residual 46 / 38, 768 x 768 17.5 / 15.9, 4001 rows 2048 x 5632 90 / 77, 2048 x 2048 38 / 35.
// Measured and dropped there: loads among the products (4001 rows 151 / 165), s_setprio around them (even), four waves of 128 x 128 each (160 /
// 209), 64-byte pieces of activations five steps ahead (151 / 154), halves on 128 x 128 (90 / 94) and on 192-row tiles.  In the small tiles:
// loads spread among the products, deeper rings (no gain, fewer workgroups a CU), four waves a tile of 128 x 192 (99 / 52 us against 93 / 45).
//
// Workgroup ids go round-robin over the eight XCDs: an XCD gets a contiguous run of tiles, eight activation tiles side
// by side, so that a run shares its operands in that XCD's L2.
//
// Replaces the F.linear calls of ohara/models/llama.py:84-86,142,322 and
// ohara/modules/mlp.py:152 when the call carries more than 64 rows.
#include "gemm_epilogue.h"
#include "lds_tile.h"

#include <algorithm>

namespace {

constexpr int CUS = 256;

// Tile `pid` of a run: eight activation tiles side by side.
struct TilePlace {
  int row0, strip0;
};
template <class C>
__device__ __forceinline__ TilePlace tile_place(int pid, int MT, int NT) {
  constexpr int GM = 8;
  const int grp = pid / (GM * NT), first = grp * GM, gsz = min(GM, MT - first), r = pid - grp * GM * NT;
  return {(first + r % gsz) * C::TM, (r / gsz) * C::TS};
}

// What a wave does with its sums: rows rbase + 16 t + (lane & 15), strips sbase + u.  (The arguments by value: what is used of them is loaded in one place, where
// by reference every use waits for its own: 128 rows 2304 x 768 with rotary 0.2 us.)
template <int EPI, class C>
__device__ __forceinline__ void tile_epilogue(GemmArgs a, const f32x4 (&acc)[C::FN][C::FM], int rbase, int sbase, int nstrips, int lane) {
  constexpr int FM = C::FM, FN = C::FN;
  const int m = lane & 15, g = lane >> 4;
  // A thread finishes FM * FN fragments.  What their epilogues read (residual rows, biases, rotary
  // values) is fetched for a strip's before the first is used, instead of one dependent round trip
  // per fragment.
  // Rotary epilogue: position, sequence and cache row depend on the activation row alone (FM per
  // thread, and rows of a tile are consecutive: no division per row when a sequence is at least a tile
  // long), the region (q / k / v) and the feature index inside the head on the strip alone (uniform
  // over the wave).  Worked out per fragment they were 40 % of this kernel's instructions.
  if (rbase >= a.B) return;
  if (EPI == EPI_ROPE && (a.rows || a.S >= FM * 16) && ((a.ldo | a.Dh) & 15) == 0 && ((a.H * a.Dh) & 15) == 0 && !a.stage) {
    const int nq = a.H * a.Dh, nk = a.Hkv * a.Dh;
    const int gbase = a.row0 + rbase;                          // global row of the wave's first row
    const int seq0 = a.rows ? 0 : gbase / a.S, rem0 = gbase - seq0 * a.S;   // uniform over the wave
    int pos_t[FM];
    size_t qoff_t[FM], coff_t[FM];
#pragma unroll
    for (int t = 0; t < FM; ++t) {
      const int x = rem0 + min(t * 16 + m, a.B - 1 - rbase);  // rows past the end: the last row, never stored
      const int grow = gbase + t * 16 + m;
      int seq;
      if (a.rows) {
        pos_t[t] = a.rows[x];
        seq = a.rows[a.nrows + x];
      } else {
        const bool wrap = x >= a.S;
        seq = seq0 + (wrap ? 1 : 0);
        pos_t[t] = (a.pos_dev ? a.pos_dev[(size_t)seq * a.pos_stride] : a.pos) + x - (wrap ? a.S : 0);
      }
      qoff_t[t] = (size_t)grow * a.ldo;
      coff_t[t] = (((size_t)seq * a.Tmax + pos_t[t]) * a.Hkv) * a.Dh;
    }
    const bool wide = ((a.ldo | (a.Hkv * a.Dh)) & 7) == 0 && (((uintptr_t)a.out | (uintptr_t)a.kcache | (uintptr_t)a.vcache) & 15) == 0;
    auto column = [&](int r) { return r - (r < nq ? 0 : r < nq + nk ? nq : nq + nk); };  // inside q, k or v
    auto region_of = [&](int r) { return r < nq ? 0 : r < nq + nk ? 1 : 2; };
    auto table_row = [&](int t) { return (size_t)min(max(pos_t[t], 0), a.Tmax - 1) * (a.Dh >> 1); };
    auto turned = [&](f32x4 y, uint32_t cv, uint32_t sv) {
      float v[4] = {rbf(y[0]), rbf(y[1]), rbf(y[2]), rbf(y[3])};
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) {
        const float c = pr ? hi_bf(cv) : lo_bf(cv), sn = pr ? hi_bf(sv) : lo_bf(sv);
        const float e = v[2 * pr], od = v[2 * pr + 1];
        // separate fp32 multiplies and add/sub, as the reference's eager ops round
        v[2 * pr] = __fsub_rn(__fmul_rn(e, c), __fmul_rn(od, sn));
        v[2 * pr + 1] = __fadd_rn(__fmul_rn(e, sn), __fmul_rn(od, c));
      }
      return make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    };
    // 16 bytes a lane of the left and the right strip of a pair: lanes of even g the left one's, of odd g the right one's
    auto paired = [&](uint2 l, uint2 r) {
      const u32x2 x = __builtin_amdgcn_permlane16_swap(l.x, r.x, false, false), y = __builtin_amdgcn_permlane16_swap(l.y, r.y, false, false);
      return make_uint4(x[0], y[0], x[1], y[1]);
    };
    if constexpr (FN == 2 || FN == 4) {
      // A wave's strips in one head, as heads of whole 16 FN features have them: a row's table values are 16 FN bytes, a quarter a lane in one
      // load and exchanged, all rows' in one round trip.  (A load of 4 bytes for every strip and row, a round trip a strip: 8192 rows
      // 2304 x 768, 256 x 256 70.3 us against 49.2 for the plain store, now 50.7 / 44.7; 128 x 256 50.5 / 46.7, now 42.7 / 42.0.)
      if (wide && a.Dh % (16 * FN) == 0 && nstrips - sbase >= FN && sbase * 16 < nq + 2 * nk && (((uintptr_t)a.cos | (uintptr_t)a.sin) & 15) == 0) {
        const int rr = sbase * 16, region = region_of(rr), col = column(rr);  // uniform
        size_t at[FM];
#pragma unroll
        for (int t = 0; t < FM; ++t) at[t] = region == 0 ? qoff_t[t] : coff_t[t];
        constexpr int NB = FM < 4 ? FM : 4;  // rows ahead: all of them are 64 registers more than there are in a tile of 256 x 256
        uint32_t cv[NB][FN], sv[NB][FN];
        const int d = col % a.Dh / 2 + 2 * FN * g;
        auto fetch = [&](int t) {
          auto quarter = [](const bf16_t* p, uint32_t (&v)[FN]) {
            if constexpr (FN == 4) {
              const uint4 q = ldg16(p);
              v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
            } else {
              const uint2 q = ldg8(p);
              v[0] = q.x, v[1] = q.y;
            }
          };
          quarter(a.cos + table_row(t) + d, cv[t % NB]);
          quarter(a.sin + table_row(t) + d, sv[t % NB]);
        };
        if (region < 2) {
#pragma unroll
          for (int t = 0; t < NB; ++t) fetch(t);
          __builtin_amdgcn_sched_barrier(0);
        }
        bf16_t* base = (region == 0 ? a.out : region == 1 ? a.kcache : a.vcache) + col + 16 * (g & 1) + 8 * (g >> 1);
        auto by_strip = [](uint32_t (&v)[FN]) {  // lane group g: from its quarter of the row to its own values of every strip
          if constexpr (FN == 4) {
            const u32x2 p = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false), q = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
            const u32x2 c = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false), d = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
            v[0] = c[0], v[1] = c[1], v[2] = d[0], v[3] = d[1];
          } else {
            const u32x2 p = __builtin_amdgcn_permlane16_swap(v[0], v[1], false, false), c = __builtin_amdgcn_permlane32_swap(p[0], p[1], false, false);
            v[0] = c[0], v[1] = c[1];
          }
        };
#pragma unroll
        for (int t = 0; t < FM; ++t) {
          uint2 w[FN];
          if (region < 2) {
            by_strip(cv[t % NB]);
            by_strip(sv[t % NB]);
#pragma unroll
            for (int u = 0; u < FN; ++u) w[u] = turned(acc[u][t], cv[t % NB][u], sv[t % NB][u]);
            __builtin_amdgcn_sched_barrier(0);
            if (t + NB < FM) fetch(t + NB);
          } else {
#pragma unroll
            for (int u = 0; u < FN; ++u) w[u] = make_uint2(pack_bf(acc[u][t][0], acc[u][t][1]), pack_bf(acc[u][t][2], acc[u][t][3]));
          }
          const bool in = rbase + t * 16 + m < a.B && pos_t[t] >= 0 && pos_t[t] < a.Tmax;
          bf16_t* o = base + at[t];
#pragma unroll
          for (int u = 0; u < FN; u += 2) {
            const uint4 both = paired(w[u], w[u + 1]);
            if (in) *reinterpret_cast<uint4*>(o + 16 * u) = both;
          }
        }
        return;
      }
    }
    uint2 left[FM];  // the strip before, where this one completes 16 bytes a lane with it
#pragma unroll
    for (int u = 0; u < FN; ++u) {
      const int strip = sbase + u;
      const int rr = strip * 16;  // uniform: the whole strip lies in one region and one head
      if (strip >= nstrips || rr >= nq + 2 * nk) continue;
      const bool first = wide && !(u & 1) && u + 1 < FN && strip + 1 < nstrips && rr + 16 < nq + 2 * nk, second = wide && (u & 1);
      const int region = region_of(rr);
      uint32_t cv[FM], sv[FM];
      if (region < 2) {
        const int d = column(rr) % a.Dh + 4 * g;
#pragma unroll
        for (int t = 0; t < FM; ++t) {
          cv[t] = ldg4(a.cos + table_row(t) + (d >> 1));
          sv[t] = ldg4(a.sin + table_row(t) + (d >> 1));
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      // where this lane stores: its four columns of the strip, or eight of this strip or the one before
      const int mine = second ? rr - (g & 1 ? 0 : 16) : rr;
      const int reg = region_of(mine), col = column(mine) + (second ? 8 * (g >> 1) : 4 * g);
      bf16_t* base = reg == 0 ? a.out : reg == 1 ? a.kcache : a.vcache;
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const int b = rbase + t * 16 + m;
        const f32x4 y = acc[u][t];
        const uint2 w = region < 2 ? turned(y, cv[t], sv[t]) : make_uint2(pack_bf(y[0], y[1]), pack_bf(y[2], y[3]));
        if (first) {
          left[t] = w;
          continue;
        }
        const bool in = b < a.B && pos_t[t] >= 0 && pos_t[t] < a.Tmax;
        bf16_t* o = base + (reg == 0 ? qoff_t[t] : coff_t[t]) + col;
        if (second) {
          const uint4 both = paired(left[t], w);
          if (in) *reinterpret_cast<uint4*>(o) = both;
        } else if (in) {
          *reinterpret_cast<uint2*>(o) = w;
        }
      }
    }
    return;
  }
  // Two strips' (four strips') columns lie side by side in a row of the output; exchanged among the lanes of a row they are stored,
  // and a residual read, 16 bytes a lane.
  const bool wide = ((a.N | a.ldo) & 7) == 0 && ((uintptr_t)a.out & 15) == 0;
  if (EPI == EPI_SWIGLU && FN > 1 && wide) {
#pragma unroll
    for (int t = 0; t < FM; ++t) {
      const int b = rbase + t * 16 + m;
      float low = acc[0][t][0];
#pragma unroll
      for (int u = 0; u < FN; ++u) low = fminf(low, fminf(acc[u][t][0], acc[u][t][1]));
      uint32_t w[FN];  // two columns of strip u
      if (__any(low < -86.5f)) {  // (-87 after rounding)
#pragma unroll
        for (int u = 0; u < FN; ++u)
          w[u] = pack_bf(rbf(silu_f(rbf(acc[u][t][0]))) * rbf(acc[u][t][2]), rbf(silu_f(rbf(acc[u][t][1]))) * rbf(acc[u][t][3]));
      } else {
#pragma unroll
        for (int u = 0; u < FN; ++u)
          w[u] = pack_bf(rbf(silu_from_m87(rbf(acc[u][t][0]))) * rbf(acc[u][t][2]),
                         rbf(silu_from_m87(rbf(acc[u][t][1]))) * rbf(acc[u][t][3]));
      }
      bf16_t* o = a.out + (size_t)b * a.ldo + sbase * 8;
      const int left = b < a.B ? a.N - sbase * 8 : 0;  // columns this row still has
      int u = 0;
      if constexpr (FN >= 4) {
        const u32x2 p = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false), q = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        const u32x2 c = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false), d = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
        if (8 * g < left) *reinterpret_cast<uint4*>(o + 8 * g) = make_uint4(c[0], c[1], d[0], d[1]);
        u = 4;
      } else {
        const u32x2 c = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false);
        const int at = 8 * (g & 1) + 4 * (g >> 1);
        if (at < left) *reinterpret_cast<uint2*>(o + at) = make_uint2(c[0], c[1]);
        u = 2;
      }
#pragma unroll
      for (; u < FN; ++u)
        if (8 * u + 2 * g < left) *reinterpret_cast<uint32_t*>(o + 8 * u + 2 * g) = w[u];
    }
    return;
  }
  if ((EPI == EPI_STORE || EPI == EPI_RESIDUAL) && FN > 1 && wide &&
      (EPI == EPI_STORE || ((a.ldr & 7) == 0 && ((uintptr_t)a.resid & 15) == 0))) {
#pragma unroll
    for (int u = 0; u + 1 < FN; u += 2) {
      const int col = (sbase + u + (g & 1)) * 16 + 8 * (g >> 1);
      uint4 res[FM];
      if (EPI == EPI_RESIDUAL) {
#pragma unroll
        for (int t = 0; t < FM; ++t)
          res[t] = *reinterpret_cast<const uint4*>(a.resid + (size_t)min(rbase + t * 16 + m, a.B - 1) * a.ldr + min(col, a.N - 8));
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const int b = rbase + t * 16 + m;
        const u32x2 c = __builtin_amdgcn_permlane16_swap(pack_bf(acc[u][t][0], acc[u][t][1]), pack_bf(acc[u + 1][t][0], acc[u + 1][t][1]), false, false);
        const u32x2 d = __builtin_amdgcn_permlane16_swap(pack_bf(acc[u][t][2], acc[u][t][3]), pack_bf(acc[u + 1][t][2], acc[u + 1][t][3]), false, false);
        uint4 v = make_uint4(c[0], d[0], c[1], d[1]);
        if (EPI == EPI_RESIDUAL) {
          auto sum = [](uint32_t r, uint32_t y) { return pack_bf(lo_bf(r) + lo_bf(y), hi_bf(r) + hi_bf(y)); };
          v = make_uint4(sum(res[t].x, v.x), sum(res[t].y, v.y), sum(res[t].z, v.z), sum(res[t].w, v.w));
        }
        if (b < a.B && col < a.N) *reinterpret_cast<uint4*>(a.out + (size_t)b * a.ldo + col) = v;
      }
    }
    if (FN & 1) {
      constexpr int u = FN - 1;
      EpiPre pre[FM];
#pragma unroll
      for (int t = 0; t < FM; ++t) gemm_epilogue_fetch<EPI>(a, rbase + t * 16 + m, min(sbase + u, nstrips - 1), g, pre[t]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const int b = rbase + t * 16 + m;
        if (b < a.B && sbase + u < nstrips) gemm_epilogue<EPI, true>(a, b, sbase + u, g, acc[u][t], pre[t]);
      }
    }
    return;
  }
  constexpr bool READS = EPI == EPI_RESIDUAL || EPI == EPI_ROPE || EPI == EPI_BIAS || EPI == EPI_BIAS_GELU ||
                         EPI == EPI_BIAS_ADD2 || EPI == EPI_PHI_IN || EPI == EPI_BIAS_XIELU;
  if (READS && a.N >= 4 && ((a.N | a.ldo | a.ldr | (EPI == EPI_BIAS_ADD2 ? a.ldr2 : 0)) & 3) == 0) {
#pragma unroll
    for (int u = 0; u < FN; ++u) {  // a strip at a time: more sets of operands would cost a resident workgroup
      EpiPre pre[FM];
#pragma unroll
      for (int t = 0; t < FM; ++t) gemm_epilogue_fetch<EPI>(a, rbase + t * 16 + m, min(sbase + u, nstrips - 1), g, pre[t]);
      __builtin_amdgcn_sched_barrier(0);
      if (sbase + u >= nstrips) continue;
#pragma unroll
      for (int t = 0; t < FM; ++t) {
        const int b = rbase + t * 16 + m;
        if (b < a.B) gemm_epilogue<EPI, true>(a, b, sbase + u, g, acc[u][t], pre[t]);
      }
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < FN; ++u) {
    if (sbase + u >= nstrips) continue;
#pragma unroll
    for (int t = 0; t < FM; ++t) {
      const int b = rbase + t * 16 + m;
      if (b < a.B) gemm_epilogue<EPI>(a, b, sbase + u, g, acc[u][t]);
    }
  }
}

// ALIGNED: activation rows start on 16 bytes and a tile of them spans less than 4 GiB (false: through registers, any)
template <int EPI, class C, bool ALIGNED>
__global__ __launch_bounds__(C::NW * 64, 2) void gemm_tile_kernel(GemmArgs a, int MT, int NT, int nstrips) {
  constexpr int FM = C::FM, FN = C::FN;
  extern __shared__ __align__(16) unsigned char smem[];
  const int T = MT * NT;
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int base = T >> 3, rem = T & 7;
  if (q >= base + (xcd < rem ? 1 : 0)) return;
  const auto [row0, strip0] = tile_place<C>(xcd * base + min(xcd, rem) + q, MT, NT);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  XOffsets<C, ALIGNED> x;
#pragma unroll
  for (int i = 0; i < C::XPW; ++i) x.set(i, wave, lane, (typename XOffsets<C, ALIGNED>::type)(min(row0 + x.row(i, wave, lane), a.B - 1) - row0) * a.ldx);
  f32x4 acc[FN][FM];
  tile_product<C, ALIGNED>(acc, reinterpret_cast<const char*>(a.x + (size_t)row0 * a.ldx), x, a.wp, strip0, nstrips, a.K, wave, lane, smem);
  tile_epilogue<EPI, C>(a, acc, row0 + wave / C::WN * FM * 16, strip0 + wave % C::WN * FN, nstrips, lane);
}

// A workgroup a CU, which takes every 32nd tile of its XCD's run, where there are more tiles than CUs.  Its loads run from one tile into the next: what
// HalvesStream asks for in a tile's last steps are the first steps of the one behind it, which arrive under the epilogue.
// us, a workgroup a tile / this: 8192 rows 6144 x 768 with SwiGLU 77.8 / 73.2 (66 to 69 with the shorter silu), plain 77.2 / 73.3, 384 deep 55.8 / 48.6; 4001 rows 11264 x 2048 with SwiGLU 151 /
// 144, 11200 rows 399 / 377; 8192 rows 7680 x 2560 237 / 233.  What is left of a boundary there, 8 of 24 us a tile: the epilogue's arithmetic (SwiGLU 4 us), or where
// much is stored the memory (100 MB of a plain store 16.6 of 72.3 us); zeros instead of random numbers 53 us: the chip's clock under its load.
template <int EPI, class C>
__global__ __launch_bounds__(C::NW * 64, 2) void gemm_rounds_kernel(GemmArgs a, int MT, int NT, int nstrips) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int T = MT * NT, xcd = blockIdx.x & 7, base = T >> 3, rem = T & 7;
  const int first = xcd * base + min(xcd, rem), run = base + (xcd < rem ? 1 : 0), step = gridDim.x >> 3;
  int q = blockIdx.x >> 3;
  if (q >= run) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  HalvesStream<C> stream(a.wp, a.K, nstrips, wave, lane, smem);
  auto where = [&](TilePlace p) {  // the loads' place
    XOffsets<C, true> x;
#pragma unroll
    for (int i = 0; i < C::XPW; ++i) {
      x.set(i, wave, lane, (uint32_t)(min(p.row0 + x.row(i, wave, lane), a.B - 1) - p.row0) * a.ldx);
      stream.xoff[i] = x.off[i];
    }
    stream.xb = reinterpret_cast<const char*>(a.x + (size_t)p.row0 * a.ldx);
  };
  // What a wave stores at least of a whole tile with these epilogues, which ask for nothing but their place inside the output.
  constexpr int STORES = EPI == EPI_SWIGLU ? C::FM : EPI == EPI_STORE || EPI == EPI_RESIDUAL ? C::FM * (C::FN / 2) : 0;
  auto whole = [&](TilePlace p) { return p.row0 + C::TM <= a.B && (p.strip0 + C::TS) * (EPI == EPI_SWIGLU ? 8 : 16) <= a.N; };
  TilePlace here = tile_place<C>(first + q, MT, NT);
  where(here);
  stream.begin(here.strip0);
  bool stored = false;
  for (;;) {
    f32x4 acc[C::FN][C::FM];
    q += step;
    const bool more = q < run;
    const TilePlace next = more ? tile_place<C>(first + q, MT, NT) : here;  // (behind the last one: its own first steps, unused)
    stream.template walk<STORES>(acc, next.strip0, stored, [&] { where(next); });
    tile_epilogue<EPI, C>(a, acc, here.row0 + wave / C::WN * C::FM * 16, here.strip0 + wave % C::WN * C::FN, nstrips, lane);
    if (!more) break;
    stored = whole(here);
    here = next;
  }
  wait_loads<0>();  // (into LDS that is no longer this workgroup's otherwise)
}

template <int EPI, class C, bool ALIGNED = true>
int launch_tile(const GemmArgs& a, int nstrips, hipStream_t st) {
  const int64_t MT = (a.B + C::TM - 1) / C::TM, NT = (nstrips + C::TS - 1) / C::TS;
  if (MT * NT > INT32_MAX - 8) return OHARA_ESIZE;
  if constexpr (C::HALVES) {
    if (MT * NT > CUS && a.K % 64 == 0 && a.K >= 64 * C::XS) {
      (void)hipFuncSetAttribute((const void*)gemm_rounds_kernel<EPI, C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
      hipLaunchKernelGGL((gemm_rounds_kernel<EPI, C>), dim3(CUS), dim3(C::NW * 64), C::LDS, st, a, (int)MT, (int)NT, nstrips);
      return ohara_launch_status();
    }
  }
  if (C::LDS > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)gemm_tile_kernel<EPI, C, ALIGNED>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  hipLaunchKernelGGL((gemm_tile_kernel<EPI, C, ALIGNED>), dim3((unsigned)(MT * NT + 7) / 8 * 8), dim3(C::NW * 64), C::LDS, st, a,
                     (int)MT, (int)NT, nstrips);
  return ohara_launch_status();
}

// A part of the depth a workgroup, its fp32 sums to [part][row][16 nstrips]: where tiles over the whole depth are too few for the CUs or
// each of them takes in too much (50 GB/s a CU: 32 x 32 over 5632 are 720 KB).
template <class C>
__global__ __launch_bounds__(C::NW * 64, 2) void gemm_part_kernel(GemmArgs a, int MT, int NT, int nstrips, int parts, float* out) {
  constexpr int FM = C::FM, FN = C::FN;
  extern __shared__ __align__(16) unsigned char smem[];
  const int T = MT * NT * parts, xcd = blockIdx.x & 7, q = blockIdx.x >> 3;
  const int base = T >> 3, rem = T & 7;
  if (q >= base + (xcd < rem ? 1 : 0)) return;
  const int id = xcd * base + min(xcd, rem) + q, part = id / (MT * NT), pid = id - part * MT * NT;  // (an XCD: a part or two)
  const int row0 = (pid % MT) * C::TM, strip0 = (pid / MT) * C::TS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / C::WN, wn = wave % C::WN, m = lane & 15, g = lane >> 4;
  const int depth = a.K / parts;  // a multiple of 128
  XOffsets<C, true> x;
#pragma unroll
  for (int i = 0; i < C::XPW; ++i) x.set(i, wave, lane, (typename XOffsets<C, true>::type)(min(row0 + x.row(i, wave, lane), a.B - 1) - row0) * a.ldx);
  f32x4 acc[FN][FM];
  tile_product<C, true>(acc, reinterpret_cast<const char*>(a.x + (size_t)row0 * a.ldx + (size_t)part * depth), x, a.wp + (size_t)part * (depth / 32) * 64,
                        strip0, nstrips, depth, wave, lane, smem, a.K / 32);
  const int rbase = row0 + wm * FM * 16, sbase = strip0 + wn * FN;
#pragma unroll
  for (int u = 0; u < FN; ++u)
#pragma unroll
    for (int t = 0; t < FM; ++t) {
      const int b = rbase + t * 16 + m;
      if (b < a.B && sbase + u < nstrips)
        *reinterpret_cast<f32x4*>(out + (((size_t)part * a.B + b) * nstrips + sbase + u) * 16 + 4 * g) = acc[u][t];
    }
}

template <class C>
int launch_part(const GemmArgs& a, int nstrips, int parts, float* out, hipStream_t st) {
  const int64_t MT = (a.B + C::TM - 1) / C::TM, NT = (nstrips + C::TS - 1) / C::TS;
  if (MT * NT * parts > INT32_MAX - 8) return OHARA_ESIZE;
  if (C::LDS > 64 * 1024) (void)hipFuncSetAttribute((const void*)gemm_part_kernel<C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  hipLaunchKernelGGL((gemm_part_kernel<C>), dim3((unsigned)(MT * NT * parts + 7) / 8 * 8), dim3(C::NW * 64), C::LDS, st, a, (int)MT, (int)NT, nstrips,
                     parts, out);
  return ohara_launch_status();
}

//           waves fragments k-steps slots ahead (in halves: k-steps a phase, slots of activations and weights)
typedef Tile<2, 2, 1, 1, 4, 3, 1> T32;       //  32 x  32
typedef Tile<2, 2, 2, 2, 4, 2, 0> T64;       //  64 x  64
typedef Tile<2, 4, 2, 2, 2, 3, 1> T64x128;
typedef Tile<2, 4, 4, 2, 2, 2, 0> T128;
typedef Tile<2, 4, 4, 3, 2, 2, 0> T128x192;
typedef Tile<4, 1, 1, 3, 4, 3, 1> T64x48;
typedef Tile<2, 2, 2, 3, 4, 3, 0> T64x96;
// For fewer than 1024 rows, mostly a CU to themselves (few_rows_tile)
typedef Tile<1, 4, 3, 1, 4, 3, 0> T48x64;
typedef Tile<1, 4, 5, 1, 4, 3, 0> T80x64;
typedef Tile<2, 2, 3, 2, 2, 3, 0> T96x64;
typedef Tile<2, 2, 3, 3, 4, 3, 0> T96;
typedef Tile<2, 2, 4, 3, 2, 3, 0> T128x96;
typedef Tile<2, 2, 2, 2, 4, 3, 0> W64;       // as T64, T128 and T128x192, a slot more
typedef Tile<2, 4, 4, 2, 2, 3, 0> W128;
typedef Tile<2, 4, 4, 3, 2, 3, 0> W128x192;
typedef Tile<2, 4, 6, 2, 2, 3, 0> T192x128;
typedef HalvesTile<2, 4, 8, 4, 1, 3, 4> T256;
typedef HalvesTile<2, 4, 4, 4, 2, 3, 3> H128x256;
typedef HalvesTile<2, 4, 4, 3, 2, 3, 3> H128x192;

// Which tile: the one that should take least time.  A large tile needs less LDS traffic a product, a small one keeps more
// CUs busy and its chain of steps is shorter.  The times are fitted to measurements (63 shapes: 96 to 11200 rows, 768 to 17920 packed
// rows, K 768 to 10240); the choice they give is within 0.4 % of the best of the six on average, 13 % at worst.
struct TileTime {
  int rows, strips;
  int slots;    // workgroups that share a CU
  float alone;  // us a step of 64 takes one workgroup on a CU
  float more;   // what another one beside it adds, as a share of that (one slot: what a whole round of them adds)
  float full;   // us a step takes each of the workgroups of a full chip
  float ends;   // us the start and the epilogue add
};
constexpr TileTime TIMES[6] = {
    {T32::TM, T32::TS, 3, 0.14f, 0.376f, 0.079f, 0.43f},        {T64::TM, T64::TS, 2, 0.295f, 0.23f, 0.189f, 0.6f},
    {T64x128::TM, T64x128::TS, 2, 0.363f, 0.61f, 0.312f, 1.3f}, {T128::TM, T128::TS, 2, 0.60f, 0.56f, 0.453f, 1.45f},
    {T128x192::TM, T128x192::TS, 2, 0.747f, 0.64f, 0.6f, 3.15f}, {T256::TM, T256::TS, 1, 1.35f, 0.0f, 1.6f, 6.7f},
};
// From 1024 rows on, the tiles in halves among them: drawn through 1117 products of 1024 to 16384 rows, 256 to 18000 packed rows, K 256 to 5632, with
// the epilogues below, each as it stands in a model (128 MB of other work before it, then its activations written; weights, residual and output as that
// leaves them): the choice is within 0.9 % of the best of the eight on average, 0.7 % on the products left out of the fit.  A tile alone on its CU
// pays its ends once in every round.  (All with a workgroup a tile; since gemm_rounds_kernel the halves of more tiles than CUs take 5 to 13 % less than these
// times, and the choice is 0.5 to 2 % above the best of seven tiles on the widths of a model.)  Fewer rows are a round of small tiles or parts of the depth, to which the times above are fitted.
// (Timed one behind the other, with residual and output in the L2s, the tiles of two a CU come out up to 15 % better than they are: 8192 rows 768 x 768 with
// a residual 128 x 192 18.4 us there and 20.2 in the model, in halves 20.4 and 18.1.)
constexpr TileTime MANY[10] = {
    {T32::TM, T32::TS, 3, 0.114f, 0.157f, 0.113f, 0.706f}, {T64::TM, T64::TS, 2, 0.409f, 0.093f, 0.28f, 1.074f},
    {T64x128::TM, T64x128::TS, 2, 0.533f, 0.f, 0.525f, 2.505f}, {T128::TM, T128::TS, 2, 0.884f, 0.527f, 0.456f, 4.059f},
    {T128x192::TM, T128x192::TS, 2, 0.914f, 0.562f, 0.564f, 7.427f}, {T256::TM, T256::TS, 1, 0.842f, 0.814f, 1.527f, 15.093f},
    {H128x256::TM, H128x256::TS, 1, 0.67f, 0.262f, 0.846f, 8.608f}, {H128x192::TM, H128x192::TS, 1, 0.37f, 1.327f, 0.861f, 5.699f},
    {T64x48::TM, T64x48::TS}, {T64x96::TM, T64x96::TS},  // (by the rule below)
};
constexpr int LARGEST = 5;  // 256 x 256
// What an epilogue adds to a tile's ends there, us (beside the plain store's): nothing hides it where a CU has one tile.  Those of a residual, biases and gelu are
// measured; the rotary one is by whole table rows where a wave's strips lie in one head, in pieces of 4 bytes where they do not, and so of heads of n.
// us, one table for all epilogues / this: gelu, 2500 rows 4096 x 1024 50.4 / 40.5, 5500 rows 93.7 / 78.1, 2048 rows 17920 x 2560 246 / 213; rotary, heads
// of 32, 16384 rows 768 x 256 28.4 / 18.6, of 96, 5500 rows 1920 x 1152 42.8 / 36.5, of 48, 8192 rows 2304 x 1536 80 / 70.
enum Epilogue { PLAIN, GATED, RESIDUAL, BIAS, ADD2, HEAVY, ROTARY_64, ROTARY_32, ROTARY };  // ROTARY_n: heads of a multiple of n
constexpr float EXTRA[9][8] = {
    {},
    {0.f, 0.01f, 0.02f, 0.04f, 0.06f, 0.92f, 0.46f, 0.35f},
    {0.08f, 0.32f, 0.38f, 0.62f, 1.52f, 3.26f, 1.75f, 1.48f},
    {0.03f, 0.43f, 0.59f, 1.1f, 1.44f, 6.1f, 3.8f, 2.4f},
    {0.12f, 1.18f, 2.08f, 3.91f, 5.65f, 18.5f, 9.5f, 6.7f},
    {0.22f, 1.69f, 2.42f, 5.63f, 8.6f, 24.3f, 12.4f, 8.96f},
    {0.11f, 0.43f, 0.87f, 1.74f, 7.f, 2.4f, 1.2f, 7.f},
    {0.f, 0.f, 0.f, 0.f, 11.67f, 16.28f, 8.14f, 11.67f},
    {0.12f, 0.5f, 1.f, 2.f, 3.84f, 11.52f, 5.76f, 3.84f},
};
Epilogue epilogue_of(int epi, int dh, bool stage) {
  switch (epi) {
    case EPI_STORE: return PLAIN;
    case EPI_SWIGLU: return GATED;
    case EPI_RESIDUAL: return RESIDUAL;
    case EPI_BIAS: return BIAS;
    case EPI_BIAS_ADD2: return ADD2;
    case EPI_ROPE: return stage ? ROTARY : dh % 64 == 0 ? ROTARY_64 : dh % 32 == 0 ? ROTARY_32 : ROTARY;
    default: return HEAVY;
  }
}
// Fewer than 1024 rows: 64 x 48 and 64 x 96 where such tiles fill the chip once and those of 32 or 64 would a third round or half of one more:
// a CU takes in 50 to 90 GB/s, and one tile of 64 x 48 reads 112 rows of operands for the 3072 results of three of 32 x 32, which read 192.
// us, the best of the six / 64 x 48: 128 rows 6144 x 768 with SwiGLU 6.8 / 5.9, 96 rows 6.0 / 5.7, 33 rows 11264 x 2048 14.2 / 11.8, 192 rows
// 3072 x 2048 with rotary 13.7 / 11.7, 256 rows 14.8 / 12.1, 320 rows 2048 x 2048 12.6 / 11.5 (two rounds of 32 x 32: 160 rows 3072 x 2048
// 10.8 / 11.4), but not with an arithmetic epilogue, where its waves have twelve strips' rows each and the chain is short: with gelu 192 rows 3072 x 768 6.5 / 7.1,
// 600 rows 1024 x 1024 7.9 / 8.8, 224 rows 2560 x 2560 12.6 / 13.1, 10240 deep 54 / 41.
// 64 x 96 where what is read is the weights or a long depth, or 64 x 64 is a round and a half, and nothing but the sums is stored: 65 to 128 rows 11264 x 2048
// 17.2 to 18.0 / 15.0 to 15.7, 320 rows 4096 x 4096 28.1 / 24.2 (192 rows 6144 x 768 7.6 / 7.4, 160 rows 6.8 / 7.0; with rotary 384 rows 3072 x 2048 13.8 /
// 15.5, 1024 deep 8.5 / 10.2; with a residual 600 rows 2048 x 2048 13.8 / 14.8, 850 rows 1536 x 1536 10.7 / 11.6; 256 rows 5632 x 1024 with SwiGLU 8.2 / 8.7).
int one_round_tile(int rows, int strips, int K, Epilogue epi, int parts) {
  auto tiles = [&](int r, int s) { return ((int64_t)rows + r - 1) / r * ((strips + s - 1) / s) * parts; };
  const int64_t narrow = tiles(T64x48::TM, T64x48::TS), wide = tiles(T64x96::TM, T64x96::TS);
  if (K >= 512 && narrow >= 192 && narrow <= 256 && tiles(32, 2) > 512) return epi != HEAVY || K >= 4096 ? 8 : -1;
  return epi <= GATED && rows > 64 && K >= 1024 && wide >= 192 && wide <= 256 && (rows <= 128 || K >= 4096 || tiles(64, 4) >= 384) ? 9 : -1;
}
// `lone`: one full round and nothing behind it takes the chain's time, as a round that lacks a tile does; workgroups of several rounds drift apart.  us, where
// that decides: 16384 rows 768 x 3072 with a residual 78.3 in 512 tiles of 128 x 192, 74.9 in 192 of 256 x 256; 768 x 768 23.1 / 22.1; 8192 rows 1024 x 1024
// with a bias 22.5 of 128 x 128, 20.7 of 128 x 256 in halves.  (TIMES are fitted without.)
// In parts of the depth: K and the strips are a part's, which no tile reaches over.  us with the merge, counted as one product of all parts' strips / so: 375 rows
// 2640 x 11264 in eight parts, 252 tiles of 128 x 256 that are 264, 49.3 / 39.5 (of 128 x 128); 375 rows 784 x 4096 in four 17.1 / 14.3; 612 rows 20.3 / 16.9;
// 1702 rows 848 x 7168 45.8 / 35.6; of 1355 such calls 55 change, 9 % quicker on average, one of them 13 % slower (80 rows 784 x 4096 9.1 / 10.3).
float tile_time(const TileTime& t, int rows, int strips, int K, float extra = 0.f, bool lone = false, int parts = 1) {
  const int64_t tiles = ((int64_t)rows + t.rows - 1) / t.rows * ((strips + t.strips - 1) / t.strips) * parts;
  const int64_t waves = lone && tiles == CUS * t.slots ? 0 : tiles / (CUS * t.slots), rest = tiles - waves * CUS * t.slots;
  float step = waves * t.slots * t.full;
  if (rest) {
    const float others = t.slots == 1 ? rest * (1.f / CUS) : (float)((rest + CUS - 1) / CUS - 1);
    const float chain = t.alone * (1.f + t.more * others), chip = rest * (1.f / CUS) * t.full;
    step += rest <= CUS || chain > chip ? chain : chip;
  }
  const float rounds = t.slots == 1 ? (float)((tiles + CUS - 1) / CUS) : tiles > CUS ? tiles * (1.f / CUS) : 1.f;
  return step * K * (1.f / 64.f) + (t.ends + extra) * rounds;
}

int fastest_tile(int rows, int strips, int K, Epilogue epi = PLAIN, int parts = 1) {
  const bool many = rows >= 1024;
  if (const int i = one_round_tile(rows, strips, K, epi, parts); !many && i >= 0) return i;
  int best = 0;
  float low = INFINITY;
  for (int i = 0; i < (K < 64 ? 5 : many ? 8 : 6); ++i) {  // (halves walk whole steps)
    const float t = many ? tile_time(MANY[i], rows, strips, K, EXTRA[epi][i], true, parts) : tile_time(TIMES[i], rows, strips, K, 0.f, false, parts);
    if (t < low) {
      low = t;
      best = i;
    }
  }
  return best;
}

// Fewer than 1024 rows are a round or two of tiles, and what decides is whether they are one: 192 rows 11264 x 2048 were 264 tiles of 64 x 128, eight CUs with
// two, 22.1 us, and are 236 of 96 x 96, 18.2.  So there are tiles of more sizes, a ring of three slots each.  The times below are fitted to 1224 products
// (17 of a model's widths and depths whole, 8 in parts; 33 to 1023 rows; each tile that makes 48 to 1600 workgroups; cold weights), those of a
// tile alone on its CU within 3 to 5 %, of those that share one within 7 to 12 %.  Such a tile is taken where they promise 4 % (10 with an arithmetic
// epilogue, whose waves hold more of it): of the 1201 products with a choice 340 change, 12 % quicker on average (as much as 30), 21 lose more than 3 %, the worst 9
// (768 x 3072 in two parts, 860 rows: 10.7 / 11.7).  Of 2401 others, drawn, with the rules below and their weights from memory, 974 are more than 2 % quicker than
// without such tiles, 37 slower, the worst 7 (65 rows 12288 x 768 with rotary 10.3 / 11.0); with weights that stay in the 256 MB of cache 80 x 64 loses up to 16.
// us, before / now: 224 rows 11264 x 2048 with SwiGLU 26.7 / 21.1, 320 rows 3072 x 2048 14.9 / 11.4, 1000 rows 27.7 / 20.4, 400 rows 15.4 / 13.1.
constexpr int NEW_TILES = 10;  // the first of these tiles
constexpr TileTime FEW[19] = {
    {T32::TM, T32::TS, 3, 0.147f, 0.412f, 0.081f, 0.482f},          {T64::TM, T64::TS, 2, 0.302f, 0.252f, 0.208f, 0.779f},
    {T64x128::TM, T64x128::TS, 2, 0.374f, 0.684f, 0.337f, 1.577f},  {T128::TM, T128::TS, 2, 0.637f, 0.476f, 0.563f, 1.948f},
    {T128x192::TM, T128x192::TS, 2, 0.756f, 0.68f, 0.68f, 3.227f},  {T256::TM, T256::TS, 1, 1.35f, 0.f, 1.6f, 6.7f},
    {H128x256::TM, H128x256::TS}, {H128x192::TM, H128x192::TS},     // (below)
    {T64x48::TM, T64x48::TS, 1, 0.195f, 0.254f, 0.228f, 1.248f},    {T64x96::TM, T64x96::TS, 1, 0.287f, 0.234f, 0.336f, 1.634f},
    {T48x64::TM, T48x64::TS, 1, 0.199f, 0.191f, 0.231f, 1.229f},    {T80x64::TM, T80x64::TS, 1, 0.261f, 0.193f, 0.302f, 1.51f},
    {T96x64::TM, T96x64::TS, 2, 0.358f, 0.406f, 0.256f, 1.253f},    {T96::TM, T96::TS, 1, 0.355f, 0.242f, 0.426f, 1.968f},
    {T128x96::TM, T128x96::TS, 1, 0.441f, 0.181f, 0.507f, 2.426f},  {W64::TM, W64::TS, 1, 0.23f, 0.19f, 0.264f, 1.314f},
    {W128::TM, W128::TS, 1, 0.468f, 0.247f, 0.592f, 2.966f},        {W128x192::TM, W128x192::TS, 1, 0.599f, 0.262f, 0.758f, 4.159f},
    {T192x128::TM, T192x128::TS, 1, 0.6f, 0.25f, 0.764f, 4.011f},
};
// Tiles in halves among them: slower than the others until the operands of a large product come through them, and then by as much as a quarter
// quicker.  Fitted to 9400 products of 200 to 1023 rows (1024 to 18000 packed rows, K 384 to 4096, weights of HBM), and compared with the times above and what those
// lack on the same products, 2 us, with an arithmetic epilogue or where it is 128 x 192 4 (845 rows 6848 x 1344 with SwiGLU 24.6 / 20.2, 804 rows 12288 x 1024 with rotary
// 36.3 / 31.5, 474 rows 3008 x 5120 in four parts 32.3 / 28.9); no fewer tiles than leave most CUs idle, no depth under 768, where 515 more of those products
// would change, 0.4 % quicker on average, and 152 of them lose more than 3 %.  (39 whole products with a residual, 4096 to 10240 deep, beyond the fit, take 24 % less.)
// Of those of 768 and more 3900 change, 9 % quicker on average, 180 lose more than 3 %; of 1760 with rotary 650 change (14 %, none loses), of 1820 heads of Phi
// blocks 600 (6 %), of 2390 products in parts 1600 (10 %, 70 lose).  us, before / in halves: 512 rows 11264 x 2048 with SwiGLU 32.7 / 28.0, 1000 rows 48.7 / 44.4;
// 700 rows 6144 x 768 13.6 / 12.3; 700 rows 7680 x 2560 42.0 / 34.3; 700 rows 2560 x 10240 in four parts with their merge 51.7 / 47.4, 450 rows 48.3 / 39.4.
constexpr TileTime HALVES[3] = {
    {T256::TM, T256::TS, 1, 0.521f, 1.671f, 1.479f, 11.155f},
    {H128x256::TM, H128x256::TS, 1, 0.507f, 0.766f, 0.768f, 6.323f},
    {H128x192::TM, H128x192::TS, 1, 0.437f, 0.736f, 0.627f, 5.293f},
};
// Where the times promise what is not so, us there / with the tile that stays: tiles of 64 x 48 that are a round against those of 48 x 64 (all 41 such products of
// 3900 lose: 45 rows 10272 x 1920 with SwiGLU 14.8 / 13.6, 47 rows 9216 x 1536 with rotary 13.3 / 11.8), and tiles of 64 x 128 of which a few CUs have two against 96 x
// 64 (217 rows of a Phi head 8272 x 2528, 260 of them: 32.6 / 30.1 with 128 x 96, 28.3 with 64 x 128; from 268 on those lose).
int few_rows_tile(int rows, int strips, int K, Epilogue epi, int parts = 1) {
  const int now = fastest_tile(rows, strips, K, epi, parts);
  if (rows >= 1024) return now;
  auto time = [&](const TileTime& t, float extra = 0.f) { return tile_time(t, rows, strips, K, extra, false, parts); };
  const int64_t wide = ((int64_t)rows + T64x128::TM - 1) / T64x128::TM * ((strips + T64x128::TS - 1) / T64x128::TS) * parts;
  const bool just_over = now == 2 && wide > CUS && wide < CUS + CUS / 25;
  int best = now;
  float low = (epi == HEAVY ? 0.9f : 0.96f) * time(FEW[now]);
  for (int i = NEW_TILES; i < 19; ++i) {
    if ((now == 8 && i == 10) || (just_over && i == 12)) continue;
    const float t = time(FEW[i]);
    if (t < low) {
      low = t;
      best = i;
    }
  }
  if (K < 768) return best;
  low = time(FEW[best]) + (epi == HEAVY || best == 4 ? 4.f : 2.f);
  for (int i = 0; i < 3; ++i) {
    const TileTime& h = HALVES[i];
    if (((int64_t)rows + h.rows - 1) / h.rows * ((strips + h.strips - 1) / h.strips) * parts < (i ? 96 : 136)) continue;
    const float extra = epi == HEAVY ? (i ? 3.f : 6.f) : epi >= ROTARY_32 ? EXTRA[epi][LARGEST + i] : 0.f;
    const float t = time(h, extra);
    if (t < low) {
      low = t;
      best = LARGEST + i;
    }
  }
  return best;
}
constexpr bool has_new_tiles(int epi) { return epi == EPI_RESIDUAL || epi == EPI_SWIGLU || epi == EPI_ROPE || epi == EPI_PHI_IN || epi == EPI_STORE; }
// A plain store has them from 20000 packed rows on, a vocabulary: under that ohara_gemm_tile_of says what it runs, whatever the number of rows.  us, without / with: 32000 x
// 2048, 128, 192, 256, 384, 700 rows 35.7 40.7 45.7 52.2 94.7 / 36.2 34.0 40.5 51.7 88.5; 65536 x 768, 128, 300, 384 rows 28.4 48.4 55.9 / 28.1 43.3 49.1.  (With a
// bias, as Phi's is stored, there are none of them: that epilogue's tiles are the six and the two of a round.)
int tile_of(int rows, int strips, int K, int epi, Epilogue kind) {
  return has_new_tiles(epi) && (epi != EPI_STORE || strips >= 1250) ? few_rows_tile(rows, strips, K, kind) : fastest_tile(rows, strips, K, kind);
}

// A part of the rows in whole rounds of 256 x 256, one a CU, and the rest by itself, where the last round would be nearly empty (0 rows: all in one launch).
// The times of two launches are those above, added, and 5 us for the second one's start; taken from 3 % on.  us, one / two launches: 8192 rows 2304 x 768 with
// rotary 43.9 / 41.7, heads of 64 43.4 / 39.1, 16384 rows 79.0 / 72.3, 5500 rows 6144 x 768 with SwiGLU 59.8 / 53.9, 5421 rows 2992 x 2560 99.4 / 81.8, 8192 rows
// 2560 x 10240 375 / 326.  Of 456 products that the sum without those 5 us puts first 215 lose by it, those under 768 deep by 10 % on average and with a
// bias by up to 40; of the 148 that this takes, 7 % quicker, 15 lose, one of them 33 % and the others 9 % at most.  (First rounds of 128 x 256 lose more often than not.)
int split_rows(int rows, int strips, int K, Epilogue epi) {
  if (rows < 1024 || K < 768) return 0;
  auto time = [&](int i, int r) { return tile_time(MANY[i], r, strips, K, EXTRA[epi][i], true); };
  auto least = [&](int r) {
    float low = INFINITY;
    for (int i = 0; i < 8; ++i) low = std::min(low, time(i, r));
    return low;
  };
  const int64_t across = (strips + T256::TS - 1) / T256::TS, down = ((int64_t)rows + T256::TM - 1) / T256::TM;
  const int64_t first = across * down / 256 * 256 / across * T256::TM;
  if (first < 1 || first >= rows) return 0;
  return time(LARGEST, (int)first) + least(rows - (int)first) + 5.f < 0.97f * least(rows) ? (int)first : 0;
}

template <int EPI>
int launch_of(int tile, const GemmArgs& a, int nstrips, hipStream_t st) {
  if constexpr (has_new_tiles(EPI)) {
    switch (tile) {
      case 10: return launch_tile<EPI, T48x64>(a, nstrips, st);
      case 11: return launch_tile<EPI, T80x64>(a, nstrips, st);
      case 12: return launch_tile<EPI, T96x64>(a, nstrips, st);
      case 13: return launch_tile<EPI, T96>(a, nstrips, st);
      case 14: return launch_tile<EPI, T128x96>(a, nstrips, st);
      case 15: return launch_tile<EPI, W64>(a, nstrips, st);
      case 16: return launch_tile<EPI, W128>(a, nstrips, st);
      case 17: return launch_tile<EPI, W128x192>(a, nstrips, st);
      case 18: return launch_tile<EPI, T192x128>(a, nstrips, st);
      default: break;
    }
  }
  switch (tile) {
    case 0: return launch_tile<EPI, T32>(a, nstrips, st);
    case 1: return launch_tile<EPI, T64>(a, nstrips, st);
    case 2: return launch_tile<EPI, T64x128>(a, nstrips, st);
    case 3: return launch_tile<EPI, T128>(a, nstrips, st);
    case 4: return launch_tile<EPI, T128x192>(a, nstrips, st);
    case 5: return launch_tile<EPI, T256>(a, nstrips, st);
    case 6: return launch_tile<EPI, H128x256>(a, nstrips, st);
    case 7: return launch_tile<EPI, H128x192>(a, nstrips, st);
    case 8: return launch_tile<EPI, T64x48>(a, nstrips, st);
    default: return launch_tile<EPI, T64x96>(a, nstrips, st);
  }
}
template <int EPI>
int launch_epi(const GemmArgs& a, int nstrips, hipStream_t st) {
  if (((uintptr_t)a.x & 15) != 0 || (uint64_t)T256::TM * a.ldx * 2 > UINT32_MAX) return launch_tile<EPI, T64, false>(a, nstrips, st);
  const Epilogue epi = epilogue_of(EPI, a.Dh, a.stage);
  const int split = split_rows(a.B, nstrips, a.K, epi);
  if (!split) return launch_of<EPI>(tile_of(a.B, nstrips, a.K, EPI, epi), a, nstrips, st);
  GemmArgs first = a, rest = a;
  first.B = split;
  rest.B = a.B - split;
  rest.x += (size_t)split * a.ldx;
  rest.row0 += split;
  if (EPI != EPI_ROPE && EPI != EPI_PHI_IN) {  // (those find their rows from row0)
    rest.out += (size_t)split * a.ldo;
    if (a.resid) rest.resid += (size_t)split * a.ldr;
    if (a.resid2) rest.resid2 += (size_t)split * a.ldr2;
    if (a.ids) rest.ids += split;
  }
  const int rc = launch_of<EPI>(LARGEST, first, nstrips, st);
  return rc ? rc : launch_of<EPI>(tile_of(rest.B, nstrips, a.K, EPI, epi), rest, nstrips, st);
}

float least_time(int rows, int strips, int K) {
  float low = tile_time(TIMES[0], rows, strips, K);
  for (int i = 1; i < 6; ++i) low = std::min(low, tile_time(TIMES[i], rows, strips, K));
  return low;
}

}  // namespace

// In how many parts the depth is multiplied: those of least time, the tiles' and the merge's, which is the sums written and
// read at 8 TB/s (they stay in the caches) and merge_us.  Priced with the six tiles of TIMES at any number of rows, also where another one is launched, and as if
// tiles reached from part to part:
// us, as chosen / best: 2048 x 5632, 1800 rows 63 whole / 55 in two parts, 768 x 3072, 1024 rows 23 whole / 18.6 in two; over 15 shapes and 29 numbers of
// rows from 33 to 4096 4 % above the best choice on average.  us with what follows the product, whole / in parts:
//   2048 x 5632, residual and norm, 33, 65, 192, 400, 700, 1500 rows  21.1 21.6 26.8 41.2 42.2 58.8 / 11.2 14.6 19.0 28.6 33.2 54.5
//   768 x 3072                      65, 128, 256, 512, 700            11.9 11.9 12.0 13.7 17.6      /  7.5  8.0  9.9 12.3 14.2
//   2560 x 10240, bias and addends  33, 128, 256, 700, 1000           31.7 43.0 59.4 72.3 116       / 20.1 28.3 32.7 52.8 71.1
// and 2048 x 2048 in parts at 33 rows (10.3 / 7.6), whole from 700 on (17.1).  (At 4 TB/s the rule left 512 x 768 x 3072 and 700 rows of
// the other two whole.)
int ohara_depth_parts(int rows, int packed_rows, int k, float merge_us) {
  const int strips = packed_rows / 16;
  int best = 1;
  float low = 0.95f * least_time(rows, strips, k);
  for (int p = 2; p <= 8; p *= 2) {
    if (k % (128 * p) || k / p < (p == 2 ? 384 : 512) || (int64_t)strips * p > INT32_MAX / 16) continue;
    const float t = least_time(rows, strips * p, k / p) + (float)p * rows * strips * 16 * 8 * (1.f / 8e6f) + merge_us;
    if (t < low) {
      low = t;
      best = p;
    }
  }
  return best;
}

// a.x on 16 bytes, its rows a.ldx % 8 == 0 apart; parts as ohara_depth_parts; sums: [part][row][packed_rows].
int ohara_launch_gemm_parts(const GemmArgs& a, int packed_rows, int parts, float* sums, hipStream_t st) {
  const int nstrips = packed_rows / 16;
  if (parts < 2 || a.K % (128 * parts) || ((uintptr_t)a.x & 15) || (a.ldx & 7) || (uint64_t)T256::TM * a.ldx * 2 > UINT32_MAX) return OHARA_EINVAL;
  switch (few_rows_tile(a.B, nstrips, a.K / parts, PLAIN, parts)) {
    case 0: return launch_part<T32>(a, nstrips, parts, sums, st);
    case 1: return launch_part<T64>(a, nstrips, parts, sums, st);
    case 2: return launch_part<T64x128>(a, nstrips, parts, sums, st);
    case 3: return launch_part<T128>(a, nstrips, parts, sums, st);
    case 4: return launch_part<T128x192>(a, nstrips, parts, sums, st);
    case 5: return launch_part<T256>(a, nstrips, parts, sums, st);
    case 6: return launch_part<H128x256>(a, nstrips, parts, sums, st);
    case 7: return launch_part<H128x192>(a, nstrips, parts, sums, st);
    case 8: return launch_part<T64x48>(a, nstrips, parts, sums, st);
    case 9: return launch_part<T64x96>(a, nstrips, parts, sums, st);
    case 10: return launch_part<T48x64>(a, nstrips, parts, sums, st);
    case 11: return launch_part<T80x64>(a, nstrips, parts, sums, st);
    case 12: return launch_part<T96x64>(a, nstrips, parts, sums, st);
    case 13: return launch_part<T96>(a, nstrips, parts, sums, st);
    case 14: return launch_part<T128x96>(a, nstrips, parts, sums, st);
    case 15: return launch_part<W64>(a, nstrips, parts, sums, st);
    case 16: return launch_part<W128>(a, nstrips, parts, sums, st);
    case 17: return launch_part<W128x192>(a, nstrips, parts, sums, st);
    default: return launch_part<T192x128>(a, nstrips, parts, sums, st);
  }
}

// Launcher shared with the skinny entry points (declared there).
int ohara_launch_gemm_tile(const GemmArgs& a, int epi, int packed_rows, hipStream_t st) {
  const int nstrips = packed_rows / 16;
  switch (epi) {
    case EPI_STORE: return launch_epi<EPI_STORE>(a, nstrips, st);
    case EPI_RESIDUAL: return launch_epi<EPI_RESIDUAL>(a, nstrips, st);
    case EPI_SWIGLU: return launch_epi<EPI_SWIGLU>(a, nstrips, st);
    case EPI_ROPE: return launch_epi<EPI_ROPE>(a, nstrips, st);
    case EPI_BIAS: return launch_epi<EPI_BIAS>(a, nstrips, st);
    case EPI_BIAS_GELU: return launch_epi<EPI_BIAS_GELU>(a, nstrips, st);
    case EPI_BIAS_ADD2: return launch_epi<EPI_BIAS_ADD2>(a, nstrips, st);
    case EPI_PHI_IN: return launch_epi<EPI_PHI_IN>(a, nstrips, st);
    case EPI_SOFTCAP: return launch_epi<EPI_SOFTCAP>(a, nstrips, st);
    case EPI_GELU_LOOKUP: return launch_epi<EPI_GELU_LOOKUP>(a, nstrips, st);
    case EPI_BIAS_XIELU: return launch_epi<EPI_BIAS_XIELU>(a, nstrips, st);
    case EPI_GLU: return launch_epi<EPI_GLU>(a, nstrips, st);
    default: return OHARA_EINVAL;
  }
}

extern "C" int ohara_gemm_tile_of(int rows, int packed_rows, int k) {
  if (rows < 1 || packed_rows < 1 || k < 1) return OHARA_EINVAL;
  const TileTime& t = MANY[fastest_tile(rows, (packed_rows + 15) / 16, k)];  // (its sizes are those of both)
  return t.rows * 1000 + t.strips * 16;
}

extern "C" int ohara_gemm_tile_with(int rows, int packed_rows, int k, int epilogue, int parts) {
  if (rows < 1 || packed_rows < 1 || k < 1 || epilogue < EPI_STORE || epilogue > EPI_BIAS_XIELU || parts < 1 || k % parts) return OHARA_EINVAL;
  const int strips = (packed_rows + 15) / 16;
  const int i = parts > 1 ? few_rows_tile(rows, strips, k / parts, PLAIN, parts) : tile_of(rows, strips, k, epilogue, epilogue_of(epilogue, 64, false));
  return FEW[i].rows * 1000 + FEW[i].strips * 16 + (i >= LARGEST && i < LARGEST + 3);
}

extern "C" int ohara_gemm_first_rows(int rows, int packed_rows, int k, int epilogue, int dh) {
  if (rows < 1 || packed_rows < 1 || k < 1 || epilogue < EPI_STORE || epilogue > EPI_BIAS_XIELU || (epilogue == EPI_ROPE && dh < 1)) return OHARA_EINVAL;
  return split_rows(rows, (packed_rows + 15) / 16, k, epilogue_of(epilogue, dh, false));
}

extern "C" int ohara_gemm_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, int rows, int epilogue,
                               const uint16_t* resid, int ldr, uint16_t* out, int ldo, void* stream) {
  if (!x || !wp || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;  // 16-byte activation loads
  if (epilogue == OHARA_EPI_RESIDUAL && (!resid || ldr < n)) return OHARA_EINVAL;
  if (epilogue < OHARA_EPI_STORE || epilogue > OHARA_EPI_SWIGLU) return OHARA_EINVAL;
  if (ldo < n) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx;
  a.B = rows; a.N = n; a.K = k;
  a.out = out; a.ldo = ldo; a.resid = resid; a.ldr = ldr;
  const int packed_rows = epilogue == OHARA_EPI_SWIGLU ? 2 * ((n + 7) / 8 * 8) : (n + 15) / 16 * 16;
  return ohara_launch_gemm_tile(a, epilogue, packed_rows, (hipStream_t)stream);
}
