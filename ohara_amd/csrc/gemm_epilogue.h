// Shared by the skinny (decode) and tiled (prefill) GEMM kernels: argument block and the
// fused epilogues.  Rounding points follow the reference's bf16 eager path:
//   residual add       ohara/models/llama.py:199-200
//   SwiGLU             ohara/modules/mlp.py:152
//   rotary + KV append ohara/embeddings_pos/rotary.py:55-93, ohara/modules/kv_cache.py:104-105
//   bias / new_gelu / parallel-block sum of Phi   ohara/models/phi.py:37-52, :147-151
//   soft cap of the fp32 sum (vocabulary projections with capped logits)
//   gelu of the fp32 sum times an embedding of the row's token
//   clamped gated unit of the fp32 sums
//   bias and two-sided activation of the fp32 sums
#pragma once
#include "common.h"

enum { EPI_STORE = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2, EPI_ROPE = 3, EPI_BIAS = 4, EPI_BIAS_GELU = 5, EPI_BIAS_ADD2 = 6, EPI_PHI_IN = 7, EPI_SOFTCAP = 8, EPI_GELU_LOOKUP = 9, EPI_GLU = 10, EPI_BIAS_XIELU = 11 };

struct GemmArgs {
  const uint4* wp;
  const bf16_t* x;
  int ldx;
  const bf16_t* norm_w;
  float eps;
  int B, N, K;  // rows, logical output width (EPI_SWIGLU: hidden width F) and depth
  bf16_t* out;
  int ldo;
  const bf16_t* resid;
  int ldr;
  // rotary + append
  int H, Hkv, Dh, Tmax, pos;
  int S, row0;  // rows are (sequence, position) pairs: row = seq * S + s, position = pos + s
  int ny, nstrips;  // skinny kernel: 16-row chunks per strip (workgroups of a strip share an XCD) and strips
  const int32_t* pos_dev;
  const int32_t* rows;  // when set: the position of every row, then (nrows of them each) the row of the cache its sequence is in
  int nrows;
  int pos_stride;  // 0: *pos_dev is the position of every sequence; 1: pos_dev[seq] (ragged batches)
  const bf16_t* cos;
  const bf16_t* sin;
  bf16_t* kcache;
  bf16_t* vcache;
  int stage;  // rotary epilogue: k / v rows go to (rows, Hkv*Dh) buffers at the row index instead of into a cache
  // nn.Linear with bias (EPI_BIAS*): y = bf16(acc + bias[n]); EPI_BIAS_ADD2: bf16(bf16(resid + y) + resid2)
  const bf16_t* bias;
  const bf16_t* resid2;
  int ldr2;
  // LayerNorm prologue (NORM == 2): norm_w / norm_b
  const bf16_t* norm_b;
  // EPI_PHI_IN: packed rows [q; k; v; fc1] off one normalised input (phi.py:81-83, :50): rows below
  // split_n are the QKV projection (q -> out, k / v rows -> cache position pos + s, un-rotated), the
  // rest go through new_gelu into out2
  int split_n;
  bf16_t* out2;
  int ldo2;
  float cap;  // EPI_SOFTCAP: cap * tanh(acc / cap)
  // EPI_GELU_LOOKUP: bf16(gelu_tanh(acc) * table[ids[row] * ldt + n]); ids belong to the rows of `out`
  const bf16_t* table;
  const int64_t* ids;
  int ldt, vocab;
  OharaGlu glu;  // EPI_GLU: packed rows as EPI_SWIGLU
  float above, below;  // EPI_BIAS_XIELU
};

// gemm_tile.hip: the tiled kernel for calls with many rows (a.B rows, no fused norm).
int ohara_launch_gemm_tile(const GemmArgs& a, int epi, int packed_rows, hipStream_t st);
int ohara_depth_parts(int rows, int packed_rows, int k, float merge_us);
constexpr int OHARA_PARTS_LDX = (1 << 23) - 1;  // rows further apart: a tile's (256 rows) are not addressed with 32 bits; not in parts
int ohara_launch_gemm_parts(const GemmArgs& a, int packed_rows, int parts, float* sums, hipStream_t st);

// Up to 64 rows: where a product in tiles is the quicker one, and where it is with the norm ahead of it as a launch of its own, than the strip
// kernels, which take a workgroup for every 16 rows of a strip (and norm them there).  W: those workgroups.  us, cold weights, at 17, 32, 33 and
// 64 rows (W: strips x 2, 2, 3, 4):
//   plain, strips / tiles   1024 x 2048 5.0 5.1 5.1 5.4 / 6.7 6.8 6.8 6.8;  2048 x 2048 5.5 5.5 7.8 8.0 / 6.8 6.9 6.9 6.9;  6144 x 2048 12.3 11.2 14.8
//     18.2 / 9.5 9.3 10.0 11.6;  2048 x 1152 4.2 4.6 5.6 6.2 / 5.1 5.2 5.2 5.2;  2560 x 1152 5.9 5.9 5.7 7.6 / 5.2;  1024 x 4096 7.6 7.5 7.9 8.0 / 10.7
//     10.7 10.7 10.8;  2048 x 4096 8.6 8.1 14.0 13.9 / 14.1 14.0 13.9 13.9;  with rotary, bias, gelu or SwiGLU alike: W > 256, a workgroup a CU
//   normed strips / norm and tiles   K to 1536: 2048 x 1280 5.6 5.9 7.4 8.2 / 7.9 8.0 8.0 8.1;  2560 x 1536 7.9 8.5 8.0 11.0 / 8.4 8.4 8.5 8.5;
//     6144 x 1280 9.4 10.2 15.4 18.3 / 9.7 9.8 10.5 11.7;  11264 x 1536 with SwiGLU 12.7 13.2 21.4 23.5 / 13.9 14.9 15.2 17.1: W > 512, from 33 rows.
//     K to 2048: 2048 x 1792 6.7 6.9 11.3 12.1 / 9.0 9.0 9.1 9.2;  6144 x 2048 12.5 13.2 19.9 23.2 / 12.2 12.1 12.8 14.3;  11264 x 2048 with SwiGLU 16.5 17.6
//     28.0 30.7 / 16.1 17.4 17.6 20.1;  32000 x 2048 30.9 31.3 112 161 / 30.8 31.1 30.9 31.3: W > 256, from 33 rows (up to 32 they are even alone; a
//     forward of eight layers, 17, 24 and 32 sequences a token: 2048 wide, 16 heads on 4 461 455 465 / 467 462 466, 1792, 14 on 2 1475 1480 1496 /
//     1556 1562 1563).  Deeper: 1024 x 2560 11.6 12.5 12.0 12.4, 7680 x 2560 33.8 32.3 40.5 54.2 / 16.8 15.6 16.4 19.2, a forward 1045 1022 995 /
//     662 661 657: always, from 17.
// To 1024: 6144 x 768 5.7 6.2 7.5 8.4 / 7.0 7.0 7.7 7.7, 3072 x 1024 6.1 6.3 7.2 8.2 / 7.2 7.3 7.3 7.4: 65 rows.  (By K alone, 17 rows past 1024, narrow
// projections lost up to 70 % and forwards of 17 to 32 rows up to 10.  A residual's product has nothing to norm: 65 rows, see its entry point.)
inline int64_t ohara_strip_workgroups(int rows, int packed_rows) { return (int64_t)((rows + 15) / 16) * (packed_rows / 16); }
inline bool ohara_tiles_win(int rows, int k, int packed_rows) {
  return rows > 64 || (rows > 16 && k > 1024 && ohara_strip_workgroups(rows, packed_rows) > 256);
}
inline bool ohara_norm_ahead(int rows, int k, int packed_rows) {
  if (rows > 64 || k > 2048) return rows > 16;
  return rows > 32 && k > 1024 && ohara_strip_workgroups(rows, packed_rows) > (k > 1536 ? 256 : 512);
}

namespace {

// phi.py:37-40 op by op, every result rounded as the eager bf16 ops round, two at a time; torch.pow(x, 3.0) on bf16 is (x * x) * x with both
// products rounded.  The values are bf16 numbers.  Us, with the library's tanh and roundings one by one / so: 700 rows 17920 x 2560 80 / 72, 1500 159 /
// 138, one row 18.0 / 17.7.
__device__ __forceinline__ void new_gelu(float (&v)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i += 2) {
    auto both = [&](auto f) {  // f of the pair, rounded
      const uint32_t p = pack_bf(f(0), f(1));
      return uint2{__float_as_uint(lo_bf(p)), __float_as_uint(hi_bf(p))};
    };
    const float x[2] = {v[i], v[i + 1]};
    auto of = [](uint2 u, int j) { return __uint_as_float(j ? u.y : u.x); };
    const uint2 sq = both([&](int j) { return x[j] * x[j]; });
    const uint2 cu = both([&](int j) { return of(sq, j) * x[j]; });
    const uint2 t1 = both([&](int j) { return 0.044715f * of(cu, j); });
    const uint2 t2 = both([&](int j) { return x[j] + of(t1, j); });
    const uint2 t3 = both([&](int j) { return 0.7978845608028654f * of(t2, j); });
    const uint2 t4 = both([&](int j) { return tanh_of_bf16(of(t3, j)); });
    const uint2 t5 = both([&](int j) { return 1.0f + of(t4, j); });
    const uint2 hx = both([&](int j) { return 0.5f * x[j]; });
#pragma unroll
    for (int j = 0; j < 2; ++j) v[i + j] = of(hx, j) * of(t5, j);
  }
}

// What an epilogue reads besides the accumulators, fetched ahead: a kernel that finishes many fragments
// per thread (the tiled GEMM: sixteen) issues the loads of all of them before the first is used instead of
// one dependent round trip per fragment.  gemm_epilogue_fetch requires N, ldo, ldr, ldr2 to be multiples
// of 4 (the caller checks once); fragments and rows outside the matrix read clamped addresses and are
// never finished.
struct EpiPre {
  uint2 r1, r2, bv;  // residual rows, bias
  uint32_t c, s;     // two cos and two sin values of the rotary table
  int pos;
};
template <int EPI>
__device__ __forceinline__ void gemm_epilogue_fetch(const GemmArgs& a, int b, int strip, int g, EpiPre& p) {
  const int r0 = min(strip * 16 + 4 * g, a.N - 4);
  const int bc = min(b, a.B - 1);
  if (EPI == EPI_RESIDUAL) p.r1 = *reinterpret_cast<const uint2*>(a.resid + (size_t)bc * a.ldr + r0);
  if (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_ADD2 || EPI == EPI_PHI_IN || EPI == EPI_BIAS_XIELU)
    p.bv = *reinterpret_cast<const uint2*>(a.bias + r0);
  if (EPI == EPI_BIAS_ADD2) {
    p.r1 = *reinterpret_cast<const uint2*>(a.resid + (size_t)bc * a.ldr + r0);
    p.r2 = *reinterpret_cast<const uint2*>(a.resid2 + (size_t)bc * a.ldr2 + r0);
  }
  if (EPI == EPI_ROPE) {
    const int grow = a.row0 + bc;
    const int seq = grow / a.S;
    p.pos = a.rows ? a.rows[grow] : (a.pos_dev ? a.pos_dev[(size_t)seq * a.pos_stride] : a.pos) + (grow - seq * a.S);
    const int nq = a.H * a.Dh;
    const int rr = strip * 16 + 4 * g;
    const int d = (rr < nq ? rr : rr - nq) % a.Dh;
    const int pc = min(max(p.pos, 0), a.Tmax - 1);
    p.c = *reinterpret_cast<const uint32_t*>(a.cos + (size_t)pc * (a.Dh >> 1) + (d >> 1));
    p.s = *reinterpret_cast<const uint32_t*>(a.sin + (size_t)pc * (a.Dh >> 1) + (d >> 1));
  }
}

// One MFMA output fragment: the four consecutive packed rows 16*strip + 4*g .. +3 of activation
// row b (relative to a.out / a.resid; global row a.row0 + b for the rotary epilogue).
template <int EPI, bool PRE = false>  // PRE: the operands were fetched ahead into `p`
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& a, int b, int strip, int g, f32x4 acc, const EpiPre& p = EpiPre{}) {
  const int r0 = strip * 16 + 4 * g;
  if (EPI == EPI_SOFTCAP) {
    bf16_t* o = a.out + (size_t)b * a.ldo + r0;
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a.cap * tanhf(acc[i] / a.cap);
    if (r0 + 3 < a.N && ((a.ldo & 3) == 0)) {
      *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r0 + i < a.N) o[i] = f2bf(v[i]);
    }
    return;
  }
  if (EPI == EPI_GELU_LOOKUP) {  // N, ldo and ldt are multiples of 4
    if (r0 >= a.N) return;
    int64_t id = a.ids[b];
    if (id < 0 || id >= a.vocab) id = 0;  // the host validates ids; never read out of bounds
    const uint2 ev = *reinterpret_cast<const uint2*>(a.table + (size_t)id * a.ldt + r0);
    const float e[4] = {lo_bf(ev.x), hi_bf(ev.x), lo_bf(ev.y), hi_bf(ev.y)};
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gelu_tanh(acc[i]) * e[i];
    *reinterpret_cast<uint2*>(a.out + (size_t)b * a.ldo + r0) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    return;
  }
  if (EPI == EPI_GLU) {  // rows as in EPI_SWIGLU; N and ldo are multiples of 2
    const int f = strip * 8 + 2 * g;
    if (f < a.N)
      *reinterpret_cast<uint32_t*>(a.out + (size_t)b * a.ldo + f) =
          pack_bf(clamped_glu(acc[0], acc[2], a.glu.limit, a.glu.alpha, a.glu.offset),
                  clamped_glu(acc[1], acc[3], a.glu.limit, a.glu.alpha, a.glu.offset));
    return;
  }
  if (EPI == EPI_BIAS_XIELU) {  // N % 4 == 0 and 4-element aligned leading dimensions
    if (r0 >= a.N) return;
    const uint2 bv = PRE ? p.bv : *reinterpret_cast<const uint2*>(a.bias + r0);
    const float v[4] = {xielu(acc[0] + lo_bf(bv.x), a.above, a.below), xielu(acc[1] + hi_bf(bv.x), a.above, a.below),
                        xielu(acc[2] + lo_bf(bv.y), a.above, a.below), xielu(acc[3] + hi_bf(bv.y), a.above, a.below)};
    *reinterpret_cast<uint2*>(a.out + (size_t)b * a.ldo + r0) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    return;
  }
  const float y0 = rbf(acc[0]), y1 = rbf(acc[1]), y2 = rbf(acc[2]), y3 = rbf(acc[3]);
  if (EPI == EPI_STORE || EPI == EPI_RESIDUAL) {
    float v[4] = {y0, y1, y2, y3};
    bf16_t* o = a.out + (size_t)b * a.ldo + r0;
    if (EPI == EPI_RESIDUAL) {
      const bf16_t* r = a.resid + (size_t)b * a.ldr + r0;
      if (r0 + 3 < a.N && ((a.ldr & 3) == 0)) {
        const uint2 rv = PRE ? p.r1 : *reinterpret_cast<const uint2*>(r);
        v[0] = lo_bf(rv.x) + v[0]; v[1] = hi_bf(rv.x) + v[1]; v[2] = lo_bf(rv.y) + v[2]; v[3] = hi_bf(rv.y) + v[3];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (r0 + i < a.N) v[i] = bf2f(r[i]) + v[i];
      }
    }
    if (r0 + 3 < a.N && ((a.ldo & 3) == 0)) {
      *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (r0 + i < a.N) o[i] = f2bf(v[i]);
    }
  } else if (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_ADD2) {
    // N % 4 == 0 and 4-element aligned leading dimensions are required by the entry point
    if (r0 >= a.N) return;
    const uint2 bv = PRE ? p.bv : *reinterpret_cast<const uint2*>(a.bias + r0);
    float v[4] = {rbf(acc[0] + lo_bf(bv.x)), rbf(acc[1] + hi_bf(bv.x)), rbf(acc[2] + lo_bf(bv.y)),
                  rbf(acc[3] + hi_bf(bv.y))};
    if (EPI == EPI_BIAS_GELU) {
      new_gelu(v);
    } else if (EPI == EPI_BIAS_ADD2) {
      const uint2 r1 = PRE ? p.r1 : *reinterpret_cast<const uint2*>(a.resid + (size_t)b * a.ldr + r0);
      const uint2 r2 = PRE ? p.r2 : *reinterpret_cast<const uint2*>(a.resid2 + (size_t)b * a.ldr2 + r0);
      v[0] = rbf(lo_bf(r1.x) + v[0]) + lo_bf(r2.x);
      v[1] = rbf(hi_bf(r1.x) + v[1]) + hi_bf(r2.x);
      v[2] = rbf(lo_bf(r1.y) + v[2]) + lo_bf(r2.y);
      v[3] = rbf(hi_bf(r1.y) + v[3]) + hi_bf(r2.y);
    }
    *reinterpret_cast<uint2*>(a.out + (size_t)b * a.ldo + r0) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
  } else if (EPI == EPI_PHI_IN) {
    if (r0 >= a.N) return;
    const uint2 bv = PRE ? p.bv : *reinterpret_cast<const uint2*>(a.bias + r0);
    float v[4] = {rbf(acc[0] + lo_bf(bv.x)), rbf(acc[1] + hi_bf(bv.x)), rbf(acc[2] + lo_bf(bv.y)),
                  rbf(acc[3] + hi_bf(bv.y))};
    const int grow = a.row0 + b;
    bf16_t* o;
    if (r0 >= a.split_n) {
      new_gelu(v);
      o = a.out2 + (size_t)grow * a.ldo2 + (r0 - a.split_n);
    } else {
      const int dm = a.split_n / 3;
      if (r0 < dm) {
        o = a.out + (size_t)grow * a.ldo + r0;
      } else {
        const int seq = grow / a.S;
        const int pos = (a.pos_dev ? *a.pos_dev : a.pos) + (grow - seq * a.S);
        if (pos < 0 || pos >= a.Tmax) return;
        const bool isk = r0 < 2 * dm;
        o = (isk ? a.kcache : a.vcache) + ((size_t)seq * a.Tmax + pos) * dm + (r0 - (isk ? dm : 2 * dm));
      }
    }
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
  } else if (EPI == EPI_SWIGLU) {
    // rows: gate f, gate f+1, up f, up f+1 with f = 8*strip + 2*g; N = hidden width F
    const int f = strip * 8 + 2 * g;
    const float s0 = rbf(silu_f(y0)), s1 = rbf(silu_f(y1));
    bf16_t* o = a.out + (size_t)b * a.ldo + f;
    if (f + 1 < a.N && ((a.ldo & 1) == 0)) {
      *reinterpret_cast<uint32_t*>(o) = pack_bf(s0 * y2, s1 * y3);
    } else {
      if (f < a.N) o[0] = f2bf(s0 * y2);
      if (f + 1 < a.N) o[1] = f2bf(s1 * y3);
    }
  } else {  // EPI_ROPE: rows [q (H*Dh); k (Hkv*Dh); v (Hkv*Dh)], one position per sequence
    const int grow = a.row0 + b;
    const int seq = a.rows ? a.rows[a.nrows + grow] : grow / a.S;
    const int pos = PRE ? p.pos : a.rows ? a.rows[grow] : (a.pos_dev ? a.pos_dev[(size_t)seq * a.pos_stride] : a.pos) + (grow - seq * a.S);
    const int nq = a.H * a.Dh, nk = a.Hkv * a.Dh;
    if (r0 >= nq + 2 * nk || pos < 0 || pos >= a.Tmax) return;
    float v[4] = {y0, y1, y2, y3};
    bf16_t* o;
    if (r0 < nq + nk) {
      const int d = (r0 < nq ? r0 : r0 - nq) % a.Dh;
      const bf16_t* cs = a.cos + (size_t)pos * (a.Dh >> 1) + (d >> 1);
      const bf16_t* sn = a.sin + (size_t)pos * (a.Dh >> 1) + (d >> 1);
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) {
        const float c = PRE ? (pr ? hi_bf(p.c) : lo_bf(p.c)) : bf2f(cs[pr]), s = PRE ? (pr ? hi_bf(p.s) : lo_bf(p.s)) : bf2f(sn[pr]);
        const float e = v[2 * pr], od = v[2 * pr + 1];
        // separate fp32 multiplies and add/sub, as the reference's eager ops round
        v[2 * pr] = __fsub_rn(__fmul_rn(e, c), __fmul_rn(od, s));
        v[2 * pr + 1] = __fadd_rn(__fmul_rn(e, s), __fmul_rn(od, c));
      }
      if (r0 < nq) {
        o = a.out + (size_t)grow * a.ldo + r0;
      } else {
        o = a.stage ? a.kcache + (size_t)grow * nk + (r0 - nq)
                    : a.kcache + (((size_t)seq * a.Tmax + pos) * a.Hkv) * a.Dh + (r0 - nq);
      }
    } else {
      o = a.stage ? a.vcache + (size_t)grow * nk + (r0 - nq - nk)
                  : a.vcache + (((size_t)seq * a.Tmax + pos) * a.Hkv) * a.Dh + (r0 - nq - nk);
    }
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
  }
}

}  // namespace
