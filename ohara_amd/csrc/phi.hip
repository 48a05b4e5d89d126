// Phi's side of the KV-cache decode path (ohara/models/phi.py): what differs from Llama.
//   LayerNorm with bias                     phi.py:132, :160 (nn.LayerNorm: fp32 statistics, one rounding)
//   append of the UN-rotated key / value    phi.py:95 (kv_cache.py:104-105)
//   attention in fp32 with the partial half-split rotation applied after the cache read
//                                           phi.py:98-117, rotary.py:131-184
// The projections with bias, new_gelu and the parallel-block sum are epilogues of the skinny
// GEMM (gemm_epilogue.h).
#include "mfma_frag.h"
#include "phi_attn.h"

#include <type_traits>

namespace {

// ---- LayerNorm: one workgroup per row ---------------------------------------------------
// What bounds it: round trips, of few rows, one after the other.  So the row, the weight and the bias are asked for together and stay in
// registers, C eighths a thread (C 0: any width, the row
// read three times).  us, before / now: 1 x 2560 2.9 / 2.5, 700 x 2560 4.7 / 4.3, 4096 x 2560 15.1 / 12.0, 4096 x 4096 19.5 / 16.0.
template <int C>
__global__ __launch_bounds__(256) void layernorm_kernel(const bf16_t* x, int ldx, const bf16_t* w, const bf16_t* b,
                                                        bf16_t* out, int ldo, int d, float eps) {
  __shared__ float red[2][4];
  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bf16_t* xr = x + (size_t)row * ldx;
  uint4 xv[C ? C : 1], wv[C ? C : 1], bv[C ? C : 1];
#pragma unroll
  for (int c = 0; c < C; ++c) xv[c] = ldg16(xr + min((tid + 256 * c) * 8, d - 8));
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int k = min((tid + 256 * c) * 8, d - 8);
    wv[c] = ldg16(w + k);
    bv[c] = ldg16(b + k);
  }
  if (C) __builtin_amdgcn_sched_barrier(0);
  auto each = [&](auto f) {  // f(column, the row's eight, weight, bias)
    if (C) {
#pragma unroll
      for (int c = 0; c < C; ++c)
        if ((tid + 256 * c) * 8 < d) f((tid + 256 * c) * 8, xv[c], [&] { return wv[c]; }, [&] { return bv[c]; });
    } else {
      for (int k = tid * 8; k < d; k += 256 * 8) f(k, ldg16(xr + k), [&] { return ldg16(w + k); }, [&] { return ldg16(b + k); });
    }
  };
  // pass 1: mean
  float s = 0.f;
  each([&](int, uint4 v, auto, auto) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) s += lo_bf(u[i]) + hi_bf(u[i]);
  });
  s = wave_sum(s);
  if (lane == 0) red[0][wave] = s;
  __syncthreads();
  const float mean = (((red[0][0] + red[0][1]) + red[0][2]) + red[0][3]) / (float)d;
  // pass 2: biased variance around the mean
  float q = 0.f;
  each([&](int, uint4 v, auto, auto) {
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float a0 = lo_bf(u[i]) - mean, a1 = hi_bf(u[i]) - mean;
      q += a0 * a0 + a1 * a1;
    }
  });
  q = wave_sum(q);
  if (lane == 0) red[1][wave] = q;
  __syncthreads();
  const float var = (((red[1][0] + red[1][1]) + red[1][2]) + red[1][3]) / (float)d;
  const float rstd = 1.0f / sqrtf(var + eps);
  each([&](int k, uint4 v, auto weight, auto bias) {
    const uint4 g = weight(), c = bias();
    const uint32_t u[4] = {v.x, v.y, v.z, v.w}, gu[4] = {g.x, g.y, g.z, g.w}, cu[4] = {c.x, c.y, c.z, c.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = pack_bf((lo_bf(u[i]) - mean) * rstd * lo_bf(gu[i]) + lo_bf(cu[i]),
                     (hi_bf(u[i]) - mean) * rstd * hi_bf(gu[i]) + hi_bf(cu[i]));
    *reinterpret_cast<uint4*>(out + (size_t)row * ldo + k) = make_uint4(o[0], o[1], o[2], o[3]);
  });
}

// ---- append: rows (seq, s) of k and v -> cache position pos + s ------------------------------
__global__ void kv_append_kernel(const bf16_t* k, const bf16_t* v, int ld, int rows, int S, int hd, int t_max, int pos,
                                 const int32_t* pos_dev, bf16_t* kc, bf16_t* vc) {
  const int n8 = hd >> 3;
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= rows * n8) return;
  const int row = idx / n8, c = (idx - row * n8) * 8;
  const int seq = row / S, t = (pos_dev ? *pos_dev : pos) + (row - seq * S);
  if (t < 0 || t >= t_max) return;
  const size_t dst = ((size_t)seq * t_max + t) * hd + c;
  *reinterpret_cast<uint4*>(kc + dst) = ldg16(k + (size_t)row * ld + c);
  *reinterpret_cast<uint4*>(vc + dst) = ldg16(v + (size_t)row * ld + c);
}

template <bool EIGHTS>
__global__ __launch_bounds__(256, 4) void phi_attn_kernel(PhiAttnArgs a) {
  phi_attend<1, EIGHTS>(a, blockIdx.x);
}

// ---- attention over many new tokens (prefill) -----------------------------------------------
// phi.py:103-104: the pair (i, i + half) of a row, `up` the partner's place; which of a sum's two products is rounded first is fixed, for queries
// and for keys.
__device__ __forceinline__ float turned_first(float x, float up, float co, float sn) { return __builtin_fmaf(x, co, -__fmul_rn(up, sn)); }
__device__ __forceinline__ float turned_query(float x, float down, float co, float sn) { return __builtin_fmaf(x, co, __fmul_rn(down, sn)); }
__device__ __forceinline__ float turned_key(float x, float down, float co, float sn) { return __builtin_fmaf(down, sn, __fmul_rn(x, co)); }

// The queries q0 + m of a wave with a bit in `which`, whose sums are not finite: an infinite key's terms meet zeros in the kernel below, a masked value's
// infinity a weight of zero.  So both products are fp32 ones here, of sixteen positions at a time, which the lanes that multiply them read themselves, and of
// positions that some of the queries do not see a query takes its own only.  It is the launch's last part, a wave's chain of round trips and products.  us, finite
// / a NaN key in all heads, where each such query walked by itself, a position at a time / so: 32 heads of 80, 100 tokens 10 / 856 / 28, 700 23 / 6600 / 104, 2000
// 110 / 24800 / 469; 16 of 128, all rotated, 700 43 / 6730 / 173.
template <int D, int NR>
__device__ __forceinline__ void phi_walk_rows(const PhiAttnArgs& a, int seq, int h, int q0, unsigned int which, int lane) {
  constexpr int NC = (D + 31) / 32, DT = D / 16;
  asm volatile("" : "+v"(lane));  // (computed anew: the caller's offsets would stay in registers through its loop)
  const int l16 = lane & 15, g = lane >> 4, half = a.rot >> 1;
  const int sq = min(q0 + l16, a.S - 1), pq = a.pos + sq, last = a.pos + min(q0 + 31 - __clz(which), a.S - 1);
  const size_t hd = (size_t)a.H * D, at0 = (size_t)seq * a.t_max * hd + (size_t)h * D;
  // features 32 c + 8 g and on of a row; zeros past the head
  struct Eighth {
    uint4 x, o, c0, c1, s0, s1;
  };
  auto ask = [&](const bf16_t* row, int position, int c) {
    const int f = 32 * c + 8 * g;
    Eighth e;
    e.x = ldg16(row + min(f, D - 8));
    if (c < NR) {
      const int partner = f < half ? f + half : f < a.rot ? f - half : 0;
      const size_t at = (size_t)position * half + (f < half ? f : f < a.rot ? f - half : 0);
      e.o = ldg16(row + partner);
      e.c0 = ldg16(a.cos + at);
      e.c1 = ldg16(a.cos + at + 4);
      e.s0 = ldg16(a.sin + at);
      e.s1 = ldg16(a.sin + at + 4);
    }
    return e;
  };
  auto turn = [&](const Eighth& e, int c, bool query, float (&v)[8]) {
    const int f = 32 * c + 8 * g;
    const uint32_t xw[4] = {e.x.x, e.x.y, e.x.z, e.x.w};
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = f >= D ? 0.f : u & 1 ? hi_bf(xw[u / 2]) : lo_bf(xw[u / 2]);
    if (c >= NR) return;
    const uint32_t ow[4] = {e.o.x, e.o.y, e.o.z, e.o.w};
    const uint32_t cw[8] = {e.c0.x, e.c0.y, e.c0.z, e.c0.w, e.c1.x, e.c1.y, e.c1.z, e.c1.w}, sw[8] = {e.s0.x, e.s0.y, e.s0.z, e.s0.w, e.s1.x, e.s1.y, e.s1.z, e.s1.w};
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float z = u & 1 ? hi_bf(ow[u / 2]) : lo_bf(ow[u / 2]), co = __uint_as_float(cw[u]), sn = __uint_as_float(sw[u]);
      v[u] = f < half ? turned_first(v[u], z, co, sn) : f < a.rot ? (query ? turned_query(v[u], z, co, sn) : turned_key(v[u], z, co, sn)) : v[u];
    }
  };
  float q[NC][8], m = PHI_LOWEST, l = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) turn(ask(a.q + ((size_t)seq * a.S + sq) * a.ldq + h * D, pq, c), c, true, q[c]);
  const float mul = sqrtf(1.0f / (float)D) * OHARA_LOG2E;
  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int t0 = 0; t0 <= last; t0 += 16) {
    f32x4 s = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int t = min(t0 + l16, last);
    Eighth key[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) key[c] = ask(a.kc + at0 + (size_t)t * hd, t, c);
    const bool whole = t0 + 15 <= a.pos + q0;  // (uniform) every query sees all of it
    bf16_t v[4][DT];                           // of position t0 + 4 g + i, feature 16 t + l16
    if (whole) {
      const bf16_t* row = a.vc + at0 + (size_t)(t0 + 4 * g) * hd + l16;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < DT; ++t) v[i][t] = row[i * hd + 16 * t];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float k[8];
      turn(key[c], c, false, k);
      s = mma_f(k, q[c], s);
    }
    float p[4], mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (t0 + 4 * g + r > pq) s[r] = -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = lane_xor_max<32>(lane_xor_max<16>(mx));
    const float mn = fmaxf(m, ceilf(mx * mul)), corr = pow2_neg_int(m - mn);
    m = mn;
    l *= corr;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], mul, -mn));
      l += p[r];
    }
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) o[t][r] *= corr;
    if (whole) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(bf2f(v[i][t]), p[i], o[t], 0, 0, 0);
      continue;
    }
#pragma unroll 1
    for (int j0 = 0; j0 < 16; j0 += 4)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float w = __shfl(p[r], j0 * 4 + l16);
        const bool in = t0 + j0 + r <= pq;
        const bf16_t* row = a.vc + at0 + (size_t)min(t0 + j0 + r, last) * hd + 4 * g;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
          const uint2 x = in ? ldg8(row + 16 * t) : make_uint2(0, 0);
          o[t][0] = __builtin_fmaf(w, lo_bf(x.x), o[t][0]);
          o[t][1] = __builtin_fmaf(w, hi_bf(x.x), o[t][1]);
          o[t][2] = __builtin_fmaf(w, lo_bf(x.y), o[t][2]);
          o[t][3] = __builtin_fmaf(w, hi_bf(x.y), o[t][3]);
        }
      }
  }
  l = lane_xor_sum<32>(lane_xor_sum<16>(l));
  if (q0 + l16 >= a.S || !(which >> l16 & 1)) return;
  const float inv = 1.0f / l;
  bf16_t* row = a.out + ((size_t)seq * a.S + sq) * hd + (size_t)h * D + 4 * g;
#pragma unroll
  for (int t = 0; t < DT; ++t) *reinterpret_cast<uint2*>(row + 16 * t) = make_uint2(pack_bf(o[t][0] * inv, o[t][1] * inv), pack_bf(o[t][2] * inv, o[t][3] * inv));
}

// One workgroup per (sequence, head, 64 queries); each of its four waves owns 16 queries.  Keys and values go through LDS in tiles of 64 positions.
// The reference computes in fp32 (phi.py:98-117): rotated features and weights are fp32 numbers, cached values and features that are not rotated
// bf16 ones.  The first are taken apart into three bf16 terms (mfma_frag.h; keys as a tile is put into LDS), and both products are
// v_mfma_f32_16x16x32_bf16 with fp32 sums: six of the nine products of terms for rotated features (what the other three add lies 2^-27 below), one for
// the rest, three for weights times values - exact but for the sums.  At head width 80, 32 features rotated, a block of 16 queries x 16 positions is
// 15.5 such products of 16 cycles, where the fp32 instruction (v_mfma_f32_16x16x4_f32) took 40 of 32.  Both products are formed transposed,
//   S^T (position x query) = K . Q^T        O^T (feature x query) = V^T . P^T,
// as in attention_prefill.hip: a lane's scores belong to one query, and are the B operand of the second product where they stand; its A operand is read
// from rows of values by ds_read_b64_tr_b16.
//
// What bounds it: where workgroups have a CU to themselves the longest one's chain of tiles, 2.2 us each, in which products, softmax, the weights' terms and
// the next tile's keys take turns (putting those among the products changed nothing); where two share it the vector unit, on which the last three
// are twice the products' cycles.  32 heads of 80, us with fp32 products and tiles of 32 / so: 100 tokens 14.7 / 9.6, 300 30 / 15.5, 700 68 / 28, 1500
// 157 / 60, 2040 281 / 98; 2 x 700 76 / 33, 4 x 1500 580 / 213; 64 behind 1000 93 / 37.  Results that differ from the rounded ones of 64 bits: 700 tokens
// 0.030 / 0.019 %, 2040 0.044 / 0.029 %.
// TEAMS = 2: two such fours of waves with tiles of their own take turns along the positions, and add up at the end (phi_teams).
template <int DT, int NR>  // head width / 16; chunks of 32 features with rotated ones among them
struct PhiTile {
  static constexpr int D = 16 * DT, NC = (D + 31) / 32;
  // A key's row: the first terms of the first NR chunks, their second, their third ones, then the other chunks; an odd number of
  // 16-byte pieces, as sixteen rows' reads want it.  A value's row: an odd number of 32 bytes.
  static constexpr int PLANE = 64 * NR, KROW = 16 * ((4 * NC + 8 * NR) | 1), VROW = 32 * (DT | 1);
  // positions: 64 where two workgroups with two tiles each share a CU's LDS (2 x 700 tokens, heads of 128, all rotated: 64 145 us, 32 60)
  static constexpr int T = 4 * 64 * (KROW + VROW) <= 160 * 1024 ? 64 : 32, BUF = T * (KROW + VROW);
  static __device__ __forceinline__ constexpr int byte_of(int feature) { return 2 * feature + (feature < 32 * NR ? 0 : 2 * PLANE); }
};
template <int DT, int NR, int TEAMS>
__global__ __launch_bounds__(256 * TEAMS, 2) void phi_attn_prefill_kernel(PhiAttnArgs a, int nqb, int heads) {
  typedef PhiTile<DT, NR> L;
  constexpr int D = L::D, NC = L::NC, T = L::T, QB = 64;
  // a thread's parts of a tile: fours of rotated pairs, eighths of the other features, of values
  constexpr int NP = (NR * T + 63) / 64, CE = 2 * DT - 4 * NR + 2, NU = CE > 0 ? (CE * T + 255) / 256 : 1, NV = (2 * DT * T + 255) / 256;
  extern __shared__ __align__(16) unsigned char all[];  // two tiles a team
  const int team = TEAMS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = TEAMS == 1 ? threadIdx.x : threadIdx.x & 255;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  unsigned char* const smem = all + team * 2 * L::BUF;
  const int l16 = lane & 15, g = lane >> 4;
  const int half = a.rot >> 1;
  // an XCD (ids go round-robin over the eight) gets every eighth head; long contexts first
  const int x8 = blockIdx.x & 7, q8 = blockIdx.x >> 3, nh = (heads + 7) >> 3;
  const int head = (q8 % nh) * 8 + x8;
  if (head >= heads) return;
  const int seq = head / a.H, h = head - seq * a.H;
  const int s0 = (nqb - 1 - q8 / nh) * QB;
  const size_t hd = (size_t)a.H * D;
  const int pos0 = a.pos, wq0 = s0 + 16 * wave;
  const int t_end = pos0 + min(s0 + QB - 1, a.S - 1);
  const bf16_t* kb = a.kc + (size_t)seq * a.t_max * hd + (size_t)h * D;
  const bf16_t* vb = a.vc + (size_t)seq * a.t_max * hd + (size_t)h * D;

  // This thread's part of a tile, asked for a tile ahead: four pairs of rotated features (NP times), eighths of rows of the others and of values.
  const int quads = half >> 2, eighths = (D - a.rot) >> 3, first = a.rot >> 3;
  int rp[NP], rf[NP], up[NU], uc[NU];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int idx = tid + 256 * i;
    rp[i] = idx / quads;
    rf[i] = 4 * (idx - rp[i] * quads);
  }
#pragma unroll
  for (int i = 0; i < NU; ++i) {
    const int idx = tid + 256 * i;
    up[i] = eighths ? idx / eighths : T;
    uc[i] = eighths ? 8 * (first + idx - up[i] * eighths) : 0;
  }
  uint2 k1[NP], k2[NP];
  uint4 ca[NP], sa[NP], ku[NU], vv[NV];
  auto fetch = [&](int t0) {  // (past the last position: that one's, masked)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int t = min(t0 + min(rp[i], T - 1), t_end);
      const bf16_t* row = kb + (size_t)t * hd + rf[i];
      k1[i] = ldg8(row);
      k2[i] = ldg8(row + half);
      ca[i] = ldg16(a.cos + (size_t)t * half + rf[i]);
      sa[i] = ldg16(a.sin + (size_t)t * half + rf[i]);
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) ku[i] = ldg16(kb + (size_t)min(t0 + min(up[i], T - 1), t_end) * hd + uc[i]);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = min(tid + 256 * i, T * 2 * DT - 1), p = idx / (2 * DT);
      vv[i] = ldg16(vb + (size_t)min(t0 + p, t_end) * hd + 8 * (idx - p * 2 * DT));
    }
  };
  auto put = [&](unsigned char* tile) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (rp[i] >= T) continue;
      const float x[4] = {lo_bf(k1[i].x), hi_bf(k1[i].x), lo_bf(k1[i].y), hi_bf(k1[i].y)};
      const float y[4] = {lo_bf(k2[i].x), hi_bf(k2[i].x), lo_bf(k2[i].y), hi_bf(k2[i].y)};
      const uint32_t cw[4] = {ca[i].x, ca[i].y, ca[i].z, ca[i].w}, sw[4] = {sa[i].x, sa[i].y, sa[i].z, sa[i].w};
      float lo[4], hi[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float co = __uint_as_float(cw[u]), sn = __uint_as_float(sw[u]);
        lo[u] = turned_first(x[u], y[u], co, sn);
        hi[u] = turned_key(y[u], x[u], co, sn);
      }
      bf16_t* at = reinterpret_cast<bf16_t*>(tile + rp[i] * L::KROW) + rf[i];
      WideLds<bf16_t>::put4(at, L::PLANE / 2, lo);
      WideLds<bf16_t>::put4(at + half, L::PLANE / 2, hi);
    }
#pragma unroll
    for (int i = 0; i < NU; ++i)
      if (up[i] < T) *reinterpret_cast<uint4*>(tile + up[i] * L::KROW + L::byte_of(uc[i])) = ku[i];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + 256 * i, p = idx / (2 * DT);
      if (idx < T * 2 * DT) *reinterpret_cast<uint4*>(tile + T * L::KROW + p * L::VROW + 16 * (idx - p * 2 * DT)) = vv[i];
    }
  };

  // This lane's query (those beyond the call's tokens repeat the last one and are not stored), eighths g of its chunks.
  const int sq = min(wq0 + l16, a.S - 1), pq = pos0 + sq;
  Wide<bf16_t> qw[NR];
  uint4 qf[NC > NR ? NC - NR : 1];
  {
    const bf16_t* row = a.q + ((size_t)seq * a.S + sq) * a.ldq + h * D;
    uint4 x[NC], o[NR], c0[NR], c1[NR], n0[NR], n1[NR];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int f = 32 * c + 8 * g;
      x[c] = ldg16(row + min(f, D - 8));
      if (c < NR) {
        const bool rotated = f < a.rot, low = f < half;
        const size_t at = (size_t)pq * half + (rotated ? (low ? f : f - half) : 0);
        o[c] = ldg16(row + (rotated ? (low ? f + half : f - half) : 0));
        c0[c] = ldg16(a.cos + at);
        c1[c] = ldg16(a.cos + at + 4);
        n0[c] = ldg16(a.sin + at);
        n1[c] = ldg16(a.sin + at + 4);
      }
    }
    fetch(team * T);
    // what no tile's part is put on: features past the head, second and third terms of those that are not rotated
    for (int i = tid; i < 2 * T * (L::KROW / 16); i += 256) {
      const int r = i / (L::KROW / 16);
      *reinterpret_cast<uint4*>(smem + (r / T) * L::BUF + (r % T) * L::KROW + 16 * (i - r * (L::KROW / 16))) = make_uint4(0, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int f = 32 * c + 8 * g;
      const uint32_t xw[4] = {x[c].x, x[c].y, x[c].z, x[c].w};
      if (c < NR) {
        const uint32_t ow[4] = {o[c].x, o[c].y, o[c].z, o[c].w};
        const uint32_t cw[8] = {c0[c].x, c0[c].y, c0[c].z, c0[c].w, c1[c].x, c1[c].y, c1[c].z, c1[c].w};
        const uint32_t sw[8] = {n0[c].x, n0[c].y, n0[c].z, n0[c].w, n1[c].x, n1[c].y, n1[c].z, n1[c].w};
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const float y = u & 1 ? hi_bf(xw[u / 2]) : lo_bf(xw[u / 2]), z = u & 1 ? hi_bf(ow[u / 2]) : lo_bf(ow[u / 2]);
          const float co = __uint_as_float(cw[u]), sn = __uint_as_float(sw[u]);
          v[u] = f < half ? turned_first(y, z, co, sn) : f < a.rot ? turned_query(y, z, co, sn) : f < D ? y : 0.f;
        }
        wide_from(qw[c], v);
      } else {
        qf[c - NR] = f < D ? x[c] : make_uint4(0, 0, 0, 0);
      }
    }
  }
  __syncthreads();
  put(smem);
  __syncthreads();

  const int wave_hi = pos0 + min(wq0 + 15, a.S - 1);  // last position any query of the wave sees
  const float mul = sqrtf(1.0f / (float)D) * OHARA_LOG2E;
  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;
  const uint32_t kat = l16 * L::KROW + g * 16;                                      // keys of positions 16 b + l16
  const uint32_t vat = T * L::KROW + (4 * g + (l16 >> 2)) * L::VROW + (l16 & 3) * 8;  // values, as ds_read_b64_tr_b16 takes them
  auto window = [&](auto count, int t0, uint32_t kat, uint32_t vat) {  // 32 positions of a tile, or all of it
    constexpr int NW = decltype(count)::value, NB = 2 * NW;
    uint4 kf[NB][NC + 2 * NR];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int c = 0; c < NC + 2 * NR; ++c) kf[b][c] = lds16_at(kat + b * (16 * L::KROW) + c * 64);
    __builtin_amdgcn_sched_barrier(0);
    f32x4 s[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) s[b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto add = [&](int piece, uint4 q) {
#pragma unroll
      for (int b = 0; b < NB; ++b) s[b] = mma_bf(kf[b][piece], q, s[b]);
    };
#pragma unroll
    for (int c = 0; c < NR; ++c) {
      add(2 * NR + c, qw[c].t[0]);
      add(NR + c, qw[c].t[1]);
      add(c, qw[c].t[2]);
      add(NR + c, qw[c].t[0]);
      add(c, qw[c].t[1]);
    }
#pragma unroll
    for (int c = 0; c < NR; ++c) add(c, qw[c].t[0]);
#pragma unroll
    for (int c = NR; c < NC; ++c) add(2 * NR + c, qf[c - NR]);
    __builtin_amdgcn_sched_barrier(0);
    if (t0 + 16 * NB - 1 > pos0 + wq0) {  // (uniform) not every query of the wave sees all of it
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (t0 + 16 * b + 4 * g + r > pq) s[b][r] = -INFINITY;
    }
    float mx = s[0][0];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[b][r]);
    mx = lane_xor_max<32>(lane_xor_max<16>(mx));
    const float mn = fmaxf(m, ceilf(mx * mul));  // a whole number: what is rescaled is rescaled exactly, and seldom
    const float corr = pow2_neg_int(m - mn), off = mn == -INFINITY ? 0.f : mn;
    m = mn;
    Wide<bf16_t> pf[NW];
    float ps = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      float p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        p[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[2 * w + i / 4][i % 4], mul, -off));
        ps += p[i];
      }
      wide_from(pf[w], p);
    }
    lsum = lsum * corr + ps;
    if (__any(corr != 1.0f)) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[t][r] *= corr;
    }
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      uint4 vf[DT];
#pragma unroll
      for (int t = 0; t < DT; ++t) {
        const uint32_t at = vat + w * (32 * L::VROW) + t * 32;
        const uint2 lo = lds_tr8(at), hi = lds_tr8(at + 16 * L::VROW);
        vf[t] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 2; i >= 0; --i)
#pragma unroll
        for (int t = 0; t < DT; ++t) o[t] = mma_bf(vf[t], pf[w].t[i], o[t]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  constexpr bool BOTH = T == 64 && NC + 2 * NR <= 5;  // (more fragments than that do not fit)
  uint32_t cur = 0;
  for (int round = 0; round <= t_end; round += TEAMS * T) {  // (the last round may have no tile for the second team)
    const int t0 = round + team * T, next = t0 + TEAMS * T;
    const bool more = next <= t_end;
    if (more) fetch(next);  // in flight during this tile's products
    const uint32_t kt = lds0 + cur + kat, vt = lds0 + cur + vat;
    if (BOTH && t0 + 32 <= wave_hi) {
      window(std::integral_constant<int, 2>(), t0, kt, vt);
    } else {
      if (t0 <= wave_hi) window(std::integral_constant<int, 1>(), t0, kt, vt);
      if (!BOTH && T == 64 && t0 + 32 <= wave_hi) window(std::integral_constant<int, 1>(), t0 + 32, kt + 32 * L::KROW, vt + 32 * L::VROW);
    }
    cur = L::BUF - cur;
    if (more) put(smem + cur);
    __syncthreads();
  }
  lsum = lane_xor_sum<32>(lane_xor_sum<16>(lsum));
  if constexpr (TEAMS == 2) {  // the second team's sums, weighted to the larger of the two maxima (whole numbers: exactly)
    constexpr int N = 4 * DT + 2;
    static_assert(4 * N * 64 * 4 <= 2 * TEAMS * L::BUF, "");
    float* there = reinterpret_cast<float*>(all) + (wave * N) * 64 + lane;
    if (team) {
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) there[(4 * t + i) * 64] = o[t][i];
      there[(N - 2) * 64] = m;
      there[(N - 1) * 64] = lsum;
    }
    __syncthreads();
    if (team) return;
    const float m2 = there[(N - 2) * 64], M = fmaxf(m, m2);
    const float w1 = pow2_neg_int(m - M), w2 = m2 == -INFINITY ? 0.f : pow2_neg_int(m2 - M);
    lsum = lsum * w1 + there[(N - 1) * 64] * w2;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) o[t][i] = o[t][i] * w1 + there[(4 * t + i) * 64] * w2;
  }
  float sum = lsum;
#pragma unroll
  for (int t = 0; t < DT; ++t) sum += (o[t][0] + o[t][1]) + (o[t][2] + o[t][3]);
  const unsigned int odd = columns_not_finite(sum);
  if (wq0 + l16 < a.S && !(odd >> l16 & 1)) {
    const float inv = 1.0f / lsum;
    bf16_t* orow = a.out + ((size_t)seq * a.S + sq) * hd + (size_t)h * D + 4 * g;
#pragma unroll
    for (int t = 0; t < DT; ++t)
      *reinterpret_cast<uint2*>(orow + 16 * t) =
          make_uint2(pack_bf(o[t][0] * inv, o[t][1] * inv), pack_bf(o[t][2] * inv, o[t][3] * inv));
  }
  if (odd) phi_walk_rows<D, NR>(a, seq, h, wq0, odd, lane);
}

// Features rotated in other numbers than eights, or tables off 16 bytes: keys and values in LDS as fp32, the keys rotated there, in tiles of 32 positions;
// both products fp32 ones.
constexpr int PF_Q = 64, PF_T = 32;
template <int DT>  // head width / 16
__global__ __launch_bounds__(256, 2) void phi_attn_pairs_kernel(PhiAttnArgs a, int nqb, int heads) {
  constexpr int D = 16 * DT, LD = D + 4, C8 = D / 8, NV = (PF_T * C8 + 255) / 256;
  constexpr int BUF = 2 * PF_T * LD;  // floats: keys | values of a tile
  extern __shared__ __align__(16) float sm[];  // two of them; the rotated queries before the loop
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int half = a.rot >> 1;
  // an XCD (ids go round-robin over the eight) gets every eighth head; long contexts first
  const int x8 = blockIdx.x & 7, q8 = blockIdx.x >> 3, nh = (heads + 7) >> 3;
  const int head = (q8 % nh) * 8 + x8;
  if (head >= heads) return;
  const int seq = head / a.H, h = head - seq * a.H;
  const int s0 = (nqb - 1 - q8 / nh) * PF_Q;
  const size_t hd = (size_t)a.H * D;
  const int pos0 = a.pos;

  auto widen = [](uint4 v, float (&f)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = lo_bf(w[i]);
      f[2 * i + 1] = hi_bf(w[i]);
    }
  };
  auto put8 = [](float* dst, const float (&f)[8], bool in) {
    *reinterpret_cast<float4*>(dst) = in ? make_float4(f[0], f[1], f[2], f[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    *reinterpret_cast<float4*>(dst + 4) = in ? make_float4(f[4], f[5], f[6], f[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
  };

  // rotated queries -> LDS -> registers (rows beyond the call's tokens are zero)
  for (int idx = tid; idx < PF_Q * D; idx += 256) {
    const int qi = idx / D, j = idx - qi * D;
    const int sq = s0 + qi;
    float v = 0.f;
    if (sq < a.S) {
      const bf16_t* qrow = a.q + ((size_t)seq * a.S + sq) * a.ldq + h * D;
      const size_t cb = (size_t)(pos0 + sq) * half;
      v = bf2f(qrow[j]);
      if (j < half) v = v * a.cos[cb + j] - bf2f(qrow[j + half]) * a.sin[cb + j];
      else if (j < a.rot) v = bf2f(qrow[j - half]) * a.sin[cb + j - half] + v * a.cos[cb + j - half];
    }
    sm[qi * LD + j] = v;
  }
  __syncthreads();
  float qreg[D / 4];
#pragma unroll
  for (int kk = 0; kk < D / 4; ++kk) qreg[kk] = sm[(16 * wave + l16) * LD + 4 * kk + g];
  __syncthreads();

  // this lane's query column; columns beyond the call's tokens repeat the last one and are not stored
  const int sq = min(s0 + 16 * wave + l16, a.S - 1);
  const int pq = pos0 + sq;
  const int wave_hi = pos0 + min(s0 + 16 * wave + 15, a.S - 1);  // last position any query of the wave sees
  const int t_end = pos0 + min(s0 + PF_Q - 1, a.S - 1);
  const float scale = sqrtf(1.0f / (float)D);
  const bf16_t* kb = a.kc + (size_t)seq * a.t_max * hd + (size_t)h * D;
  const bf16_t* vb = a.vc + (size_t)seq * a.t_max * hd + (size_t)h * D;

  f32x4 o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, lsum = 0.f;

  // this thread's eighths of a tile's rows
  uint4 kr[NV], vr[NV];
  auto place = [&](int i, int& p, int& c) {
    const int idx = tid + 256 * i;
    p = idx / C8;
    c = idx - p * C8;
  };
  auto fetch = [&](int t0) {  // (rows past the last position: that one's, put as zeros)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      int p, c;
      place(i, p, c);
      const int t = min(t0 + min(p, PF_T - 1), t_end);
      kr[i] = ldg16(kb + (size_t)t * hd + 8 * c);
      vr[i] = ldg16(vb + (size_t)t * hd + 8 * c);
    }
  };
  auto put = [&](int t0, float* ks) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      int p, c;
      place(i, p, c);
      if (p >= PF_T) continue;
      float k[8], v[8];
      widen(kr[i], k);
      widen(vr[i], v);
      put8(ks + p * LD + 8 * c, k, t0 + p <= t_end);
      put8(ks + PF_T * LD + p * LD + 8 * c, v, t0 + p <= t_end);
    }
  };

  fetch(0);
  put(0, sm);
  __syncthreads();
  float* ks = sm;
  for (int t0 = 0; t0 <= t_end; t0 += PF_T) {
    const bool more = t0 + PF_T <= t_end;
    if (more) fetch(t0 + PF_T);  // in flight during this tile's products
    // rotate the tile's keys in place: pair (i, i + half) of every position
    for (int idx = tid; idx < PF_T * half; idx += 256) {
      const int p = idx / half, i = idx - p * half;
      if (t0 + p <= t_end) {
        const float c = a.cos[(size_t)(t0 + p) * half + i], sn = a.sin[(size_t)(t0 + p) * half + i];
        const float k1 = ks[p * LD + i], k2 = ks[p * LD + i + half];
        ks[p * LD + i] = k1 * c - k2 * sn;
        ks[p * LD + i + half] = k1 * sn + k2 * c;
      }
    }
    __syncthreads();
    const float* vs = ks + PF_T * LD;
    if (t0 <= wave_hi) {  // (wave-uniform: else nothing of the tile is visible to the wave's queries)
      // operands are read together before the products (left to itself, the compiler waits for each), and the two blocks' chains of
      // products take turns
      float kf[2][D / 4];
#pragma unroll
      for (int blk = 0; blk < 2; ++blk)
#pragma unroll
        for (int kk = 0; kk < D / 4; ++kk) kf[blk][kk] = ks[(16 * blk + l16) * LD + g + 4 * kk];
      __builtin_amdgcn_sched_barrier(0);
      f32x4 s2[2] = {(f32x4){0.f, 0.f, 0.f, 0.f}, (f32x4){0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int kk = 0; kk < D / 4; ++kk)
#pragma unroll
        for (int blk = 0; blk < 2; ++blk) s2[blk] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[blk][kk], qreg[kk], s2[blk], 0, 0, 0);
#pragma unroll
      for (int blk = 0; blk < 2; ++blk) {
        const int tb = t0 + 16 * blk;
        if (tb > wave_hi) break;
        float vf[4][DT];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int t = 0; t < DT; ++t) vf[kk][t] = vs[(16 * blk + 4 * g + kk) * LD + l16 + 16 * t];
        __builtin_amdgcn_sched_barrier(0);
        f32x4 sc = s2[blk];
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[r] = tb + 4 * g + r <= pq ? sc[r] * scale : -INFINITY;
          mx = fmaxf(mx, sc[r]);
        }
        mx = lane_xor_max<32>(lane_xor_max<16>(mx));
        const float mn = fmaxf(m, mx);  // finite: position 0 is in the first block and visible to every query
        const float corr = __expf(m - mn);
        float ps = 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sc[r] = __expf(sc[r] - mn);
          ps += sc[r];
        }
        lsum = lsum * corr + ps;
        m = mn;
#pragma unroll
        for (int t = 0; t < DT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[t][r] *= corr;
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
#pragma unroll
          for (int t = 0; t < DT; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[kk][t], sc[kk], o[t], 0, 0, 0);
      }
    }
    float* next = ks == sm ? sm + BUF : sm;
    if (more) put(t0 + PF_T, next);
    __syncthreads();
    ks = next;
  }
  lsum = lane_xor_sum<32>(lane_xor_sum<16>(lsum));
  if (s0 + 16 * wave + l16 < a.S) {
    const float inv = 1.0f / lsum;
    bf16_t* orow = a.out + ((size_t)seq * a.S + sq) * hd + (size_t)h * D + 4 * g;
#pragma unroll
    for (int t = 0; t < DT; ++t)
      *reinterpret_cast<uint2*>(orow + 16 * t) =
          make_uint2(pack_bf(o[t][0] * inv, o[t][1] * inv), pack_bf(o[t][2] * inv, o[t][3] * inv));
  }
}

// Teams of a workgroup: two where the longest chain of tiles is what the launch takes - workgroups to a CU each, or fewer tiles to a CU than
// four fifths of that chain - and has some tiles to share.  us, one / two, 32 heads of 80: 128 tokens 10.0 / 10.0, 300 15.6 / 14.2, 500 21.7 / 18.8, 700 27.6 / 23.3,
// 1500 59.8 / 71.4, 2 x 300 16.4 / 17.7, 4 x 200 14.8 / 19.8, 200 behind 500 27.7 / 23.1, 64 behind 1500 52.3 / 41.6; 24 of 128, 700 tokens 35.4 / 28.7; 16 of 64, all
// rotated, 1000 39.1 / 31.0, 16 x 16 behind 300 17.3 / 15.6; 40 of 128, 64 rotated, 500 31.6 / 27.1, 800 44.6 / 50.8.
int phi_teams(int64_t batch, int64_t S, int64_t h, int64_t pos) {
  const int64_t blocks = (S + PF_Q - 1) / PF_Q, heads = batch * h, longest = (pos + S + 63) / 64;
  const int64_t all = heads * blocks * (pos / 64) + heads * blocks * (blocks + 1) / 2;  // tiles, about
  if (longest < 4) return 1;
  return blocks * ((heads + 7) / 8 * 8) <= 256 || (longest >= 8 && 5 * all <= 4 * 256 * longest) ? 2 : 1;
}

template <int DT>
int launch_phi_prefill(const PhiAttnArgs& a, int batch, hipStream_t st) {
  const int64_t nqb = (a.S + PF_Q - 1) / PF_Q, heads = (int64_t)a.H * batch, grid = nqb * ((heads + 7) / 8 * 8);
  if (grid > INT32_MAX) return OHARA_ESIZE;
  if (!phi_eights(a)) {
    constexpr int LDS = 2 * 2 * PF_T * (16 * DT + 4) * (int)sizeof(float);
    if (LDS > 64 * 1024) (void)hipFuncSetAttribute((const void*)phi_attn_pairs_kernel<DT>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
    hipLaunchKernelGGL(phi_attn_pairs_kernel<DT>, dim3((unsigned)grid), dim3(256), LDS, st, a, (int)nqb, (int)heads);
    return ohara_launch_status();
  }
  constexpr int NC = (DT + 1) / 2;  // a.rot is at most 16 DT
  auto of = [&](auto chunks) {
    constexpr int NR = decltype(chunks)::value < NC ? decltype(chunks)::value : NC, BUF = PhiTile<DT, NR>::BUF;
    auto by = [&](auto teams) {
      constexpr int TEAMS = decltype(teams)::value, LDS = TEAMS * 2 * BUF;
      auto kernel = phi_attn_prefill_kernel<DT, NR, TEAMS>;
      if (LDS > 64 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
      hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256 * TEAMS), LDS, st, a, (int)nqb, (int)heads);
      return ohara_launch_status();
    };
    return phi_teams(batch, a.S, a.H, a.pos) == 2 ? by(std::integral_constant<int, 2>()) : by(std::integral_constant<int, 1>());
  };
  switch ((a.rot + 31) / 32) {
    case 1: return of(std::integral_constant<int, 1>());
    case 2: return of(std::integral_constant<int, 2>());
    case 3: return of(std::integral_constant<int, 3>());
    default: return of(std::integral_constant<int, 4>());
  }
}

}  // namespace

extern "C" {

int ohara_layernorm_bf16(const uint16_t* x, int ldx, const uint16_t* weight, const uint16_t* bias, uint16_t* out, int ldo,
                         int rows, int d, float eps, void* stream) {
  if (!x || !weight || !bias || !out || rows < 1 || d < 8) return OHARA_EINVAL;
  if ((d & 7) || (ldx & 7) || (ldo & 7) || ldx < d || ldo < d) return OHARA_EINVAL;
  auto kernel = d <= 2048 ? layernorm_kernel<1> : d <= 4096 ? layernorm_kernel<2> : d <= 8192 ? layernorm_kernel<4> : layernorm_kernel<0>;
  hipLaunchKernelGGL(kernel, dim3(rows), dim3(256), 0, (hipStream_t)stream, x, ldx, weight, bias, out, ldo, d, eps);
  return ohara_launch_status();
}

int ohara_kv_append_bf16(const uint16_t* k, const uint16_t* v, int ld, int batch, int seq_len, int h, int dh, int pos,
                         const int32_t* pos_dev, uint16_t* kcache, uint16_t* vcache, int t_max, void* stream) {
  if (!k || !v || !kcache || !vcache || batch < 1 || seq_len < 1 || h < 1 || dh < 1 || t_max < 1) return OHARA_EINVAL;
  const int64_t hd = (int64_t)h * dh;
  if ((hd & 7) || (ld & 7) || ld < hd) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  if (pos_dev && seq_len != 1) return OHARA_EINVAL;
  const int64_t total = (int64_t)batch * seq_len * (hd >> 3);
  if (total > INT32_MAX) return OHARA_ESIZE;
  hipLaunchKernelGGL(kv_append_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, k, v, ld,
                     batch * seq_len, seq_len, (int)hd, t_max, pos, pos_dev, kcache, vcache);
  return ohara_launch_status();
}

int64_t ohara_phi_attn_workspace_bytes(int batch, int h, int dh, int n_split) {
  if (batch < 1 || h < 1 || dh < 1 || n_split < 1) return OHARA_EINVAL;
  const int64_t counters = (((int64_t)batch * h * (int64_t)sizeof(int)) + 255) & ~(int64_t)255;
  return counters + (int64_t)batch * h * n_split * (dh + 2) * (int64_t)sizeof(float);
}

int ohara_phi_attn_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos,
                        const float* sin, int rot, int batch, int seq_len, int h, int dh, int t_max, int pos,
                        const int32_t* pos_dev, int n_split, void* workspace, uint16_t* out, void* stream) {
  PhiAttnArgs a;
  const int rc = phi_attn_args(a, q, ldq, kcache, vcache, cos, sin, rot, batch, seq_len, h, dh, t_max, pos, pos_dev, n_split, workspace, out);
  if (rc) return rc;
  if (seq_len >= 16 && !pos_dev && (dh == 16 || dh == 32 || dh == 64 || dh == 80 || dh == 128) && h <= 65535 &&
      batch <= 65535) {
    // many new tokens: queries in tiles of 64 against key / value tiles in LDS
    switch (dh / 16) {
      case 1: return launch_phi_prefill<1>(a, batch, (hipStream_t)stream);
      case 2: return launch_phi_prefill<2>(a, batch, (hipStream_t)stream);
      case 4: return launch_phi_prefill<4>(a, batch, (hipStream_t)stream);
      case 5: return launch_phi_prefill<5>(a, batch, (hipStream_t)stream);
      default: return launch_phi_prefill<8>(a, batch, (hipStream_t)stream);
    }
  }
  hipLaunchKernelGGL(phi_eights(a) ? phi_attn_kernel<true> : phi_attn_kernel<false>, dim3((unsigned)(batch * seq_len * h * n_split)), dim3(256), 0, (hipStream_t)stream, a);
  return ohara_launch_status();
}

int ohara_phi_attn_linear_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos, const float* sin, int rot,
                               int batch, int h, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split, void* workspace, uint16_t* out,
                               const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, uint16_t* y, int ldy, void* stream) {
  PhiAttnArgs t;
  int rc = phi_attn_args(t, q, ldq, kcache, vcache, cos, sin, rot, batch, 1, h, dh, t_max, pos, pos_dev, n_split, workspace, out);
  if (rc) return rc;
  if (!x || !wp || !bias || !y || n < 1 || k < 1 || (k & 7) || (ldx & 7) || ldx < k || (n & 3) || (ldy & 3) || ldy < n) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = batch; a.N = n; a.K = k;
  a.out = y; a.ldo = ldy; a.bias = bias;
  if (ohara_launch_phi_attn_linear(t, a, (hipStream_t)stream, &rc)) return rc;
  rc = ohara_phi_attn_bf16(q, ldq, kcache, vcache, cos, sin, rot, batch, 1, h, dh, t_max, pos, pos_dev, n_split, workspace, out, stream);
  return rc ? rc : ohara_linear_bias_bf16(x, ldx, wp, n, k, bias, batch, OHARA_LIN_BIAS, nullptr, 0, nullptr, 0, y, ldy, stream);
}

int ohara_phi_attn_out_bf16(const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos, const float* sin, int rot,
                            int batch, int h, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split, void* workspace, const uint16_t* x, int ldx,
                            const uint16_t* wp, int n, int k, const uint16_t* bias, uint16_t* y, int ldy, const uint16_t* wp_out, const uint16_t* bias_out,
                            const uint16_t* add, int ld_add, uint16_t* out, int ldo, void* stream) {
  PhiAttnArgs t;
  const int rc = phi_attn_args(t, q, ldq, kcache, vcache, cos, sin, rot, batch, 1, h, dh, t_max, pos, pos_dev, n_split, workspace, out);
  if (rc) return rc;
  if (!x || !wp || !bias || !y || n < 1 || k < 1 || (k & 7) || (ldx & 7) || ldx < k || (n & 3) || (ldy & 3) || ldy < n) return OHARA_EINVAL;
  if (!wp_out || !bias_out || !add || (ld_add & 3) || ld_add < n || (ldo & 3) || ldo < n || !workspace || ((uintptr_t)workspace & 15)) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = batch; a.N = n; a.K = k;
  a.out = y; a.ldo = ldy; a.bias = bias;
  GemmArgs o{};
  o.wp = reinterpret_cast<const uint4*>(wp_out);
  o.B = batch; o.N = n; o.K = h * dh;
  o.out = out; o.ldo = ldo; o.bias = bias_out;
  o.resid = y; o.ldr = ldy; o.resid2 = add; o.ldr2 = ld_add;
  return ohara_launch_phi_attn_out(t, a, o, (hipStream_t)stream);
}

int ohara_phi_prefill_teams(int batch, int seq_len, int h, int pos) {
  return batch < 1 || seq_len < 1 || h < 1 || pos < 0 ? OHARA_EINVAL : phi_teams(batch, seq_len, h, pos);
}

}  // extern "C"
