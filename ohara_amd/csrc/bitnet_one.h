// One decode step of ONE sequence of the BitNet-b1.58 Llama in one launch, without a grid barrier inside the layers.
// Included by bitnet_mega.hip, whose arithmetic (codes, scales, orders of sums) it shares.
//
// What bounds it: a layer's weights are 12.8 MB (2.5 us at a copy's rate), its six hand-offs between workgroups are a chain.  So
//   * every hand-off is a row in a mailbox whose words are polled for (persistent.h): 0.7 - 0.9 us from the store to the last reader,
//     against 1.6 - 2.1 us for a grid barrier and a cold fetch of the row behind it;
//   * a chunk's attention partials are polled for too, by ONE workgroup a head, which merges them and hands on 256 bytes.  (Before,
//     each of the 128 workgroups of the output projection read all partials, 133 KB at 16 heads: 5.1 us of that phase.)
//   * the down projection keeps its K whole: its eleven kilobytes a wave are no stream worth a second hand-off of sums;
//   * all weights and norm weights of the layer ahead lie in LDS (116 KB), requested where the workgroup has nothing to do next: a
//     wave's loads return in order, so what is requested ahead of a poll holds it up, and with one wave a SIMD every instruction
//     between a poll and the stores it leads to is five cycles of the layer (asking for weights there was 0.9 us a layer);
//   * a row's reductions take one workgroup barrier each, and gate's and up's codes share theirs: both norm the same row;
//   * a strip's sixteen outputs are finished by a lane each (the sixteen columns of the product are the same row), not by four lanes;
//   * nobody has two units of a phase: the host takes the general kernel where the grid is too small for that.
// Twenty-four layers of 2048 x 5632: at context 2048 747 us a step with five grid barriers a layer, 524 now, 19.8 us a layer.  Of those the
// hand-offs are 9 (each 1.3 to 1.9 with the wait for the slowest workgroup), and 10 the four integer phases between a poll and the stores it
// leads to, 2.1 to 3.1 each: reductions, codes and outputs are a chain of dependent instructions in one wave a SIMD.
#pragma once
#include "lds_tile.h"

namespace {

// What of the layer ahead lies in LDS: each wave's tiles of its first unit, each thread's pieces of the norm weights.
constexpr int ONE_T1 = 4, ONE_T3 = 2, ONE_T4 = 8, ONE_T5 = 6;          // tiles a wave: q/k/v, output, gate and up, down
constexpr int ONE_N1 = 2, ONE_N3 = 1, ONE_N4 = 3, ONE_N5 = 3;          // pieces a thread
constexpr int ONE_AHEAD_KB = 4 * (ONE_T1 + ONE_T3 + ONE_T4 + ONE_T5 + ONE_N1 + ONE_N3 + ONE_N4 + ONE_N5);

// The mailboxes of a layer, in bytes from its block: stream after the attention block | stream after the layer | q | new key and
// value rows | activations | merged attention row | attention partials.
struct OneBoxes {
  int xn, q, kv, act, row, part;
  size_t stride;  // a layer's block; a set is n_layers of them
};
__host__ __device__ inline int one_al(int v) { return (v + 255) & ~255; }
__host__ __device__ inline OneBoxes one_boxes(const OharaBitModel& m) {
  const int D = m.head_dim, hd = m.n_heads * D;
  OneBoxes b;
  b.xn = one_al(m.d_model * 2);
  b.q = 2 * b.xn;
  b.kv = b.q + one_al(hd * 2);
  b.act = b.kv + one_al(4 * m.n_kv_heads * D);
  b.row = b.act + one_al(m.d_ff * 2);
  b.part = b.row + one_al(hd * 2);
  b.stride = (size_t)b.part + one_al(m.n_heads * OHARA_MEGA_NS * (D + 32) * 4);
  return b;
}

// Sums and maxima of the workgroup with one barrier each: two slots take turns, and between a slot's readers and its next writers
// lies the other slot's barrier.
struct OneRed {
  float* slot;  // [2][8]
  int k;
  __device__ __forceinline__ float* post(float v0, float v1) {
    float* s = slot + k * 8;
    k ^= 1;
    if ((threadIdx.x & 63) == 0) {
      s[threadIdx.x >> 6] = v0;
      s[4 + (threadIdx.x >> 6)] = v1;
    }
    __syncthreads();
    return s;
  }
  __device__ __forceinline__ float sum(float v) {
    const float* s = post(wave_sum(v), 0.f);
    return ((s[0] + s[1]) + s[2]) + s[3];
  }
  __device__ __forceinline__ void max2(float& a, float& b) {
    const float* s = post(wave_max(a), wave_max(b));
    a = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    b = fmaxf(fmaxf(s[4], s[5]), fmaxf(s[6], s[7]));
  }
};

// The tiles of a unit (strip, K split over KP waves) into the wave's part of `base`, and a norm weight's pieces into the threads'.
template <int KP, int NT>
__device__ __forceinline__ void one_request(uint32_t base, int first, const uint4* wp, int KC, int strip, bool live) {
  int c0, c1;
  bit_wave_chunks<KP>(0, KC, c0, c1);
  c0 = __builtin_amdgcn_readfirstlane(c0);
  c1 = __builtin_amdgcn_readfirstlane(live ? c1 : 0);
  const uint32_t dst = __builtin_amdgcn_readfirstlane(base + ((threadIdx.x >> 6) * NT + first) * 1024);
  const int st = __builtin_amdgcn_readfirstlane(strip);
  for (int c = 0; c0 + c < c1; ++c)
    load_lds16(dst + c * 1024, wp + ((size_t)st * KC + c0 + c) * 64, (threadIdx.x & 63) * 16);
}
template <int NP = 1>  // pieces past the row: its last one again, which meets zeros
__device__ __forceinline__ void one_request_norm(uint32_t base, const bf16_t* w, int pieces) {
  const uint32_t dst = __builtin_amdgcn_readfirstlane(base + (threadIdx.x >> 6) * 1024);
  for (int i = 0; i < NP; ++i)
    load_lds16(dst + i * 4096, w, min((int)threadIdx.x + 256 * i, pieces - 1) * 16);
}

// This thread's pieces of a row of `pieces` pieces, polled for; beyond the row zeros.  Behind it nothing of this wave is in flight.
template <int NP>
__device__ __forceinline__ void one_poll(uint4 (&v)[NP], const char* row, int pieces, const Poll& pc) {
  const MbRsrc rs = mb_rsrc(row);
  unsigned int spins = 0;
  for (;;) {
    bool ok = true;
#pragma unroll
    for (int i = 0; i < NP; ++i) ok = mb_ld16(rs, min((int)threadIdx.x + 256 * i, pieces - 1) * 8, v[i]) && ok;
    if (__all(ok) || poll_expired(pc, spins)) break;
  }
  wait_loads<0>();
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if ((int)threadIdx.x + 256 * i >= pieces) v[i] = make_uint4(0, 0, 0, 0);
}

// The codes of a row (bitnet.py:29-33, 49-53) for one BitLinear or two that share it, behind the block's own norm where there is one
// (norm.py:16-21).  A sum of squares is a thread's pieces in their order (t, t + 256, ...), the wave's butterfly, then the four waves in
// theirs; scale, codes and their sum from the same values in the same steps as everywhere (bit_xhat8, bit_mag_max8, bit_codes8).
// `nw`: this thread's pieces of the norm weights in LDS, those of the block first.  Scales to every thread; each wave leaves its share of the sums of the codes in sumw.
template <int NP, int NSETS, bool BLOCK>
__device__ __forceinline__ void one_codes(uint4 (&x)[NP], uint32_t nw, int K, float eps, const BitLds& L, OneRed& red, float (&scale)[2]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, pieces = K >> 3;
  const uint32_t mine = nw + tid * 16;
  auto rinv_of = [&]() {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) ss += bit_sumsq8(x[i]);
    return 1.0f / sqrtf(red.sum(ss) / (float)K + eps);
  };
  if (BLOCK) {
    uint4 w[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) w[i] = lds16_at(mine + i * 4096);
    const float r = rinv_of();
#pragma unroll
    for (int i = 0; i < NP; ++i) x[i] = bit_xhat8(x[i], w[i], r);
  }
  uint4 xh[NSETS][NP];
#pragma unroll
  for (int s = 0; s < NSETS; ++s)
#pragma unroll
    for (int i = 0; i < NP; ++i) xh[s][i] = lds16_at(mine + ((BLOCK ? 1 : 0) + s) * 4096 + i * 4096);
  const float rinv = rinv_of();
  float mx[2] = {0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NSETS; ++s) {
    uint32_t mg = 0u;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      xh[s][i] = bit_xhat8(x[i], xh[s][i], rinv);
      mg = bit_mag_max8(mg, xh[s][i]);
    }
    mx[s] = bit_mag_float(mg);
  }
  red.max2(mx[0], mx[1]);
#pragma unroll
  for (int s = 0; s < NSETS; ++s) {
    scale[s] = 127.0f / fmaxf(mx[s], 1e-5f);
    int8_t* xq = L.codes + s * L.set;
    uint32_t sqw = 0u;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const uint2 pk = bit_codes8(xh[s][i], scale[s], sqw);
      const int p = tid + 256 * i;
      if (p < pieces) sts8(xq + (size_t)p * 8, pk);
    }
    const int pad8 = (L.ldq - K) >> 3;  // at most 34
    if (tid < pad8) sts8(xq + K + tid * 8, make_uint2(0, 0));
    const int sq = lanes_sum<32, 1>(bit_code_sum(sqw, NP * 8));
    if (lane == 0) L.sumw[s * 4 + wave] = sq;
  }
  __syncthreads();
}
__device__ __forceinline__ int one_code_sum(const BitLds& L, int s) {
  return (L.sumw[s * 4] + L.sumw[s * 4 + 1]) + (L.sumw[s * 4 + 2] + L.sumw[s * 4 + 3]);
}

// This wave's chunks of a strip (CNT at most) times the codes; all reads stand ahead of the first product.
template <int KP, int NT, int CNT>
__device__ __forceinline__ i32x4 one_product(uint32_t base, int first, int KC, bool live, const int8_t* xq) {
  const int lane = threadIdx.x & 63;
  int c0, c1;
  bit_wave_chunks<KP>(0, KC, c0, c1);
  i32x4 acc = {0, 0, 0, 0}, odd = acc;
  const int n = __builtin_amdgcn_readfirstlane(live ? c1 - c0 : 0);
  if (n <= 0) return acc;
  const uint32_t tiles = base + (((threadIdx.x >> 6) * NT + first) * 64 + lane) * 16;
  const uint32_t xrow = (uint32_t)(uintptr_t)(const OHARA_LDS int8_t*)xq + 16 * (lane >> 4) + (c0 << 8);
  uint4 wv[CNT], xv[CNT][4];
#pragma unroll
  for (int c = 0; c < CNT; ++c) {
    if (c >= n) break;
    wv[c] = lds16_at(tiles + c * 1024);
#pragma unroll
    for (int j = 0; j < 4; ++j) xv[c][j] = lds16_at(xrow + (c << 8) + 64 * j);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < CNT; ++c) {
    if (c >= n) break;
    const uint32_t dw[4] = {wv[c].x, wv[c].y, wv[c].z, wv[c].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const i32x4 av = {(int)(dw[j] & 0x03030303u), (int)((dw[j] >> 2) & 0x03030303u), (int)((dw[j] >> 4) & 0x03030303u),
                        (int)((dw[j] >> 6) & 0x03030303u)};
      const i32x4 bv = {(int)xv[c][j].x, (int)xv[c][j].y, (int)xv[c][j].z, (int)xv[c][j].w};
      i32x4& to = j & 1 ? odd : acc;
      to = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, to, 0, 0, 0);
    }
  }
  return acc + odd;
}
// The sixteen sums of each strip over its KP waves: every wave leaves its share in `part` ([4][16] words that nothing else uses until
// the next barrier but one), and behind the barrier lane (g, m < 4) of the strip's first wave takes output 4 g + m.
__device__ __forceinline__ void one_leave(const i32x4& acc, int* part) {
  const int lane = threadIdx.x & 63;
  if ((lane & 15) == 0) *reinterpret_cast<i32x4*>(part + (threadIdx.x >> 6) * 16 + (lane >> 4) * 4) = acc;
}
template <int KP>
__device__ __forceinline__ int one_fold(const int* part) {
  const int lane = threadIdx.x & 63;
  const int* p = part + ((threadIdx.x >> 6) & ~(KP - 1)) * 16 + (lane >> 4) * 4 + (lane & 3);
  int v[KP], t = 0;
#pragma unroll
  for (int w = 0; w < KP; ++w) v[w] = p[w * 16];
#pragma unroll
  for (int w = 0; w < KP; ++w) t += v[w];
  return t;
}
// One output (bit_scale), and a lane's output with its three neighbours' as the four values that are stored together.
__device__ __forceinline__ float one_scale(int sum, float s, float gamma) { return rbf(__fmul_rn(__fdiv_rn((float)sum, s), gamma)); }
__device__ __forceinline__ uint2 one_gather(float v) {  // (valid in the first lane of four)
  const uint32_t lo = pack_bf(v, lane_xor<1>(v));
  return make_uint2(lo, lane_xor_u32<2>(lo));
}
__device__ __forceinline__ float one_value(uint2 four) {  // this lane's of four values
  const uint32_t w = threadIdx.x & 2 ? four.y : four.x;
  return threadIdx.x & 1 ? hi_bf(w) : lo_bf(w);
}

template <int D, bool PROFILE = false>
__global__ __launch_bounds__(256) void bitnet_one_kernel(BitMegaArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const OharaBitModel& m = a.m;
  const int d = m.d_model, H = m.n_heads, Hkv = m.n_kv_heads, F = m.d_ff, V = m.vocab, HD = H * D;
  const int nwg = gridDim.x, wg = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int mm = lane & 15, gg = lane >> 4;
  // ---- LDS (one_smem_bytes counts the same) ----
  const int kmax = max(max(d, HD), F), Kp = ((kmax + 255) >> 8) << 8, Kpd = ((d + 255) >> 8) << 8;
  BitLds L;
  size_t off = 0;
  auto take = [&](size_t n) {
    unsigned char* p = smem + off;
    off += (n + 255) & ~(size_t)255;
    return p;
  };
  const uint32_t ahead = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)take((size_t)ONE_AHEAD_KB * 1024);
  const uint32_t t1 = ahead, t3 = t1 + 4096 * ONE_T1, t4 = t3 + 4096 * ONE_T3, t5 = t4 + 4096 * ONE_T4;
  const uint32_t n1 = t5 + 4096 * ONE_T5, n3 = n1 + 4096 * ONE_N1, n4 = n3 + 4096 * ONE_N3, n5 = n4 + 4096 * ONE_N4;
  L.codes = reinterpret_cast<int8_t*>(take(max((size_t)Kp + 16, (size_t)2 * (Kpd + 16))));
  L.stage = reinterpret_cast<bf16_t*>(take((size_t)(d + 8) * 2));
  L.red = reinterpret_cast<float*>(take(4096));
  L.sumw = reinterpret_cast<int*>(take(64));
  OneRed red{reinterpret_cast<float*>(take(64)), 0};
  int* fold = reinterpret_cast<int*>(take(512));  // gate's and up's parts, or one product's
  float* att = reinterpret_cast<float*>(take((size_t)(8 + 4 * D) * sizeof(float)));
  float* mrg = reinterpret_cast<float*>(take(merge_head_lds(D)));
  BitLayerDev* ltab = reinterpret_cast<BitLayerDev*>(take(0));
  {
    const uint32_t* src = reinterpret_cast<const uint32_t*>(a.layers_dev);
    uint32_t* dst = reinterpret_cast<uint32_t*>(ltab);
    const int n = m.n_layers * (int)(sizeof(BitLayerDev) / 4);
    for (int i = tid; i < n; i += 256) dst[i] = src[i];
  }
  __syncthreads();
  auto uni = [&](const void* p) {  // a pointer read from LDS, made wave-uniform
    const unsigned long long v = reinterpret_cast<unsigned long long>(p);
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return ((unsigned long long)hi << 32) | lo;
  };
  auto weights = [&](int l, int i) { return reinterpret_cast<const uint4*>(uni(ltab[l].w[i])); };
  auto norms = [&](const bf16_t* p) { return reinterpret_cast<const bf16_t*>(uni(p)); };

  GridSync gs;
  gs.init(a.bar, nwg, a.spin_limit);
  unsigned int* launches = a.bar + (gs.ng + 12) * 64;
  const unsigned int nth = *launches + 1u;  // the last workgroup out advances it
  const Poll pc{a.spin_limit, gs.err};
  const OneBoxes bx = one_boxes(m);
  const size_t set_bytes = bx.stride * m.n_layers;
  char* const boxes = a.tg + (size_t)(nth & 1u) * set_bytes;
  const ptrdiff_t other = (nth & 1u) ? -(ptrdiff_t)set_bytes : (ptrdiff_t)set_bytes;
  const int pos = a.step_state[0], step = a.step_state[1];
  const int Lc = min(pos + 1, m.t_max);
  const bool ok_pos = pos >= 0 && pos < m.t_max;
  float best_v = -INFINITY;
  int best_i = 0x7fffffff;

  const int KCd = (d + 255) >> 8, KCo = (HD + 255) >> 8, KCf = (F + 255) >> 8;
  const int ns_q = HD / 16, ns_kv = (Hkv * D) / 16, ns_d = (d + 15) / 16, ns_f = (F + 15) / 16;
  // Who does what.  A unit of q/k/v and of gate/up is two strips, two waves each; one of the output and of the down projection is a
  // strip over four waves.  Attention, gate/up and the output projection start at workgroup 0, q/k/v and the down projection end
  // with the grid, and the heads' merges stand behind the output projection.
  const int uq = (ns_q + 1) >> 1, ukv = (ns_kv + 1) >> 1, u1 = uq + 2 * ukv, u4 = (ns_f + 1) >> 1;
  const int sub = wave >> 1;
  const int i1 = wg - (nwg - u1), i5 = wg - (nwg - ns_d), ih = wg - min(ns_d, nwg - H);
  const bool has1 = i1 >= 0, has3 = wg < ns_d, has4 = wg < u4, has5 = i5 >= 0, merges = ih >= 0 && ih < H;
  const int which = i1 < uq ? BQ : (i1 < uq + ukv ? BK : BV);
  const int strip1 = 2 * (which == BQ ? i1 : which == BK ? i1 - uq : i1 - uq - ukv) + sub, strip4 = 2 * wg + sub;
  const bool live1 = has1 && strip1 < (which == BQ ? ns_q : ns_kv), live4 = has4 && strip4 < ns_f;
  ProfT<PROFILE> pf((a.prof && tid == 0) ? (wg == 0 ? a.prof : i5 == 0 ? a.prof + 512 : nullptr) : nullptr);

  // ---- requests of the layer ahead ----
  auto ask1 = [&](int l) {
    if (!has1 || l >= m.n_layers) return;
    one_request<2, ONE_T1>(t1, 0, weights(l, which), KCd, strip1, live1);
    one_request_norm(n1, norms(ltab[l].norm1), d >> 3);
    one_request_norm(n1 + 4096, norms(ltab[l].nw[which]), d >> 3);
  };
  auto ask3 = [&](int l) {
    if (!has3 || l >= m.n_layers) return;
    one_request<4, ONE_T3>(t3, 0, weights(l, BO), KCo, wg, true);
    one_request_norm(n3, norms(ltab[l].nw[BO]), HD >> 3);
  };
  auto ask4 = [&](int l) {
    if (!has4 || l >= m.n_layers) return;
    one_request<2, ONE_T4>(t4, 0, weights(l, BG), KCd, strip4, live4);
    one_request<2, ONE_T4>(t4, ONE_T4 / 2, weights(l, BU), KCd, strip4, live4);
    one_request_norm(n4, norms(ltab[l].norm2), d >> 3);
    one_request_norm(n4 + 4096, norms(ltab[l].nw[BG]), d >> 3);
    one_request_norm(n4 + 8192, norms(ltab[l].nw[BU]), d >> 3);
  };
  auto ask5 = [&](int l) {
    if (!has5) return;
    one_request<4, ONE_T5>(t5, 0, weights(l, BD), KCf, i5, true);
    one_request_norm<ONE_N5>(n5, norms(ltab[l].nw[BD]), F >> 3);
  };
  AttnPre<D> apre;
  auto ask_kv = [&](int l) {
    if (l < m.n_layers)
      attn_prefetch<D>(1, Hkv, m.t_max, a.ns, reinterpret_cast<const bf16_t*>(uni(ltab[l].kc)), reinterpret_cast<const bf16_t*>(uni(ltab[l].vc)),
                       Lc, apre);
  };
  ask1(0);
  ask3(0);
  if (has3) ask4(0);
  ask_kv(0);
  // the rotation of this lane's output and its neighbour's: the same in every layer
  float rope_c = 0.f, rope_s = 0.f;
  if (live1 && which != BV && ok_pos) {
    const int dd = (strip1 * 16 + 4 * gg) % D + (mm & 2);
    rope_c = bf2f(m.cos[(size_t)pos * (D >> 1) + (dd >> 1)]);
    rope_s = bf2f(m.sin[(size_t)pos * (D >> 1) + (dd >> 1)]);
  }
  int64_t id0 = ldg_i64(a.ids);
  if (id0 < 0 || id0 >= V) id0 = 0;
  const bf16_t* emb = m.token_emb + (size_t)id0 * d;

  GemmP lm{};
  lm.N = V; lm.K = d; lm.nstrips = (V + 15) / 16; lm.out = reinterpret_cast<char*>(a.logits); lm.ldo = V;
  lm.valid = a.valid_vocab > 0 ? min(a.valid_vocab, V) : V;
  lm.wp = reinterpret_cast<const uint4*>(m.w_vocab);
  float s[2];

  for (int l = 0; l < m.n_layers; ++l) {
    const BitLayerDev& LY = ltab[l];
    bf16_t* kc = reinterpret_cast<bf16_t*>(uni(LY.kc));
    bf16_t* vc = reinterpret_cast<bf16_t*>(uni(LY.vc));
    char* xt = boxes + (size_t)l * bx.stride;
    const char* xn_prev = xt - bx.stride + bx.xn;  // (l > 0)
    // four values of the stream, requested ahead of a product: seen a phase or more ago by everyone they came to, and looked at behind it
    auto arrived = [&](uint2 r, const char* row, int r0) {
      unsigned int spins = 0;
      while ((r.x == OHARA_UNWRITTEN || r.y == OHARA_UNWRITTEN) && !poll_expired(pc, spins)) r = ld_coh8(row + (size_t)r0 * 2);
      return r;
    };

    // ---- P1: norm1, codes, q / k / v, rotary, append ----
    if (has1) {
      L.shape(1, d);
      uint4 x[1];
      if (l == 0) {
        x[0] = ldg16(emb + (size_t)min(tid, (d >> 3) - 1) * 8);
        if (tid >= d >> 3) x[0] = make_uint4(0, 0, 0, 0);
        wait_loads<0>();
      } else {
        one_poll<1>(x, xn_prev, d >> 3, pc);
      }
      pf.stamp();
      one_codes<1, 1, true>(x, n1, d, m.eps, L, red, s);
      one_leave(one_product<2, ONE_T1, ONE_T1>(t1, 0, KCd, live1, L.codes), fold);
      __syncthreads();
      if (wave % 2 == 0 && live1) {
        const int r0 = strip1 * 16 + 4 * gg;
        float v = one_scale(one_fold<2>(fold) - one_code_sum(L, 0), s[0], LY.gamma[which]);
        if (which != BV) {
          const float w = lane_xor<1>(v);  // (the pair's other half)
          v = mm & 1 ? __fadd_rn(__fmul_rn(w, rope_s), __fmul_rn(v, rope_c)) : __fsub_rn(__fmul_rn(v, rope_c), __fmul_rn(w, rope_s));
        }
        const uint2 o = one_gather(v);
        if (mm == 0) {
          if (which == BQ) mb_st8(xt + bx.q, other, r0, o.x, o.y);
          else {
            mb_st8(xt + bx.kv, other, (which == BV ? Hkv * D : 0) + r0, o.x, o.y);
            if (ok_pos) st_coh8((which == BK ? kc : vc) + (size_t)pos * Hkv * D + r0, o);  // for the steps after this one
          }
        }
      }
    } else {
      pf.stamp();
    }
    pf.stamp();
    // ---- P2: attention partials, then the merge of a head's by one workgroup ----
    attn_phase<D, 1, true, false, true>(1, H, Hkv, m.t_max, 0, a.ns, apre, nullptr, reinterpret_cast<float*>(xt + bx.part), kc, vc, Lc,
                                              att, xt + bx.q, xt + bx.kv, pc, 0, 0, nullptr, L.red, other);
    pf.stamp();
    if (merges) merge_head<D>(xt + bx.part + (size_t)ih * OHARA_MEGA_NS * (D + 32) * 4, a.ns, mrg, xt + bx.row + ih * D * 2, other, pc);
    pf.stamp();
    ask1(l + 1);
    ask5(l);
    if (!has3) {  // (these are idle until gate/up; the others, at the usual sizes, behind it)
      ask4(l);
      ask_kv(l + 1);
    }
    // ---- P3: codes of the merged row, output projection, residual ----
    if (has3) {
      L.shape(1, HD);
      const int r0 = wg * 16 + 4 * gg;
      uint4 x[1];
      one_poll<1>(x, xt + bx.row, HD >> 3, pc);
      pf.stamp();
      uint2 r = make_uint2(0, 0);
      if (wave == 0) r = l == 0 ? ldg8(emb + r0) : ld_coh8(xn_prev + (size_t)r0 * 2);
      one_codes<1, 1, false>(x, n3, HD, m.eps, L, red, s);
      one_leave(one_product<4, ONE_T3, ONE_T3>(t3, 0, KCo, true, L.codes), fold);
      __syncthreads();
      if (wave == 0) {
        if (l > 0) r = arrived(r, xn_prev, r0);
        const uint2 o = one_gather(one_value(r) + one_scale(one_fold<4>(fold) - one_code_sum(L, 0), s[0], LY.gamma[BO]));
        if (mm == 0) mb_st8(xt, other, r0, o.x, o.y);
      }
    } else {
      pf.stamp();
    }
    pf.stamp();
    // ---- P4: norm2, codes of gate and up, both products, SwiGLU ----
    if (has4) {
      L.shape(1, d);
      uint4 x[1];
      one_poll<1>(x, xt, d >> 3, pc);
      pf.stamp();
      one_codes<1, 2, true>(x, n4, d, m.eps, L, red, s);
      one_leave(one_product<2, ONE_T4, ONE_T4 / 2>(t4, 0, KCd, live4, L.codes), fold);
      one_leave(one_product<2, ONE_T4, ONE_T4 / 2>(t4, ONE_T4 / 2, KCd, live4, L.codes + L.set), fold + 64);
      __syncthreads();
      if (wave % 2 == 0 && live4) {
        const float yg = one_scale(one_fold<2>(fold) - one_code_sum(L, 0), s[0], LY.gamma[BG]);
        const float yu = one_scale(one_fold<2>(fold + 64) - one_code_sum(L, 1), s[1], LY.gamma[BU]);
        const uint2 o = one_gather(rbf(silu_f(yg)) * yu);
        if (mm == 0) mb_st8(xt + bx.act, other, strip4 * 16 + 4 * gg, o.x, o.y);
      }
    } else {
      pf.stamp();
    }
    pf.stamp();
    if (has3) {
      ask3(l + 1);
      ask4(l + 1);
      ask_kv(l + 1);
    }
    // ---- P5: codes of the activations, down projection, residual ----
    if (has5) {
      L.shape(1, F);
      const int r0 = i5 * 16 + 4 * gg;
      uint4 x[ONE_N5];
      one_poll<ONE_N5>(x, xt + bx.act, F >> 3, pc);
      pf.stamp();
      uint2 r = make_uint2(0, 0);
      if (wave == 0) r = ld_coh8(xt + (size_t)r0 * 2);
      one_codes<ONE_N5, 1, false>(x, n5, F, m.eps, L, red, s);
      one_leave(one_product<4, ONE_T5, ONE_T5>(t5, 0, KCf, true, L.codes), fold);
      __syncthreads();
      if (wave == 0) {
        r = arrived(r, xt, r0);
        const uint2 o = one_gather(one_value(r) + one_scale(one_fold<4>(fold) - one_code_sum(L, 0), s[0], LY.gamma[BD]));
        if (mm == 0) mb_st8(xt + bx.xn, other, r0, o.x, o.y);
      }
    } else {
      pf.stamp();
    }
    pf.stamp();
  }
  GemmPre lpre;
  gemm_prefetch<1, 24, E_LOGITS>(lm, lpre, 1);
  // ---- final norm + vocabulary projection (bf16), running arg-max per lane ----
  {
    uint4 x[1];
    one_poll<1>(x, boxes + (size_t)(m.n_layers - 1) * bx.stride + bx.xn, d >> 3, pc);
    bf16_t* xs = L.stage;
    if (tid < d >> 3) sts16(xs + tid * 8, x[0]);
    __syncthreads();
    if (wave == 0) {  // in the order of bit_stage_final_norm: a lane's pieces are 64 apart
      uint4 v[4], g[4];
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int k = (c * 64 + lane) * 8;
        v[c] = k < d ? lds16(xs + k) : make_uint4(0, 0, 0, 0);
        g[c] = k < d ? ldg16(m.final_norm + k) : make_uint4(0, 0, 0, 0);
        ss += bit_sumsq8(v[c]);
      }
      const float rinv = 1.0f / sqrtf(wave_sum(ss) / (float)d + m.eps);
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if ((c * 64 + lane) * 8 < d) sts16(xs + (c * 64 + lane) * 8, bit_xhat8(v[c], g[c], rinv));
    }
    __syncthreads();
    lm_phase(lm, lpre, xs, d + 8, 1, best_v, best_i, pf);
  }
  if (a.select) bit_select(a, L.red, gs, best_v, best_i, 1, step, pf);
  // bookkeeping by the last workgroup out: nobody reads these again in this launch
  if (tid == 0) {
    const unsigned int out = __hip_atomic_fetch_add(a.bar + (gs.ng + 13) * 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (out + 1u == nth * gs.nwg) {
      *launches = nth;
      *gs.done = gs.k - 1;
      if (a.select) {
        a.step_state[0] = pos + 1;
        a.step_state[1] = step + 1;
      }
    }
  }
}

size_t one_smem_bytes(const OharaBitModel* m) {
  const int D = m->head_dim, hd = m->n_heads * D;
  const int kmax = m->d_model > hd ? (m->d_model > m->d_ff ? m->d_model : m->d_ff) : (hd > m->d_ff ? hd : m->d_ff);
  const size_t Kp = (size_t)((kmax + 255) >> 8) << 8, Kpd = (size_t)((m->d_model + 255) >> 8) << 8;
  size_t o = 0;
  auto take = [&](size_t n) { o += (n + 255) & ~(size_t)255; };
  take((size_t)ONE_AHEAD_KB * 1024);
  take(Kp + 16 > 2 * (Kpd + 16) ? Kp + 16 : 2 * (Kpd + 16));
  take((size_t)(m->d_model + 8) * 2);
  take(4096);
  take(64);
  take(64);
  take(512);
  take((size_t)(8 + 4 * D) * sizeof(float));
  take(merge_head_lds(D));
  return o + sizeof(BitLayerDev) * m->n_layers;
}

}  // namespace
