// Phi's side of the KV-cache decode path (ohara/models/phi.py): what differs from Llama.
//   LayerNorm with bias                     phi.py:132, :160 (nn.LayerNorm: fp32 statistics, one rounding)
//   append of the UN-rotated key / value    phi.py:95 (kv_cache.py:104-105)
//   attention in fp32 with the partial half-split rotation applied after the cache read
//                                           phi.py:98-117, rotary.py:131-184
// The projections with bias, new_gelu and the parallel-block sum are epilogues of the skinny
// GEMM (gemm_epilogue.h).
#include "phi_attn.h"

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
// One workgroup per (sequence, head, 64 queries); each of its four waves owns 16 queries.  Keys
// and values go through LDS in tiles of 32 positions, as fp32, the keys rotated on the way; scores and the
// weighted sum are fp32 matrix products (v_mfma_f32_16x16x4_f32), the same
// arithmetic type the reference uses (phi.py:98-117).  Both products are formed transposed,
//   S^T (position x query) = K . Q^T        O^T (feature x query) = V^T . P^T,
// so that a lane's four score registers are rows 4g .. 4g+3 of one query column: the softmax
// runs down registers plus two cross-group shuffles, and register r is already the B operand of
// the second product's k-step r (the A operand then reads value row 4g + r).
//
// What bounds it: the fp32 products (a block of 16 positions is 40 of 32 cycles at head width 80: 330 of the 574 us of the largest call
// below) and, where a workgroup has its CU to itself, the softmax and the widening of the next tile between them.  A tile's rows, and where
// VEC (the rotated features come in eights) the partners of its keys and their cosines and sines, are asked for a tile ahead, rotated in
// registers and put into the other half of LDS: one barrier a tile, where there were three with the table's round trip between two of
// them; the queries likewise, in one round trip instead of twenty.  Operands are read together, two blocks' scores take turns, a
// head's blocks run on one XCD.  32 heads of 80, us before / now: 100 tokens 18.8 / 13.8, 300 38 / 29, 700 94 / 67, 1500 219 / 157; 2 x 700
// 114 / 78, 4 x 1500 775 / 574.  With 32 queries a workgroup 73 at 700 tokens and 735 at 4 x 1500, with 128 86 and 572.
constexpr int PF_Q = 64, PF_T = 32;

template <int DT, bool VEC>  // head width / 16
__global__ __launch_bounds__(256, 2) void phi_attn_prefill_kernel(PhiAttnArgs a, int nqb, int heads) {
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

  // An eighth of a row: features 8 c .. 8 c + 7; of a rotated one the partners start at feature `partner`, the angles at `angle`.
  struct Eighth {
    uint4 x, p, c0, c1, s0, s1;
  };
  auto load8 = [&](const bf16_t* row, int position, int c) {
    Eighth e;
    e.x = ldg16(row + 8 * c);
    if (VEC) {
      const bool lo = 8 * c < half, rotated = 8 * c < a.rot;
      const int partner = rotated ? (lo ? 8 * c + half : 8 * c - half) : 8 * c, angle = rotated ? (lo ? 8 * c : 8 * c - half) : 0;
      e.p = ldg16(row + partner);
      const float* cp = a.cos + (size_t)position * half + angle;
      const float* sp = a.sin + (size_t)position * half + angle;
      e.c0 = ldg16(cp);
      e.c1 = ldg16(cp + 4);
      e.s0 = ldg16(sp);
      e.s1 = ldg16(sp + 4);
    }
    return e;
  };
  auto widen = [](uint4 v, float (&f)[8]) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = lo_bf(w[i]);
      f[2 * i + 1] = hi_bf(w[i]);
    }
  };
  // phi.py:103-104: the pair (i, i + half); which of a sum's two products is rounded first is fixed, for queries and for keys
  auto turned = [&](const Eighth& e, int c, float (&f)[8], bool query) {
    widen(e.x, f);
    if (VEC && 8 * c < a.rot) {
      float o8[8];
      widen(e.p, o8);
      const uint32_t cw[8] = {e.c0.x, e.c0.y, e.c0.z, e.c0.w, e.c1.x, e.c1.y, e.c1.z, e.c1.w};
      const uint32_t sw[8] = {e.s0.x, e.s0.y, e.s0.z, e.s0.w, e.s1.x, e.s1.y, e.s1.z, e.s1.w};
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float co = __uint_as_float(cw[u]), sn = __uint_as_float(sw[u]);
        f[u] = 8 * c < half ? __builtin_fmaf(f[u], co, -__fmul_rn(o8[u], sn)) : (query ? __builtin_fmaf(f[u], co, __fmul_rn(o8[u], sn)) : __builtin_fmaf(o8[u], sn, __fmul_rn(f[u], co)));
      }
    }
  };
  auto put8 = [](float* dst, const float (&f)[8], bool in) {
    *reinterpret_cast<float4*>(dst) = in ? make_float4(f[0], f[1], f[2], f[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    *reinterpret_cast<float4*>(dst + 4) = in ? make_float4(f[4], f[5], f[6], f[7]) : make_float4(0.f, 0.f, 0.f, 0.f);
  };

  // rotated queries -> LDS -> registers (rows beyond the call's tokens are zero)
  if (VEC) {
    constexpr int NQ = PF_Q * C8 / 256 + (PF_Q * C8 % 256 ? 1 : 0);
    Eighth e[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int idx = min(tid + 256 * i, PF_Q * C8 - 1), qi = idx / C8, sq = min(s0 + qi, a.S - 1);
      e[i] = load8(a.q + ((size_t)seq * a.S + sq) * a.ldq + h * D, pos0 + sq, idx - qi * C8);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
      const int idx = tid + 256 * i, qi = idx / C8, c = idx - qi * C8;
      if (qi >= PF_Q) continue;
      float f[8];
      turned(e[i], c, f, true);
      put8(sm + qi * LD + 8 * c, f, s0 + qi < a.S);
    }
  } else
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
  Eighth kr[NV];
  uint4 vr[NV];
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
      kr[i] = load8(kb + (size_t)t * hd, t, c);
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
      turned(kr[i], c, k, false);
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
    if (!VEC) {
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
    }
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

template <int DT>
int launch_phi_prefill(const PhiAttnArgs& a, int batch, hipStream_t st) {
  constexpr int LDS = 2 * 2 * PF_T * (16 * DT + 4) * (int)sizeof(float);
  const int64_t nqb = (a.S + PF_Q - 1) / PF_Q, heads = (int64_t)a.H * batch, grid = nqb * ((heads + 7) / 8 * 8);
  if (grid > INT32_MAX) return OHARA_ESIZE;
  auto kernel = phi_eights(a) ? phi_attn_prefill_kernel<DT, true> : phi_attn_prefill_kernel<DT, false>;
  if (LDS > 64 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), LDS, st, a, (int)nqb, (int)heads);
  return ohara_launch_status();
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
    // many new tokens: queries in tiles of 64 against key / value tiles in LDS, fp32 matrix products
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

}  // extern "C"
