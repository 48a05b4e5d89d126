// BitNet-b1.58 BitLinear with real integer arithmetic: 2-bit packed ternary weights x int8
// per-token activations, int32 accumulation on v_mfma_i32_16x16x64_i8.
//
// The reference (experiments/bitnet/bitnet.py:29-59) is float fake-quantisation recomputed on
// every forward; its effective semantics, which these kernels implement exactly, are
//   x_hat = RMSNorm_in(x)                                  (:49,53; own norm weight, eps 1e-5)
//   s     = 127 / max(max|x_hat|, 1e-5)      per token     (:31)
//   q     = clamp(rint(x_hat * s), -128, 127)              (:32; torch.round = half to even)
//   T     = clamp(rint(W / mean|W|), -1, 1),  gamma = max(mean|W|, 1e-5)   (:37-43)
//   acc   = sum_k q[k] * T[n,k]              int32, exact  <- the bit-exact contract
//   y     = (float(acc) / s) * gamma         (bias dropped, :58)
//
// Packed weight layout: strips of 16 rows, chunks of 256 columns; the tile (strip, chunk) is
// 64 lanes x 16 bytes; lane 16*g + m holds row 16*strip + m; its dword j serves the j-th MFMA of
// the chunk and carries, at bit 8*t + 2*r, the code T+1 of column 256*chunk + 64*j + 16*g + 4*r + t,
// so "(dword >> 2r) & 0x03030303" is register r of the MFMA operand.  Codes are 0..2, hence
// acc = sum q*code - sum q, the second term being one number per token.
#include "lds_tile.h"

namespace {

constexpr int BL_EPL = 96;  // K <= 6144 (LDS: int8 rows + four staged bf16 rows)

__device__ __forceinline__ float sumsq8_bits(uint4 v) {
  float s = 0.f;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = lo_bf(w[i]), b = hi_bf(w[i]);
    s += a * a + b * b;
  }
  return s;
}

struct QuantOut {
  float s;      // 127 / max|x_hat|
  int sumq;     // sum of the quantised row
};

// One wave normalises and quantises one row.  The row is walked three or four times (sum of
// squares [, block norm], BitLinear norm + max, quantise); between the walks it lives in `stage`
// (LDS, K bf16 values - every intermediate is a bf16 value, so nothing is lost), which keeps the
// register footprint independent of K.  Lane l owns the 8-value pieces l, l + 64, ...
// pre_w (optional) is the weight of a block-level RMSNorm applied first (ohara/models/llama.py:
// 199-200 norm1 / norm2), nw the BitLinear's own norm weight.  xq: int8 destination (LDS or
// global).  Returns (s, sum q) in every lane.  K % 8 == 0.
__device__ __forceinline__ QuantOut wave_quant_row(const bf16_t* x, const bf16_t* pre_w, const bf16_t* nw, int K,
                                                   float eps, int8_t* xq, bf16_t* stage) {
  const int lane = threadIdx.x & 63;
  const int pieces = K >> 3;
  float ss = 0.f;
  for (int p = lane; p < pieces; p += 64) {
    const uint4 u = ldg16(x + (size_t)p * 8);
    *reinterpret_cast<uint4*>(stage + p * 8) = u;
    ss += sumsq8_bits(u);
  }
  if (pre_w) {
    ss = wave_sum(ss);
    const float rinv0 = 1.0f / sqrtf(ss / (float)K + eps);
    ss = 0.f;
    for (int p = lane; p < pieces; p += 64) {
      const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
      const uint4 w = ldg16(pre_w + (size_t)p * 8);
      const uint32_t uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o[j] = pack_bf(rbf(lo_bf(uu[j]) * rinv0) * lo_bf(ww[j]), rbf(hi_bf(uu[j]) * rinv0) * hi_bf(ww[j]));
      const uint4 v = make_uint4(o[0], o[1], o[2], o[3]);
      *reinterpret_cast<uint4*>(stage + p * 8) = v;
      ss += sumsq8_bits(v);
    }
  }
  ss = wave_sum(ss);
  const float rinv = 1.0f / sqrtf(ss / (float)K + eps);
  float mx = 0.f;
  for (int p = lane; p < pieces; p += 64) {
    const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
    const uint4 w = ldg16(nw + (size_t)p * 8);
    const uint32_t uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a0 = rbf(rbf(lo_bf(uu[j]) * rinv) * lo_bf(ww[j]));  // RMSNorm output in the model dtype
      const float a1 = rbf(rbf(hi_bf(uu[j]) * rinv) * hi_bf(ww[j]));
      mx = fmaxf(mx, fmaxf(fabsf(a0), fabsf(a1)));
      o[j] = pack_bf(a0, a1);
    }
    *reinterpret_cast<uint4*>(stage + p * 8) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  mx = wave_max(mx);
  const float s = 127.0f / fmaxf(mx, 1e-5f);
  int sq = 0;
  for (int p = lane; p < pieces; p += 64) {
    const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
    const uint32_t uu[4] = {u.x, u.y, u.z, u.w};
    uint32_t pk[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = (j & 1) ? hi_bf(uu[j >> 1]) : lo_bf(uu[j >> 1]);
      const int qi = (int)fminf(fmaxf(rintf(v * s), -128.f), 127.f);
      sq += qi;
      pk[j >> 2] |= ((uint32_t)qi & 0xffu) << (8 * (j & 3));
    }
    *reinterpret_cast<uint2*>(xq + (size_t)p * 8) = make_uint2(pk[0], pk[1]);
  }
  sq = lanes_sum<32, 1>(sq);
  return QuantOut{s, sq};
}

// The same for a single row with the whole workgroup (four waves) on it: a decode step at batch 1
// has one row per projection, and one wave walking 2048-5632 values four times is most of such a
// kernel's critical path.  Thread t owns the pieces t, t + 256, ...; the three reductions go through
// `red` (four floats of LDS).  Every thread of the workgroup must call it.
__device__ __forceinline__ QuantOut block_quant_row(const bf16_t* x, const bf16_t* pre_w, const bf16_t* nw, int K,
                                                    float eps, int8_t* xq, bf16_t* stage, float* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int pieces = K >> 3;
  auto bsum = [&](float v) {
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    return ((red[0] + red[1]) + red[2]) + red[3];
  };
  float ss = 0.f;
  for (int p = tid; p < pieces; p += 256) {
    const uint4 u = ldg16(x + (size_t)p * 8);
    *reinterpret_cast<uint4*>(stage + p * 8) = u;
    ss += sumsq8_bits(u);
  }
  if (pre_w) {
    const float rinv0 = 1.0f / sqrtf(bsum(ss) / (float)K + eps);
    ss = 0.f;
    for (int p = tid; p < pieces; p += 256) {
      const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
      const uint4 w = ldg16(pre_w + (size_t)p * 8);
      const uint32_t uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        o[j] = pack_bf(rbf(lo_bf(uu[j]) * rinv0) * lo_bf(ww[j]), rbf(hi_bf(uu[j]) * rinv0) * hi_bf(ww[j]));
      const uint4 v = make_uint4(o[0], o[1], o[2], o[3]);
      *reinterpret_cast<uint4*>(stage + p * 8) = v;
      ss += sumsq8_bits(v);
    }
  }
  const float rinv = 1.0f / sqrtf(bsum(ss) / (float)K + eps);
  float mx = 0.f;
  for (int p = tid; p < pieces; p += 256) {
    const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
    const uint4 w = ldg16(nw + (size_t)p * 8);
    const uint32_t uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float a0 = rbf(rbf(lo_bf(uu[j]) * rinv) * lo_bf(ww[j]));
      const float a1 = rbf(rbf(hi_bf(uu[j]) * rinv) * hi_bf(ww[j]));
      mx = fmaxf(mx, fmaxf(fabsf(a0), fabsf(a1)));
      o[j] = pack_bf(a0, a1);
    }
    *reinterpret_cast<uint4*>(stage + p * 8) = make_uint4(o[0], o[1], o[2], o[3]);
  }
  mx = wave_max(mx);
  __syncthreads();
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = 127.0f / fmaxf(mx, 1e-5f);
  int sq = 0;
  for (int p = tid; p < pieces; p += 256) {
    const uint4 u = *reinterpret_cast<const uint4*>(stage + p * 8);
    const uint32_t uu[4] = {u.x, u.y, u.z, u.w};
    uint32_t pk[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = (j & 1) ? hi_bf(uu[j >> 1]) : lo_bf(uu[j >> 1]);
      const int qi = (int)fminf(fmaxf(rintf(v * s), -128.f), 127.f);
      sq += qi;
      pk[j >> 2] |= ((uint32_t)qi & 0xffu) << (8 * (j & 3));
    }
    *reinterpret_cast<uint2*>(xq + (size_t)p * 8) = make_uint2(pk[0], pk[1]);
  }
  sq = lanes_sum<32, 1>(sq);
  int* redi = reinterpret_cast<int*>(red);
  __syncthreads();
  if (lane == 0) redi[wave] = sq;
  __syncthreads();
  return QuantOut{s, redi[0] + redi[1] + redi[2] + redi[3]};
}

__global__ __launch_bounds__(256) void act_quant_kernel(const bf16_t* x, int ldx, const bf16_t* nw, int rows, int K,
                                                        float eps, int8_t* q, int ldq, float* s_out, int* sumq_out) {
  extern __shared__ __align__(16) unsigned char qsm[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (rows == 1) {  // the whole workgroup on the one row (the order of sums the fused kernels use for it)
    const QuantOut o = block_quant_row(x, nullptr, nw, K, eps, q, reinterpret_cast<bf16_t*>(qsm),
                                       reinterpret_cast<float*>(qsm + (size_t)K * 2));
    if (threadIdx.x == 0) {
      s_out[0] = o.s;
      sumq_out[0] = o.sumq;
    }
    return;
  }
  const int r = blockIdx.x * 4 + wave;
  if (r >= rows) return;
  const QuantOut o = wave_quant_row(x + (size_t)r * ldx, nullptr, nw, K, eps, q + (size_t)r * ldq,
                                    reinterpret_cast<bf16_t*>(qsm) + (size_t)wave * K);
  if (lane == 0) {
    s_out[r] = o.s;
    sumq_out[r] = o.sumq;
  }
}

// Many rows (more than a workgroup's LDS holds): every row is quantised once for each of up to three BitLinears that read it
// (blockIdx.y: they differ in their norm weight), and ternary_tile_kernel multiplies the codes.
struct QuantSets {
  const bf16_t* nw[3];
};
// T threads a row, its 16-byte pieces in registers (PT a thread), for all sets at once: what they share - the row, its block norm, the sums of
// squares - is worked out once, and every load goes out before the first is used.  The sums of squares are added as the kernels above add a
// row, lane l the pieces l, l + 64, ... in turn and then the lanes; the rest is exact in any order.  GATED: the row is silu(gate) * up, rounded
// as silu_mul_kernel does.  us, a wave a row and a set that walked it four or five times through LDS, each walk behind the one before / this, in a
// prompt of 300 rows: 2048 wide, one to three sets 9.2 / 5.6; 5632 wide, with the launch that multiplied gate and up 9.2 + 4.5 / 7.7.
template <int T, int PT, bool GATED>
__global__ __launch_bounds__(256) void row_quant_kernel(const bf16_t* x, int ldx, const bf16_t* up, const bf16_t* pre_w, QuantSets sets, int n_sets,
                                                        int rows, int K, float eps, int8_t* q, int ldq, float* s_out, int* sumq_out) {
  static_assert(T == 64 || T == 256, "");
  __shared__ float sums[2][T == 64 ? 1 : PT * 256], top[3][4];
  __shared__ int total[3][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, tid = T == 64 ? lane : threadIdx.x, pieces = K >> 3;
  const int r = T == 64 ? blockIdx.x * 4 + wave : blockIdx.x;
  if (T == 64 && r >= rows) return;
  uint4 v[PT], pw[PT], nw[3][PT];
#pragma unroll
  for (int i = 0; i < PT; ++i) v[i] = ldg16(x + (size_t)r * ldx + min(tid + T * i, pieces - 1) * 8);  // (past the end: the last piece, not counted)
  if (GATED) {
#pragma unroll
    for (int i = 0; i < PT; ++i) pw[i] = ldg16(up + (size_t)r * ldx + min(tid + T * i, pieces - 1) * 8);
  } else if (pre_w) {
#pragma unroll
    for (int i = 0; i < PT; ++i) pw[i] = ldg16(pre_w + min(tid + T * i, pieces - 1) * 8);
  }
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (k < n_sets) {
#pragma unroll
      for (int i = 0; i < PT; ++i) nw[k][i] = ldg16(sets.nw[k] + min(tid + T * i, pieces - 1) * 8);
    }
  __builtin_amdgcn_sched_barrier(0);
  if (GATED) {
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const uint32_t gg[4] = {v[i].x, v[i].y, v[i].z, v[i].w}, uu[4] = {pw[i].x, pw[i].y, pw[i].z, pw[i].w};
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = pack_bf(rbf(silu_f(lo_bf(gg[j]))) * lo_bf(uu[j]), rbf(silu_f(hi_bf(gg[j]))) * hi_bf(uu[j]));
      v[i] = make_uint4(o[0], o[1], o[2], o[3]);
    }
  }
  auto inverse = [&](float* sum) {  // 1 / rms of the row in v
    float ss = 0.f;
    if (T == 64) {
#pragma unroll
      for (int i = 0; i < PT; ++i)
        if (tid + T * i < pieces) ss += sumsq8_bits(v[i]);
    } else {
#pragma unroll
      for (int i = 0; i < PT; ++i) sum[tid + T * i] = sumsq8_bits(v[i]);
      __syncthreads();
      for (int p = lane; p < pieces; p += 64) ss += sum[p];
    }
    return 1.0f / sqrtf(wave_sum(ss) / (float)K + eps);
  };
  auto normed = [](uint4 u, uint4 w, float rinv) {
    const uint32_t uu[4] = {u.x, u.y, u.z, u.w}, ww[4] = {w.x, w.y, w.z, w.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = pack_bf(rbf(lo_bf(uu[j]) * rinv) * lo_bf(ww[j]), rbf(hi_bf(uu[j]) * rinv) * hi_bf(ww[j]));
    return make_uint4(o[0], o[1], o[2], o[3]);
  };
  if (!GATED && pre_w) {
    const float rinv0 = inverse(sums[0]);
#pragma unroll
    for (int i = 0; i < PT; ++i) v[i] = normed(v[i], pw[i], rinv0);
  }
  const float rinv = inverse(sums[1]);
  float most[3];
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (k < n_sets) {
      float mx = 0.f;
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        nw[k][i] = normed(v[i], nw[k][i], rinv);
        const uint32_t w[4] = {nw[k][i].x, nw[k][i].y, nw[k][i].z, nw[k][i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, fmaxf(fabsf(lo_bf(w[j])), fabsf(hi_bf(w[j]))));
      }
      most[k] = wave_max(mx);
      if (T > 64 && lane == 0) top[k][wave] = most[k];
    }
  if (T > 64) __syncthreads();
#pragma unroll
  for (int k = 0; k < 3; ++k)
    if (k < n_sets) {
      const float s = 127.0f / fmaxf(T == 64 ? most[k] : fmaxf(fmaxf(top[k][0], top[k][1]), fmaxf(top[k][2], top[k][3])), 1e-5f);
      int sq = 0;
#pragma unroll
      for (int i = 0; i < PT; ++i) {
        const int p = tid + T * i;
        const uint32_t uu[4] = {nw[k][i].x, nw[k][i].y, nw[k][i].z, nw[k][i].w};
        uint32_t pk[2] = {0u, 0u};
        int sum = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float a = (j & 1) ? hi_bf(uu[j >> 1]) : lo_bf(uu[j >> 1]);
          const int qi = (int)fminf(fmaxf(rintf(a * s), -128.f), 127.f);
          sum += qi;
          pk[j >> 2] |= ((uint32_t)qi & 0xffu) << (8 * (j & 3));
        }
        if (p < pieces) {
          sq += sum;
          *reinterpret_cast<uint2*>(q + ((size_t)k * rows + r) * ldq + (size_t)p * 8) = make_uint2(pk[0], pk[1]);
        }
      }
      sq = lanes_sum<32, 1>(sq);
      if (T > 64 && lane == 0) total[k][wave] = sq;
      if (T == 64 && lane == 0) sumq_out[(size_t)k * rows + r] = sq;
      if (tid == 0) s_out[(size_t)k * rows + r] = s;
    }
  if (T == 64) return;
  __syncthreads();
  if (tid < n_sets) sumq_out[(size_t)tid * rows + r] = total[tid][0] + total[tid][1] + total[tid][2] + total[tid][3];
}

template <bool GATED>
int launch_row_quant(const bf16_t* x, int ldx, const bf16_t* up, const bf16_t* pre_w, const QuantSets& sets, int n_sets, int rows, int K, float eps,
                     int8_t* q, int ldq, float* s, int* sumq, hipStream_t st) {
  auto go = [&](auto kernel, int per) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((rows + per - 1) / per)), dim3(256), 0, st, x, ldx, up, pre_w, sets, n_sets, rows, K, eps, q, ldq, s, sumq);
    return ohara_launch_status();
  };
  // A wave a row has no barriers and a quarter of the workgroups, a workgroup a row a quarter of the chain.  us, a wave / a workgroup a row, one set and three:
  // 256 wide, 1024, 4096 rows 4.8 5.5, 6.0 8.5 / 6.2 8.2, 12.3 18.7;  1024, 100, 1024, 4096 rows 5.0 5.9, 5.2 6.4, 7.7 13.4 / 5.0 5.5, 6.4 8.9, 13.0
  // 20.9;  2816, 300, 1024, 4096 rows 6.5 10.2, 6.8 11.2, 15.1 28.6 / 6.1 8.7, 8.2 13.2, 19.9 35.3;  4096, 1024, 4096 rows 8.0 13.8, 20.5 37.0 / 8.7 14.0,
  // 22.1 38.0;  5632, 4096 rows 36 65 / 27 48.
  if (K <= 512) return go(row_quant_kernel<64, 1, GATED>, 4);
  if (K <= 1024 && rows >= 300) return go(row_quant_kernel<64, 2, GATED>, 4);
  if (K <= 2048 && rows >= 1024) return go(row_quant_kernel<64, 4, GATED>, 4);
  if (K <= 3072 && rows >= 1024) return go(row_quant_kernel<64, 6, GATED>, 4);
  if (K <= 2048) return go(row_quant_kernel<256, 1, GATED>, 1);
  return K <= 4096 ? go(row_quant_kernel<256, 2, GATED>, 1) : go(row_quant_kernel<256, 3, GATED>, 1);
}

struct BitArgs {
  const uint4* wp;       // packed ternary
  float gamma;
  const bf16_t* x;       // FUSED: (B, K) bf16 activations
  int ldx;
  const bf16_t* nw;      // FUSED: BitLinear's RMSNorm weight
  const bf16_t* pre_w;   // FUSED, optional: weight of a block-level RMSNorm applied before it
  float eps;
  const int8_t* q;       // !FUSED: (B, ldq) int8
  int ldq;
  const float* s;        // !FUSED
  const int* sumq;       // !FUSED
  int B, N, K;
  bf16_t* out;
  int ldo;
  const bf16_t* resid;
  int ldr;
  int32_t* acc_out;      // optional (B, N) raw accumulators
  int ldacc;
};

// One workgroup, one 16-row strip of one BitLinear: quantise the activation rows into LDS (FUSED)
// or copy them in, stream the strip's packed weights, leave the int32 accumulators (codes T+1, so
// sum q still to subtract) of the strip in wave 0.  Returns false in waves 1..3.  Every thread of
// the workgroup must call it; LDS is reusable after the call's last barrier.
template <int BT, bool FUSED>
__device__ __forceinline__ bool bitlinear_strip(const BitArgs& a, int strip, unsigned char* smem, i32x4* acc,
                                                float** s_s_out, int** s_sum_out) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int KC = (a.K + 255) >> 8;      // 256-column chunks
  const int Kp = KC << 8;
  const int ldq = Kp + 16;              // LDS row stride in bytes (16-byte skew against bank conflicts)
  int8_t* xq = reinterpret_cast<int8_t*>(smem);
  float* s_s = reinterpret_cast<float*>(smem + (((size_t)BT * 16 * ldq + 255) & ~(size_t)255));
  int* s_sum = reinterpret_cast<int*>(s_s + BT * 16);
  int* red = s_sum + BT * 16;           // [3][BT][64][4]
  bf16_t* stage = reinterpret_cast<bf16_t*>(red + 3 * BT * 64 * 4);  // [4][Kp] rows being quantised (FUSED)

  // the first weights of this wave are requested before the activations are prepared
  const int per = (KC + 3) >> 2;
  const int c0 = wave * per, c1 = min(KC, c0 + per);
  const uint4* wrow = a.wp + (size_t)strip * KC * 64 + lane;
  constexpr int CH = 6;
  uint4 wpre[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) wpre[c] = (c0 + c < c1) ? ldg16_nt(wrow + (size_t)(c0 + c) * 64) : make_uint4(0, 0, 0, 0);

  // ---- activations -> int8 rows in LDS ---------------------------------------------------
  // rows beyond B and columns beyond K must read as zero; rows < B are overwritten up to K below
  {
    const int p16 = ldq / 16;
    const int kfull = a.K >> 4;  // 16-byte pieces wholly below K
    for (int i = tid; i < BT * 16 * p16; i += 256) {
      const int r = i / p16, c = i - r * p16;
      if (r >= a.B || c >= kfull) reinterpret_cast<uint4*>(xq)[i] = make_uint4(0, 0, 0, 0);
    }
  }
  __syncthreads();
  if (FUSED && a.B == 1) {
    const QuantOut o = block_quant_row(a.x, a.pre_w, a.nw, a.K, a.eps, xq, stage, reinterpret_cast<float*>(red));
    if (tid == 0) {
      s_s[0] = o.s;
      s_sum[0] = o.sumq;
    }
  } else if (FUSED) {
    for (int b = wave; b < a.B; b += 4) {
      const QuantOut o = wave_quant_row(a.x + (size_t)b * a.ldx, a.pre_w, a.nw, a.K, a.eps, xq + (size_t)b * ldq,
                                        stage + (size_t)wave * Kp);
      if (lane == 0) {
        s_s[b] = o.s;
        s_sum[b] = o.sumq;
      }
    }
  } else {
    const int n16 = (a.K + 15) >> 4;
    for (int i = tid; i < a.B * n16; i += 256) {
      const int b = i / n16, c = i - b * n16;
      reinterpret_cast<uint4*>(xq + (size_t)b * ldq)[c] = ldg16(a.q + (size_t)b * a.ldq + c * 16);
    }
    for (int b = tid; b < a.B; b += 256) {
      s_s[b] = a.s[b];
      s_sum[b] = a.sumq[b];
    }
  }
  __syncthreads();

  // ---- weight stream -----------------------------------------------------------------------
#pragma unroll
  for (int t = 0; t < BT; ++t) acc[t] = (i32x4){0, 0, 0, 0};
  for (int cb = c0; cb < c1; cb += CH) {
    uint4 wv[CH];
    if (cb == c0) {
#pragma unroll
      for (int c = 0; c < CH; ++c) wv[c] = wpre[c];
    } else {
#pragma unroll
      for (int c = 0; c < CH; ++c) wv[c] = (cb + c < c1) ? ldg16_nt(wrow + (size_t)(cb + c) * 64) : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (cb + c >= c1) continue;
      const uint32_t dw[4] = {wv[c].x, wv[c].y, wv[c].z, wv[c].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        i32x4 av;
        av[0] = (int)(dw[j] & 0x03030303u);
        av[1] = (int)((dw[j] >> 2) & 0x03030303u);
        av[2] = (int)((dw[j] >> 4) & 0x03030303u);
        av[3] = (int)((dw[j] >> 6) & 0x03030303u);
        const int k0 = ((cb + c) << 8) + 64 * j + 16 * g;
#pragma unroll
        for (int t = 0; t < BT; ++t) {
          const uint4 xv = *reinterpret_cast<const uint4*>(xq + (size_t)(m + 16 * t) * ldq + k0);
          i32x4 bv;
          bv[0] = (int)xv.x; bv[1] = (int)xv.y; bv[2] = (int)xv.z; bv[3] = (int)xv.w;
          acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, acc[t], 0, 0, 0);
        }
      }
    }
  }
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[(((wave - 1) * BT + t) * 64 + lane) * 4 + i] = acc[t][i];
  }
  __syncthreads();
  *s_s_out = s_s;
  *s_sum_out = s_sum;
  if (wave != 0) return false;
#pragma unroll
  for (int t = 0; t < BT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      acc[t][i] += red[((0 * BT + t) * 64 + lane) * 4 + i] + red[((1 * BT + t) * 64 + lane) * 4 + i] +
                   red[((2 * BT + t) * 64 + lane) * 4 + i];
  return true;
}

// y = bf16((float(acc - sum q) / s) * gamma): the four outputs of one MFMA fragment (bitnet.py:58-59)
__device__ __forceinline__ void bit_scale4(const i32x4& acc, int sq, float s, float gamma, int* ai, float* y) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    ai[i] = acc[i] - sq;  // codes are T+1
    y[i] = rbf(__fmul_rn(__fdiv_rn((float)ai[i], s), gamma));
  }
}

template <int BT, bool FUSED>
__global__ __launch_bounds__(256) void bitlinear_kernel(BitArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int strip = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, g = lane >> 4;
  i32x4 acc[BT];
  float* s_s;
  int* s_sum;
  if (!bitlinear_strip<BT, FUSED>(a, strip, smem, acc, &s_s, &s_sum)) return;
  const int r0 = strip * 16 + 4 * g;
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    const int b = m + 16 * t;
    if (b >= a.B) continue;
    int ai[4];
    float y[4];
    bit_scale4(acc[t], s_sum[b], s_s[b], a.gamma, ai, y);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = r0 + i;
      if (n >= a.N) continue;
      if (a.acc_out) a.acc_out[(size_t)b * a.ldacc + n] = ai[i];
      float v = y[i];
      if (a.resid) v = bf2f(a.resid[(size_t)b * a.ldr + n]) + v;
      a.out[(size_t)b * a.ldo + n] = f2bf(v);
    }
  }
}

// ---- fused groups of BitLinears that share their input row ---------------------------------------
// Q/K/V (bitnet.py:70-95 swaps attn.query/key/value; each keeps its own norm weight and scale, so
// each strip quantises the row with its projection's norm): one launch over the strips of all three,
// with rotary + cache append as the epilogue (rotary.py:55-93, kv_cache.py:104-105).
struct BitQkvArgs {
  BitArgs p[3];          // query, key, value: wp, gamma, nw, N; x / pre_w / K / B shared
  int strips[3];
  int H, Hkv, Dh, Tmax, S, pos;
  const int32_t* pos_dev;
  const bf16_t* cos;
  const bf16_t* sin;
  bf16_t* q_out;         // (B*S, H*Dh)
  bf16_t* kcache;
  bf16_t* vcache;
};

template <int BT>
__global__ __launch_bounds__(256) void bitlinear_qkv_kernel(BitQkvArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  int strip = blockIdx.x, which = 0;
  if (strip >= a.strips[0]) { strip -= a.strips[0]; which = 1; }
  if (which == 1 && strip >= a.strips[1]) { strip -= a.strips[1]; which = 2; }
  BitArgs pa = a.p[0];  // the three differ in weights, scale, norm weight and width only (no dynamic
                        // indexing of the argument block: that would copy it to scratch memory)
  if (which == 1) { pa.wp = a.p[1].wp; pa.gamma = a.p[1].gamma; pa.nw = a.p[1].nw; pa.N = a.p[1].N; }
  if (which == 2) { pa.wp = a.p[2].wp; pa.gamma = a.p[2].gamma; pa.nw = a.p[2].nw; pa.N = a.p[2].N; }
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, g = lane >> 4;
  i32x4 acc[BT];
  float* s_s;
  int* s_sum;
  if (!bitlinear_strip<BT, true>(pa, strip, smem, acc, &s_s, &s_sum)) return;
  const int r0 = strip * 16 + 4 * g;
  if (r0 >= pa.N) return;
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    const int b = m + 16 * t;  // row = sequence * S + s
    if (b >= pa.B) continue;
    int ai[4];
    float v[4];
    bit_scale4(acc[t], s_sum[b], s_s[b], pa.gamma, ai, v);
    const int seq = b / a.S;
    const int pos = (a.pos_dev ? *a.pos_dev : a.pos) + (b - seq * a.S);
    if (pos < 0 || pos >= a.Tmax) continue;
    bf16_t* o;
    if (which < 2) {
      const int d = r0 % a.Dh;
      const bf16_t* cs = a.cos + (size_t)pos * (a.Dh >> 1) + (d >> 1);
      const bf16_t* sn = a.sin + (size_t)pos * (a.Dh >> 1) + (d >> 1);
#pragma unroll
      for (int pr = 0; pr < 2; ++pr) {
        const float c = bf2f(cs[pr]), sv = bf2f(sn[pr]);
        const float e = v[2 * pr], od = v[2 * pr + 1];
        v[2 * pr] = __fsub_rn(__fmul_rn(e, c), __fmul_rn(od, sv));
        v[2 * pr + 1] = __fadd_rn(__fmul_rn(e, sv), __fmul_rn(od, c));
      }
      o = which == 0 ? a.q_out + (size_t)b * a.H * a.Dh + r0
                     : a.kcache + (((size_t)seq * a.Tmax + pos) * a.Hkv) * a.Dh + r0;
    } else {
      o = a.vcache + (((size_t)seq * a.Tmax + pos) * a.Hkv) * a.Dh + r0;
    }
    *reinterpret_cast<uint2*>(o) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
  }
}

// gate and up (ff.gate / ff.up) for the same strip of hidden columns in one workgroup, SwiGLU as the
// epilogue: out = bf16(bf16(silu(gate)) * up) (ohara/modules/mlp.py:152).
struct BitGateUpArgs {
  BitArgs gate, up;      // out/ldo of `gate` receive the product
};

template <int BT>
__global__ __launch_bounds__(256) void bitlinear_gate_up_kernel(BitGateUpArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int strip = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int m = lane & 15, g = lane >> 4;
  i32x4 acc_g[BT], acc_u[BT];
  float yg[BT][4];
  float* s_s;
  int* s_sum;
  const bool w0 = bitlinear_strip<BT, true>(a.gate, strip, smem, acc_g, &s_s, &s_sum);
  if (w0) {
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      const int b = m + 16 * t;
      int ai[4];
      if (b < a.gate.B) bit_scale4(acc_g[t], s_sum[b], s_s[b], a.gate.gamma, ai, yg[t]);
    }
  }
  __syncthreads();  // the row statistics in LDS are about to be overwritten
  if (!bitlinear_strip<BT, true>(a.up, strip, smem, acc_u, &s_s, &s_sum)) return;
  const int r0 = strip * 16 + 4 * g;
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    const int b = m + 16 * t;
    if (b >= a.up.B) continue;
    int ai[4];
    float yu[4];
    bit_scale4(acc_u[t], s_sum[b], s_s[b], a.up.gamma, ai, yu);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r0 + i < a.gate.N) a.gate.out[(size_t)b * a.gate.ldo + r0 + i] = f2bf(rbf(silu_f(yg[t][i])) * yu[i]);
  }
}

// T (N, K) int8 in {-1,0,1} row-major -> packed layout
__global__ void pack_ternary_kernel(const int8_t* t, int n, int k, int ldt, int KC, size_t total, uint4* dst) {
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const int lane = idx & 63;
  const size_t sc = idx >> 6;
  const int chunk = (int)(sc % KC);
  const int strip = (int)(sc / KC);
  const int m = lane & 15, g = lane >> 4;
  const int row = strip * 16 + m;
  uint32_t dw[4];
  for (int j = 0; j < 4; ++j) {
    uint32_t w = 0;
    for (int r = 0; r < 4; ++r)
      for (int b = 0; b < 4; ++b) {
        const int col = chunk * 256 + 64 * j + 16 * g + 4 * r + b;
        int code = 1;  // zero weight
        if (row < n && col < k) code = (int)t[(size_t)row * ldt + col] + 1;
        w |= (uint32_t)(code & 3) << (8 * b + 2 * r);
      }
    dw[j] = w;
  }
  dst[idx] = make_uint4(dw[0], dw[1], dw[2], dw[3]);
}

// silu(gate) * up with the reference's rounding (ohara/modules/mlp.py:152)
__global__ void silu_mul_kernel(const bf16_t* gate, const bf16_t* up, bf16_t* out, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = f2bf(rbf(silu_f(bf2f(gate[i]))) * bf2f(up[i]));
}

// Rotary on q and k rows + append of k, v to the cache (ohara/embeddings_pos/rotary.py:55-93,
// ohara/modules/kv_cache.py:104-105); one workgroup per (sequence, position) row.
__global__ __launch_bounds__(256) void rope_append_kernel(bf16_t* q, const bf16_t* k, const bf16_t* v, int S, int H,
                                                          int Hkv, int D, const bf16_t* cos, const bf16_t* sin, int pos0,
                                                          const int32_t* pos_dev, bf16_t* kc, bf16_t* vc, int Tmax) {
  const int row = blockIdx.x;
  const int seq = row / S;
  const int pos = (pos_dev ? *pos_dev : pos0) + (row - seq * S);
  if (pos < 0 || (Tmax > 0 && pos >= Tmax)) return;
  const int half = D >> 1;
  const bf16_t* cs = cos + (size_t)pos * half;
  const bf16_t* sn = sin + (size_t)pos * half;
  for (int i = threadIdx.x; i < H * half; i += 256) {
    const int h = i / half, p = i - h * half;
    bf16_t* x = q + (size_t)row * H * D + (size_t)h * D + 2 * p;
    const float e = bf2f(x[0]), o = bf2f(x[1]), c = bf2f(cs[p]), s = bf2f(sn[p]);
    x[0] = f2bf(__fsub_rn(__fmul_rn(e, c), __fmul_rn(o, s)));
    x[1] = f2bf(__fadd_rn(__fmul_rn(e, s), __fmul_rn(o, c)));
  }
  // Tmax == 0: kc / vc are row buffers like k / v (the rows an int8 cache's append quantises)
  const size_t dst_row = Tmax > 0 ? (size_t)seq * Tmax + pos : (size_t)row;
  bf16_t* kd = kc + dst_row * Hkv * D;
  bf16_t* vd = vc + dst_row * Hkv * D;
  for (int i = threadIdx.x; i < Hkv * half; i += 256) {
    const int h = i / half, p = i - h * half;
    const bf16_t* x = k + (size_t)row * Hkv * D + (size_t)h * D + 2 * p;
    const float e = bf2f(x[0]), o = bf2f(x[1]), c = bf2f(cs[p]), s = bf2f(sn[p]);
    kd[h * D + 2 * p] = f2bf(__fsub_rn(__fmul_rn(e, c), __fmul_rn(o, s)));
    kd[h * D + 2 * p + 1] = f2bf(__fadd_rn(__fmul_rn(e, s), __fmul_rn(o, c)));
  }
  for (int i = threadIdx.x; i < Hkv * D; i += 256) vd[i] = v[(size_t)row * Hkv * D + i];
}

// ---- many rows ---------------------------------------------------------------------------------
// Up to three BitLinears (their own codes, weights and outputs) as one launch of the tiled product of lds_tile.h on
// v_mfma_i32_16x16x64_i8: a workgroup owns TM rows of codes x TS strips, steps of 256 columns travel straight into LDS
// (codes: 256-byte row segments with their 16-byte pieces permuted by the row, weights: one 1 KiB tile a strip), a
// wave unpacks a strip's tile into operands once for its FM row blocks.  The sums are whole numbers, so neither the tile nor the
// order shows in them.
// What bounds it: the chain of a step (barrier, reads, unpacking, products).  A layer of the 2048 x 5632 ternary model over
// 300 rows took nine to twelve launches a projection group of the kernel above, each of which quantised its rows
// again in every one of its 128 to 352 workgroups (3.0 ms a layer); quantised once and multiplied here it takes 0.13 ms.
struct TernarySet {
  const uint4* wp;
  const int8_t* q;
  const float* s;
  const int* sumq;
  float gamma;
  int N, tiles;          // columns, tiles of columns
  bf16_t* out;           // ROPE: q rows, key cache, value cache
  int ldo;
  const bf16_t* resid;
  int ldr;
  int32_t* acc_out;
  int ldacc;
};
struct TernaryArgs {
  TernarySet set[3];
  int rows, K, ldq, MT, NT;
  int wide;              // columns and leading dimensions in fours: 8-byte stores
  // ROPE
  int S, Dh, Tmax, pos;
  const int32_t* pos_dev;
  const bf16_t* cos;
  const bf16_t* sin;
};

template <int WM, int WN, int FM, int FN, int NST, bool ROPE>
__global__ __launch_bounds__(WM * WN * 64, 2) void ternary_tile_kernel(TernaryArgs a) {
  constexpr int NW = WM * WN, TM = WM * FM * 16, TS = WN * FN, XL = TM / 4, WL = TS, LPW = (XL + WL) / NW;
  constexpr int STAGE = (XL + WL) * 1024, GM = 8;
  static_assert(XL % NW == 0 && WL % NW == 0, "loads split evenly over the waves");
  extern __shared__ __align__(16) unsigned char smem[];
  const int T = a.MT * a.NT;
  const int xcd = blockIdx.x & 7, qd = blockIdx.x >> 3;
  const int base = T >> 3, rem = T & 7;
  if (qd >= base + (xcd < rem ? 1 : 0)) return;
  const int pid = xcd * base + min(xcd, rem) + qd;
  const int grp = pid / (GM * a.NT), first = grp * GM, gsz = min(GM, a.MT - first), r = pid - grp * GM * a.NT;
  const int row0 = (first + r % gsz) * TM;
  int tn = r / gsz, which = 0;
  TernarySet w = a.set[0];  // (no dynamic indexing of the argument block: that would copy it to scratch memory)
  if (tn >= w.tiles) { tn -= w.tiles; which = 1; w = a.set[1]; }
  if (which == 1 && tn >= w.tiles) { tn -= w.tiles; which = 2; w = a.set[2]; }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int m = lane & 15, g = lane >> 4;
  const int KC = (a.K + 255) >> 8, strip0 = tn * TS, nstrips = (w.N + 15) >> 4;
  const bool tail = (a.K & 255) != 0;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(OHARA_LDS unsigned char*)smem;
  const uint32_t lane16 = lane * 16;
  const char* xb = reinterpret_cast<const char*>(w.q) + (size_t)row0 * a.ldq;
  const char* wb = reinterpret_cast<const char*>(w.wp);
  uint32_t xoff[XL / NW];
  int piece[XL / NW];
#pragma unroll
  for (int i = 0; i < XL / NW; ++i) {
    const int rr = (wave + i * NW) * 4 + (lane >> 4);
    piece[i] = (lane ^ rr) & 15;
    xoff[i] = (uint32_t)((min(row0 + rr, a.rows - 1) - row0) * a.ldq + piece[i] * 16);  // rows past the end: the last row
  }
  auto issue = [&](int s, uint32_t slot) {
    const bool last = tail && s == KC - 1;  // pieces past the row's end read its last one and are multiplied as zeros
#pragma unroll
    for (int i = 0; i < XL / NW; ++i)
      load_lds16(slot + (wave + i * NW) * 1024, xb + (size_t)s * 256,
                 xoff[i] - (last ? (uint32_t)max(0, s * 256 + piece[i] * 16 - (a.ldq - 16)) : 0u));
#pragma unroll
    for (int i = 0; i < WL / NW; ++i) {
      const int t = wave + i * NW;
      load_lds16(slot + (XL + t) * 1024, wb + ((size_t)min(strip0 + t, nstrips - 1) * KC + s) * 1024, lane16);
    }
  };
  i32x4 acc[FN][FM];
#pragma unroll
  for (int u = 0; u < FN; ++u)
#pragma unroll
    for (int t = 0; t < FM; ++t) acc[u][t] = (i32x4){0, 0, 0, 0};
#pragma unroll
  for (int s = 0; s < NST - 1; ++s)
    if (s < KC) issue(s, lds0 + s * STAGE);
  const uint32_t xrd = lds0 + (wm * FM * 16 + m) * 256;
  const uint32_t wrd = lds0 + (XL + wn * FN) * 1024 + lane16;
  uint32_t so = 0, si = (NST - 1) * STAGE;
  for (int s = 0; s < KC; ++s) {
    if (NST == 2 || s + NST - 2 >= KC) wait_loads<0>();
    else wait_loads<(NST - 2) * LPW>();
    __builtin_amdgcn_s_barrier();
    if (s + NST - 1 < KC) issue(s + NST - 1, lds0 + si);
    uint32_t wv[FN][4];
#pragma unroll
    for (int u = 0; u < FN; ++u) {
      const uint4 v = lds16_at(wrd + so + u * 1024);
      wv[u][0] = v.x; wv[u][1] = v.y; wv[u][2] = v.z; wv[u][3] = v.w;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint4 xf[FM];
#pragma unroll
      for (int t = 0; t < FM; ++t) xf[t] = lds16_at(xrd + so + t * 4096 + (uint32_t)((4 * j + g) ^ m) * 16);
      if (tail && s == KC - 1) {
        const int left = a.K - (256 * s + 64 * j + 16 * g);  // codes of this piece inside the row (K: a multiple of 8)
#pragma unroll
        for (int t = 0; t < FM; ++t) {
          if (left < 16) xf[t].z = xf[t].w = 0;
          if (left < 8) xf[t].x = xf[t].y = 0;
        }
      }
#pragma unroll
      for (int u = 0; u < FN; ++u) {
        i32x4 av;
        av[0] = (int)(wv[u][j] & 0x03030303u);
        av[1] = (int)((wv[u][j] >> 2) & 0x03030303u);
        av[2] = (int)((wv[u][j] >> 4) & 0x03030303u);
        av[3] = (int)((wv[u][j] >> 6) & 0x03030303u);
#pragma unroll
        for (int t = 0; t < FM; ++t) {
          i32x4 bv;
          bv[0] = (int)xf[t].x; bv[1] = (int)xf[t].y; bv[2] = (int)xf[t].z; bv[3] = (int)xf[t].w;
          acc[u][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(av, bv, acc[u][t], 0, 0, 0);
        }
      }
    }
    so = so + STAGE == NST * STAGE ? 0 : so + STAGE;
    si = si + STAGE == NST * STAGE ? 0 : si + STAGE;
  }

  const int sbase = strip0 + wn * FN;
#pragma unroll
  for (int t = 0; t < FM; ++t) {
    const int b = row0 + wm * FM * 16 + t * 16 + m;
    if (b >= a.rows) continue;
    const float s = w.s[b];
    const int sq = w.sumq[b];
    int pos = 0;
    size_t row = (size_t)b;
    if (ROPE) {
      const int seq = b / a.S;
      pos = (a.pos_dev ? *a.pos_dev : a.pos) + (b - seq * a.S);
      if (pos < 0 || pos >= a.Tmax) continue;
      if (which > 0) row = (size_t)seq * a.Tmax + pos;
    }
#pragma unroll
    for (int u = 0; u < FN; ++u) {
      const int r0 = (sbase + u) * 16 + 4 * g;
      if (r0 >= w.N) continue;
      int ai[4];
      float v[4];
      bit_scale4(acc[u][t], sq, s, w.gamma, ai, v);
      if (ROPE) {
        if (which < 2) {
          const int d = r0 % a.Dh;
          const uint32_t c2 = *reinterpret_cast<const uint32_t*>(a.cos + (size_t)pos * (a.Dh >> 1) + (d >> 1));
          const uint32_t s2 = *reinterpret_cast<const uint32_t*>(a.sin + (size_t)pos * (a.Dh >> 1) + (d >> 1));
#pragma unroll
          for (int pr = 0; pr < 2; ++pr) {
            const float c = pr ? hi_bf(c2) : lo_bf(c2), sn = pr ? hi_bf(s2) : lo_bf(s2);
            const float e = v[2 * pr], od = v[2 * pr + 1];
            v[2 * pr] = __fsub_rn(__fmul_rn(e, c), __fmul_rn(od, sn));
            v[2 * pr + 1] = __fadd_rn(__fmul_rn(e, sn), __fmul_rn(od, c));
          }
        }
        *reinterpret_cast<uint2*>(w.out + row * w.ldo + r0) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
        continue;
      }
      if (a.wide) {
        if (w.resid) {
          const uint2 rv = *reinterpret_cast<const uint2*>(w.resid + (size_t)b * w.ldr + r0);
          v[0] = lo_bf(rv.x) + v[0]; v[1] = hi_bf(rv.x) + v[1]; v[2] = lo_bf(rv.y) + v[2]; v[3] = hi_bf(rv.y) + v[3];
        }
        *reinterpret_cast<uint2*>(w.out + (size_t)b * w.ldo + r0) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
        if (w.acc_out) {
#pragma unroll
          for (int i = 0; i < 4; ++i) w.acc_out[(size_t)b * w.ldacc + r0 + i] = ai[i];
        }
        continue;
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = r0 + i;
        if (n >= w.N) continue;
        if (w.acc_out) w.acc_out[(size_t)b * w.ldacc + n] = ai[i];
        float y = v[i];
        if (w.resid) y = bf2f(w.resid[(size_t)b * w.ldr + n]) + y;
        w.out[(size_t)b * w.ldo + n] = f2bf(y);
      }
    }
  }
}

template <int WM, int WN, int FM, int FN, int NST, bool ROPE>
int launch_ternary_tile(TernaryArgs& a, hipStream_t st) {
  constexpr int TM = WM * FM * 16, TS = WN * FN, LDS = NST * (TM / 4 + TS) * 1024;
  a.MT = (a.rows + TM - 1) / TM;
  a.NT = 0;
  for (TernarySet& s : a.set) {
    s.tiles = ((s.N + 15) / 16 + TS - 1) / TS;
    a.NT += s.tiles;
  }
  const int64_t tiles = (int64_t)a.MT * a.NT;
  if (tiles > INT32_MAX - 8) return OHARA_ESIZE;
  if (LDS > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)ternary_tile_kernel<WM, WN, FM, FN, NST, ROPE>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL((ternary_tile_kernel<WM, WN, FM, FN, NST, ROPE>), dim3((unsigned)(tiles + 7) / 8 * 8), dim3(WM * WN * 64), LDS, st, a);
  return ohara_launch_status();
}

// 64 x 64 while that leaves CUs with a tile or two, 128 x 128 (half the LDS traffic a product) for more.
template <bool ROPE>
int launch_ternary(TernaryArgs& a, hipStream_t st) {
  int64_t strips = 0;
  for (const TernarySet& s : a.set) strips += (s.N + 15) / 16;
  if (((int64_t)a.rows + 127) / 128 * ((strips + 7) / 8) >= 384) return launch_ternary_tile<2, 4, 4, 2, 2, ROPE>(a, st);
  return launch_ternary_tile<2, 2, 2, 2, 3, ROPE>(a, st);
}

// What the tiled kernel asks for: codes on 16 bytes, a tile of them addressed with 32 bits.
bool ternary_tile_ok(const int8_t* q, int ldq) { return ((uintptr_t)q & 15) == 0 && (ldq & 15) == 0 && ldq >= 16 && ldq <= (1 << 23); }

template <bool FUSED>
int launch_bit(const BitArgs& a0, hipStream_t st) {
  const int strips = (a0.N + 15) / 16;
  const int KC = (a0.K + 255) >> 8;
  const int ldq = (KC << 8) + 16;
  // rows per pass: as many 16-row tiles (4, 2 or 1) as fit the LDS with this K
  auto smem_of = [&](int btt) {
    return (((size_t)btt * 16 * ldq + 255) & ~(size_t)255) + (size_t)btt * 16 * 8 +
           (size_t)3 * btt * 64 * 4 * sizeof(int) + (FUSED ? (size_t)4 * (KC << 8) * 2 : 0);
  };
  int cap = 64;
  while (cap > 16 && smem_of(cap / 16) > 160 * 1024) cap >>= 1;
  for (int r = 0; r < a0.B; r += cap) {
    BitArgs a = a0;
    a.B = a0.B - r < cap ? a0.B - r : cap;
    if (FUSED) a.x = a0.x + (size_t)r * a0.ldx;
    else {
      a.q = a0.q + (size_t)r * a0.ldq;
      a.s = a0.s + r;
      a.sumq = a0.sumq + r;
    }
    a.out = a0.out + (size_t)r * a0.ldo;
    if (a0.resid) a.resid = a0.resid + (size_t)r * a0.ldr;
    if (a0.acc_out) a.acc_out = a0.acc_out + (size_t)r * a0.ldacc;
    const int bt = (a.B + 15) / 16;
    const int btt = bt == 3 ? 4 : bt;
    const size_t smem = smem_of(btt);
    if (smem > 160 * 1024) return OHARA_ESIZE;
    dim3 grid(strips), block(256);
#define OHARA_BIT(BTV)                                                                                   \
  do {                                                                                                   \
    if (smem > 64 * 1024)                                                                                \
      (void)hipFuncSetAttribute((const void*)bitlinear_kernel<BTV, FUSED>,                               \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);                  \
    hipLaunchKernelGGL((bitlinear_kernel<BTV, FUSED>), grid, block, smem, st, a);                        \
  } while (0)
    if (btt == 1) OHARA_BIT(1);
    else if (btt == 2) OHARA_BIT(2);
    else OHARA_BIT(4);
#undef OHARA_BIT
    const int rc = ohara_launch_status();
    if (rc) return rc;
  }
  return OHARA_OK;
}

}  // namespace

extern "C" {

int ohara_bitlinear_pack_ternary(const int8_t* t, int n, int k, int ldt, uint32_t* dst, int64_t* bytes, void* stream) {
  if (n < 1 || k < 1) return OHARA_EINVAL;
  const int KC = (k + 255) / 256;
  const size_t total = (size_t)((n + 15) / 16) * KC * 64;
  if (bytes) *bytes = (int64_t)total * 16;
  if (!dst) return OHARA_OK;
  if (!t || ldt < k) return OHARA_EINVAL;
  hipLaunchKernelGGL(pack_ternary_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, t, n,
                     k, ldt, KC, total, reinterpret_cast<uint4*>(dst));
  return ohara_launch_status();
}

int ohara_act_quant_int8(const uint16_t* x, int ldx, const uint16_t* norm_w, float eps, int rows, int k, int8_t* q,
                         int ldq, float* s, int32_t* sumq, void* stream) {
  if (!x || !norm_w || !q || !s || !sumq || rows < 1 || k < 1 || ldx < k || ldq < k) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || (ldq & 7)) return OHARA_EINVAL;  // 16-byte loads, 8-byte stores
  if (k > BL_EPL * 64) return OHARA_ESIZE;
  hipLaunchKernelGGL(act_quant_kernel, dim3((rows + 3) / 4), dim3(256), (size_t)4 * k * 2, (hipStream_t)stream, x, ldx, norm_w, rows, k,
                     eps, q, ldq, s, sumq);
  return ohara_launch_status();
}

int ohara_gemv_ternary_i8(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* wp, int n,
                          int k, float gamma, int rows, const uint16_t* resid, int ldr, uint16_t* out, int ldo,
                          int32_t* acc_out, int ldacc, void* stream) {
  if (!q || !s || !sumq || !wp || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if ((ldq & 15) || ldq < k || ldo < n || (resid && ldr < n) || (acc_out && ldacc < n)) return OHARA_EINVAL;
  BitArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp); a.gamma = gamma;
  a.q = q; a.ldq = ldq; a.s = s; a.sumq = sumq;
  a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo; a.resid = resid; a.ldr = ldr;
  a.acc_out = acc_out; a.ldacc = ldacc;
  if (rows > 12 && (k & 7) == 0 && ternary_tile_ok(q, ldq)) {  // (a few rows: a strip a workgroup, no tile of 64 for them)
    TernaryArgs t{};
    t.rows = rows; t.K = k; t.ldq = ldq;
    t.set[0].wp = a.wp; t.set[0].q = q; t.set[0].s = s; t.set[0].sumq = sumq; t.set[0].gamma = gamma; t.set[0].N = n;
    t.set[0].out = out; t.set[0].ldo = ldo; t.set[0].resid = resid; t.set[0].ldr = ldr; t.set[0].acc_out = acc_out; t.set[0].ldacc = ldacc;
    t.wide = ((n | ldo | (resid ? ldr : 0)) & 3) == 0 && (((uintptr_t)out | (uintptr_t)resid) & 7) == 0;
    return launch_ternary<false>(t, (hipStream_t)stream);
  }
  return launch_bit<false>(a, (hipStream_t)stream);
}

int ohara_act_quant_sets_int8(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, const uint16_t* const* norm_w, int sets,
                              float eps, int rows, int k, int8_t* q, int ldq, float* s, int32_t* sumq, void* stream) {
  if (!x || !norm_w || !q || !s || !sumq || rows < 1 || k < 1 || ldx < k || ldq < k || sets < 1 || sets > 3) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || (ldq & 7)) return OHARA_EINVAL;  // 16-byte loads, 8-byte stores
  if (k > BL_EPL * 64) return OHARA_ESIZE;
  QuantSets w{};
  for (int i = 0; i < sets; ++i) {
    if (!norm_w[i]) return OHARA_EINVAL;
    w.nw[i] = norm_w[i];
  }
  return launch_row_quant<false>(x, ldx, nullptr, pre_norm_w, w, sets, rows, k, eps, q, ldq, s, sumq, (hipStream_t)stream);
}

int ohara_act_quant_swiglu_int8(const uint16_t* gate, const uint16_t* up, int ld, const uint16_t* norm_w, float eps, int rows, int k, int8_t* q,
                                int ldq, float* s, int32_t* sumq, void* stream) {
  if (!gate || !up || !norm_w || !q || !s || !sumq || rows < 1 || k < 1 || ld < k || ldq < k) return OHARA_EINVAL;
  if ((k & 7) || (ld & 7) || (ldq & 7)) return OHARA_EINVAL;  // 16-byte loads, 8-byte stores
  if (k > BL_EPL * 64) return OHARA_ESIZE;
  QuantSets w{};
  w.nw[0] = norm_w;
  return launch_row_quant<true>(gate, ld, up, nullptr, w, 1, rows, k, eps, q, ldq, s, sumq, (hipStream_t)stream);
}

int ohara_gemm_ternary_sets_i8(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* const* wp,
                               const float* gamma, int sets, int n, int k, int rows, uint16_t* const* out, int ldo, void* stream) {
  if (!q || !s || !sumq || !wp || !gamma || !out || sets < 1 || sets > 3 || n < 1 || k < 1 || rows < 1 || ldo < n) return OHARA_EINVAL;
  if ((k & 7) || ldq < k || !ternary_tile_ok(q, ldq)) return OHARA_EINVAL;
  TernaryArgs t{};
  t.rows = rows; t.K = k; t.ldq = ldq;
  t.wide = ((n | ldo) & 3) == 0;
  for (int i = 0; i < sets; ++i) {
    if (!wp[i] || !out[i]) return OHARA_EINVAL;
    TernarySet& w = t.set[i];
    w.wp = reinterpret_cast<const uint4*>(wp[i]); w.gamma = gamma[i]; w.N = n; w.out = out[i]; w.ldo = ldo;
    w.q = q + (size_t)i * rows * ldq; w.s = s + (size_t)i * rows; w.sumq = sumq + (size_t)i * rows;
    t.wide = t.wide && ((uintptr_t)out[i] & 7) == 0;
  }
  return launch_ternary<false>(t, (hipStream_t)stream);
}

int ohara_gemm_ternary_qkv_rope_append(const int8_t* q, int ldq, const float* s, const int32_t* sumq, const uint32_t* const* wp,
                                       const float* gamma, int k, int batch, int seq_len, int h, int h_kv, int dh,
                                       const uint16_t* cos, const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                                       uint16_t* kcache, uint16_t* vcache, int t_max, void* stream) {
  if (!q || !s || !sumq || !wp || !gamma || !cos || !sin || !q_out || !kcache || !vcache) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || h % h_kv || dh < 4 || (dh & 3) || t_max < 1 || k < 1) return OHARA_EINVAL;
  if ((k & 7) || ldq < k || !ternary_tile_ok(q, ldq)) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  if ((int64_t)batch * seq_len > INT32_MAX) return OHARA_ESIZE;
  TernaryArgs t{};
  t.rows = batch * seq_len; t.K = k; t.ldq = ldq;
  bf16_t* outs[3] = {q_out, kcache, vcache};
  for (int i = 0; i < 3; ++i) {
    if (!wp[i]) return OHARA_EINVAL;
    TernarySet& w = t.set[i];
    w.wp = reinterpret_cast<const uint4*>(wp[i]); w.gamma = gamma[i]; w.N = (i ? h_kv : h) * dh; w.out = outs[i]; w.ldo = w.N;
    w.q = q + (size_t)i * t.rows * ldq; w.s = s + (size_t)i * t.rows; w.sumq = sumq + (size_t)i * t.rows;
  }
  t.S = seq_len; t.Dh = dh; t.Tmax = t_max; t.pos = pos; t.pos_dev = pos_dev; t.cos = cos; t.sin = sin;
  return launch_ternary<true>(t, (hipStream_t)stream);
}

int ohara_bitlinear_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, const uint16_t* norm_w, float eps,
                         const uint32_t* wp, int n, int k, float gamma, int rows, const uint16_t* resid, int ldr,
                         uint16_t* out, int ldo, int32_t* acc_out, int ldacc, void* stream) {
  if (!x || !norm_w || !wp || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if (ldx < k || ldo < n || (resid && ldr < n) || (acc_out && ldacc < n)) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7)) return OHARA_EINVAL;  // 16-byte activation loads
  if (k > BL_EPL * 64) return OHARA_ESIZE;
  BitArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp); a.gamma = gamma;
  a.x = x; a.ldx = ldx; a.nw = norm_w; a.pre_w = pre_norm_w; a.eps = eps;
  a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo; a.resid = resid; a.ldr = ldr;
  a.acc_out = acc_out; a.ldacc = ldacc;
  return launch_bit<true>(a, (hipStream_t)stream);
}

static size_t bit_smem(int rows, int k, int* btt_out) {
  const int KC = (k + 255) >> 8;
  const int ldq = (KC << 8) + 16;
  const int bt = (rows + 15) / 16;
  const int btt = bt == 3 ? 4 : bt;
  *btt_out = btt;
  return (((size_t)btt * 16 * ldq + 255) & ~(size_t)255) + (size_t)btt * 16 * 8 + (size_t)3 * btt * 64 * 4 * sizeof(int) +
         (size_t)4 * (KC << 8) * 2;
}

int ohara_bitlinear_qkv_rope_append_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, float eps, int k,
                                         const uint16_t* const* norm_w, const uint32_t* const* wp, const float* gamma,
                                         int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                                         const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                                         uint16_t* kcache, uint16_t* vcache, int t_max, void* stream) {
  if (!x || !norm_w || !wp || !gamma || !cos || !sin || !q_out || !kcache || !vcache) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || h % h_kv || dh < 4 || (dh & 3) || t_max < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  const int rows = batch * seq_len;
  if (rows > 64 || k > BL_EPL * 64) return OHARA_ESIZE;
  BitQkvArgs a{};
  const int n[3] = {h * dh, h_kv * dh, h_kv * dh};
  int total = 0;
  for (int i = 0; i < 3; ++i) {
    if (!norm_w[i] || !wp[i]) return OHARA_EINVAL;
    BitArgs& p = a.p[i];
    p.wp = reinterpret_cast<const uint4*>(wp[i]); p.gamma = gamma[i];
    p.x = x; p.ldx = ldx; p.nw = norm_w[i]; p.pre_w = pre_norm_w; p.eps = eps;
    p.B = rows; p.N = n[i]; p.K = k;
    a.strips[i] = (n[i] + 15) / 16;
    total += a.strips[i];
  }
  a.H = h; a.Hkv = h_kv; a.Dh = dh; a.Tmax = t_max; a.S = seq_len; a.pos = pos; a.pos_dev = pos_dev;
  a.cos = cos; a.sin = sin; a.q_out = q_out; a.kcache = kcache; a.vcache = vcache;
  int btt;
  const size_t smem = bit_smem(rows, k, &btt);
  if (smem > 160 * 1024) return OHARA_ESIZE;
  hipStream_t st = (hipStream_t)stream;
#define OHARA_BITQ(BTV)                                                                                     \
  do {                                                                                                      \
    if (smem > 64 * 1024)                                                                                   \
      (void)hipFuncSetAttribute((const void*)bitlinear_qkv_kernel<BTV>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)smem);                                                                 \
    hipLaunchKernelGGL((bitlinear_qkv_kernel<BTV>), dim3(total), dim3(256), smem, st, a);                   \
  } while (0)
  if (btt == 1) OHARA_BITQ(1);
  else if (btt == 2) OHARA_BITQ(2);
  else OHARA_BITQ(4);
#undef OHARA_BITQ
  return ohara_launch_status();
}

int ohara_bitlinear_gate_up_bf16(const uint16_t* x, int ldx, const uint16_t* pre_norm_w, float eps, int k, int f,
                                 const uint16_t* gate_norm_w, const uint32_t* gate_wp, float gate_gamma,
                                 const uint16_t* up_norm_w, const uint32_t* up_wp, float up_gamma, int rows,
                                 uint16_t* out, int ldo, void* stream) {
  if (!x || !gate_norm_w || !gate_wp || !up_norm_w || !up_wp || !out || rows < 1 || k < 1 || f < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k || ldo < f) return OHARA_EINVAL;
  if (rows > 64 || k > BL_EPL * 64) return OHARA_ESIZE;
  BitGateUpArgs a{};
  BitArgs* ps[2] = {&a.gate, &a.up};
  for (int i = 0; i < 2; ++i) {
    BitArgs& p = *ps[i];
    p.wp = reinterpret_cast<const uint4*>(i ? up_wp : gate_wp); p.gamma = i ? up_gamma : gate_gamma;
    p.x = x; p.ldx = ldx; p.nw = i ? up_norm_w : gate_norm_w; p.pre_w = pre_norm_w; p.eps = eps;
    p.B = rows; p.N = f; p.K = k; p.out = out; p.ldo = ldo;
  }
  int btt;
  const size_t smem = bit_smem(rows, k, &btt);
  if (smem > 160 * 1024) return OHARA_ESIZE;
  hipStream_t st = (hipStream_t)stream;
  const int strips = (f + 15) / 16;
#define OHARA_BITG(BTV)                                                                                     \
  do {                                                                                                      \
    if (smem > 64 * 1024)                                                                                   \
      (void)hipFuncSetAttribute((const void*)bitlinear_gate_up_kernel<BTV>,                                 \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);                     \
    hipLaunchKernelGGL((bitlinear_gate_up_kernel<BTV>), dim3(strips), dim3(256), smem, st, a);              \
  } while (0)
  if (btt == 1) OHARA_BITG(1);
  else if (btt == 2) OHARA_BITG(2);
  else OHARA_BITG(4);
#undef OHARA_BITG
  return ohara_launch_status();
}

int ohara_silu_mul_bf16(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t n, void* stream) {
  if (!gate || !up || !out || n < 1) return OHARA_EINVAL;
  hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, gate, up, out,
                     (size_t)n);
  return ohara_launch_status();
}

int ohara_rope_append_bf16(uint16_t* q, const uint16_t* k, const uint16_t* v, int batch, int seq_len, int h, int h_kv,
                           int dh, const uint16_t* cos, const uint16_t* sin, int pos, const int32_t* pos_dev,
                           uint16_t* kcache, uint16_t* vcache, int t_max, void* stream) {
  if (!q || !k || !v || !cos || !sin || !kcache || !vcache) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || dh < 2 || (dh & 1) || t_max < 0) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || (t_max > 0 && pos + seq_len > t_max))) return OHARA_EINVAL;
  hipLaunchKernelGGL(rope_append_kernel, dim3(batch * seq_len), dim3(256), 0, (hipStream_t)stream, q, k, v, seq_len, h,
                     h_kv, dh, cos, sin, pos, pos_dev, kcache, vcache, t_max);
  return ohara_launch_status();
}

}  // extern "C"
