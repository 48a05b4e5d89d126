// Weight-streaming skinny GEMM for the decode projections (batch <= 64).
//
// y[b, n] = sum_k x[b, k] * W[n, k].  W is read exactly once, in a packed tile
// order whose every wave-load is one contiguous 1 KiB (64 lanes x 16 B), straight
// into the A operand of v_mfma_f32_16x16x32_bf16; the activations are the B
// operand (16 batch columns per MFMA), so batch 1..16 costs the same weight
// stream.  One workgroup (4 to 16 waves) owns one 16-row strip (group_kernel: two to
// four strips that share the normed rows; wide_kernel: whole strips per wave); the waves
// split K and their fp32 partial tiles are summed in a fixed order through LDS, so
// results do not depend on scheduling.
//
// Fusions (rounding points follow the reference's bf16 eager path):
//   prologue  RMSNorm           ohara/modules/norm.py:16-21
//   epilogue  residual add      ohara/models/llama.py:199-200
//             SwiGLU            ohara/modules/mlp.py:152
//             rotary + KV append ohara/embeddings_pos/rotary.py:55-93,
//                               ohara/modules/kv_cache.py:104-105
#include <algorithm>

#include "gemm_epilogue.h"
#include "phi_attn.h"

#include <type_traits>

namespace {

__device__ __forceinline__ float sumsq8(uint4 v) {
  float s = 0.f;
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = lo_bf(w[i]), b = hi_bf(w[i]);
    s += a * a + b * b;
  }
  return s;
}

// bf16(bf16(x * rinv) * w) on 8 packed values.
__device__ __forceinline__ uint4 norm8(uint4 xv, uint4 wv, float rinv) {
  const uint32_t xs[4] = {xv.x, xv.y, xv.z, xv.w};
  const uint32_t ws[4] = {wv.x, wv.y, wv.z, wv.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = rbf(lo_bf(xs[i]) * rinv) * lo_bf(ws[i]);
    float b = rbf(hi_bf(xs[i]) * rinv) * hi_bf(ws[i]);
    o[i] = pack_bf(a, b);
  }
  return make_uint4(o[0], o[1], o[2], o[3]);
}

// LayerNorm on 8 packed values: bf16((x - mean) * rstd * w + b), one rounding (nn.LayerNorm).
__device__ __forceinline__ uint4 lnorm8(uint4 xv, uint4 wv, uint4 bv, float mean, float rstd) {
  const uint32_t xs[4] = {xv.x, xv.y, xv.z, xv.w};
  const uint32_t ws[4] = {wv.x, wv.y, wv.z, wv.w};
  const uint32_t bs[4] = {bv.x, bv.y, bv.z, bv.w};
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = pack_bf((lo_bf(xs[i]) - mean) * rstd * lo_bf(ws[i]) + lo_bf(bs[i]),
                   (hi_bf(xs[i]) - mean) * rstd * hi_bf(ws[i]) + hi_bf(bs[i]));
  return make_uint4(o[0], o[1], o[2], o[3]);
}

__device__ __forceinline__ float sum8(uint4 v) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) s += lo_bf(w[i]) + hi_bf(w[i]);
  return s;
}

// NORM: 0 none, 1 RMSNorm (norm.py:16-21), 2 LayerNorm with bias (phi.py:132).
// NW waves per workgroup split K.  A workgroup keeps NW * CH KiB of weight loads in flight, so when
// there are too few strips to put several workgroups on every CU (few output rows, long K) 16 waves
// instead of 4 are what fills the memory pipeline.
template <int BT, int NORM, int EPI, int NW, int SP>
__device__ __forceinline__ void skinny(const GemmArgs& a, int block) {
  // k-steps whose loads are issued back to back (the many-wave variants have no norm operands to hold)
  constexpr int CH = (NORM == 0 && NW > 4) ? 10 : (BT <= 2 ? 6 : 4);
  // workgroup id -> (strip, chunk of 16*BT rows).  Ids go round-robin over the 8 XCDs; the chunks of
  // one strip get ids 8 apart, so they run on the same XCD and share its L2 copy of the weights.
  const int xcd = block & 7, local = block >> 3;
  const int strip = (local / a.ny) * 8 + xcd;
  const int rbase = (local % a.ny) * 16 * BT;
  if (strip >= a.nstrips) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5;
  const int per_wave = (KS + NW - 1) / NW;
  const int j0 = wave * per_wave;
  const int j1 = min(KS, j0 + per_wave);

  __shared__ float red[NW - 1][BT][64][4];
  __shared__ float ssq[NW][BT * 16];
  __shared__ float ssum[NORM == 2 ? NW : 1][BT * 16];

  // A launch of this kernel is a chain of memory round trips - the rows for the norm, the weights, what the epilogue
  // adds or rotates with - and lasts about as long as their sum (5-8 us for 1-9 MB at 32 rows).  What does not depend
  // on anything computed here is therefore requested first: the epilogue's operands (wave 0 finishes the fragments),
  // and, where a wave's share of K is at most SP k-steps (K <= 1024 with four waves), the rows, the norm weights and
  // the weights of the whole share in one go - the rows arrive first (loads return in order), the norm's sums run
  // while the weights are still on their way, and the rows are not fetched a second time.
  // (A request past the share costs as much as one that is used: SP is 6 where the share is.)
  const bool pre_ok = ((a.N | a.ldo | a.ldr | a.ldr2) & 3) == 0 && EPI != EPI_STORE && EPI != EPI_SWIGLU && EPI != EPI_SOFTCAP && EPI != EPI_GELU_LOOKUP && EPI != EPI_GLU;
  EpiPre ep[BT];
  if (wave == 0 && pre_ok) {
#pragma unroll
    for (int t = 0; t < BT; ++t) gemm_epilogue_fetch<EPI>(a, rbase + m + 16 * t, strip, g, ep[t]);
  }
  const uint4* wrow = a.wp + (size_t)strip * KS * 64 + lane;
  f32x4 acc[BT];
#pragma unroll
  for (int t = 0; t < BT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  float rinv[BT], mean[BT];
  if (NORM == 1 && BT == 1 && per_wave <= SP) {
    uint4 xv[SP], nw[SP], wv[SP];
    const int b = rbase + m;
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const int k0 = 32 * (j0 + c) + 8 * g;
      const bool in = j0 + c < j1 && b < a.B && k0 < a.K;
      xv[c] = ldg16(a.x + (in ? (size_t)b * a.ldx + k0 : (size_t)0));
    }
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const int k0 = 32 * (j0 + c) + 8 * g;
      nw[c] = ldg16(a.norm_w + (j0 + c < j1 && k0 < a.K ? k0 : 0));
    }
#pragma unroll
    for (int c = 0; c < SP; ++c) wv[c] = ldg16_nt(wrow + (size_t)min(j0 + c, KS - 1) * 64);
    __builtin_amdgcn_sched_barrier(0);
    float part = 0.f;
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const int k0 = 32 * (j0 + c) + 8 * g;
      if (j0 + c < j1 && b < a.B && k0 < a.K) part += sumsq8(xv[c]);
    }
    part = lanes_sum<16, 16>(part);
    part = lanes_sum<32, 32>(part);
    if (g == 0) ssq[wave][m] = part;
    __syncthreads();
    float tot = ssq[0][m];
#pragma unroll
    for (int w = 1; w < NW; ++w) tot += ssq[w][m];
    rinv[0] = 1.0f / sqrtf(tot / (float)a.K + a.eps);
    mean[0] = 0.f;
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const int k0 = 32 * (j0 + c) + 8 * g;
      const bool in = j0 + c < j1 && b < a.B && k0 < a.K;
      const bool inw = j0 + c < j1;
      const uint4 xn = in ? norm8(xv[c], (k0 < a.K) ? nw[c] : make_uint4(0, 0, 0, 0), rinv[0]) : make_uint4(0, 0, 0, 0);
      if (inw)
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c]), __builtin_bit_cast(bf16x8, xn),
                                                         acc[0], 0, 0, 0);
    }
  } else {
  if (NORM) {
    float part[BT], psum[BT];
#pragma unroll
    for (int t = 0; t < BT; ++t) part[t] = psum[t] = 0.f;
    // CH k-steps per round, all loads of a round issued before the first is used (one round trip
    // per round instead of one per k-step); pieces outside the matrix read element 0 and are not added
    for (int j = j0; j < j1; j += CH) {
      uint4 xv[CH][BT];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int k0 = 32 * (j + c) + 8 * g;
#pragma unroll
        for (int t = 0; t < BT; ++t) {
          const int b = rbase + m + 16 * t;
          const bool in = j + c < j1 && b < a.B && k0 < a.K;
          xv[c][t] = ldg16(a.x + (in ? (size_t)b * a.ldx + k0 : (size_t)0));
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int k0 = 32 * (j + c) + 8 * g;
#pragma unroll
        for (int t = 0; t < BT; ++t) {
          const int b = rbase + m + 16 * t;
          if (j + c < j1 && b < a.B && k0 < a.K) {
            part[t] += sumsq8(xv[c][t]);
            if (NORM == 2) psum[t] += sum8(xv[c][t]);
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      float p = part[t];
      p = lanes_sum<16, 16>(p);
      p = lanes_sum<32, 32>(p);
      if (g == 0) ssq[wave][16 * t + m] = p;
      if (NORM == 2) {
        float q = psum[t];
        q = lanes_sum<16, 16>(q);
        q = lanes_sum<32, 32>(q);
        if (g == 0) ssum[wave][16 * t + m] = q;
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      float tot = ssq[0][16 * t + m];
#pragma unroll
      for (int w = 1; w < NW; ++w) tot += ssq[w][16 * t + m];
      if (NORM == 2) {
        // mean and biased variance from the sums of x and x^2 (fp32; rows are O(1) activations)
        float sm = ssum[0][16 * t + m];
#pragma unroll
        for (int w = 1; w < NW; ++w) sm += ssum[w][16 * t + m];
        mean[t] = sm / (float)a.K;
        rinv[t] = 1.0f / sqrtf(fmaxf(tot / (float)a.K - mean[t] * mean[t], 0.f) + a.eps);
      } else {
        mean[t] = 0.f;
        rinv[t] = 1.0f / sqrtf(tot / (float)a.K + a.eps);
      }
    }
  }

  // A group of CH k-steps: all loads of the group (weights, norm weights, the activations of
  // every 16-row block) are issued before the first product, so their latencies overlap.
  auto group = [&](int j, int n) {  // k-steps j .. j+n-1, n <= CH
    uint4 wv[CH], nw[CH], nb[NORM == 2 ? CH : 1], xv[CH][BT];
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int k0 = 32 * (j + c) + 8 * g;
      const bool in = c < n;
      wv[c] = in ? ldg16_nt(wrow + (size_t)(j + c) * 64) : make_uint4(0, 0, 0, 0);
      nw[c] = (NORM && in && k0 < a.K) ? ldg16(a.norm_w + k0) : make_uint4(0, 0, 0, 0);
      if (NORM == 2) nb[c] = (in && k0 < a.K) ? ldg16(a.norm_b + k0) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int t = 0; t < BT; ++t) {
        const int b = rbase + m + 16 * t;
        xv[c][t] = (in && b < a.B && k0 < a.K) ? ldg16(a.x + (size_t)b * a.ldx + k0) : make_uint4(0, 0, 0, 0);
      }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
#pragma unroll
      for (int t = 0; t < BT; ++t) {
        uint4 xn = xv[c][t];
        if (NORM == 1) xn = norm8(xn, nw[c], rinv[t]);
        if (NORM == 2) {
          // rows beyond the batch and columns beyond K must stay zero (the bias would leak in)
          const bool live = rbase + m + 16 * t < a.B && 32 * (j + c) + 8 * g < a.K && c < n;
          xn = live ? lnorm8(xn, nw[c], nb[c], mean[t], rinv[t]) : make_uint4(0, 0, 0, 0);
        }
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c]),
                                                         __builtin_bit_cast(bf16x8, xn), acc[t], 0, 0, 0);
      }
    }
  };

  int j = j0;
  for (; j + CH <= j1; j += CH) group(j, CH);
  if (j < j1) group(j, j1 - j);
  }

  // Fixed-order cross-wave sum: ((w0 + w1) + w2) + w3 ...
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave - 1][t][lane][i] = acc[t][i];
  }
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int t = 0; t < BT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int w = 0; w < NW - 1; ++w) acc[t][i] += red[w][t][lane][i];
    }

#pragma unroll
  for (int t = 0; t < BT; ++t) {
    const int b = rbase + m + 16 * t;
    if (b < a.B) {
      if (pre_ok) gemm_epilogue<EPI, true>(a, b, strip, g, acc[t], ep[t]);
      else gemm_epilogue<EPI>(a, b, strip, g, acc[t]);
    }
  }
}

template <int BT, int NORM, int EPI, int NW = 4, int SP = 8>
__global__ __launch_bounds__(NW * 64) void skinny_kernel(GemmArgs a) {
  skinny<BT, NORM, EPI, NW, SP>(a, blockIdx.x);
}

// Phi's block head (EPI_PHI_IN) on rows before their LayerNorm, one or two, widths up to 256 SP: eight waves a strip, four a row's norm, which is
// layernorm_kernel's to the bit.  A wave asks for the row, the norm's weight and bias and then for its whole share of the strip, so the statistics and
// their barriers pass while the weights travel, and the norm's launch, a workgroup a row, is spared.  What it costs is every workgroup's reads of the row and
// the norm's, 15 KB beside 80 of weights; so two workgroups to a CU, which keep the row and go from strip to strip with the next one's weights ahead of them.
// us, norm and head / this in a workgroup a strip / 512 of them: 2560 x (7680 + 10240) one row 18.8 / 18.6 / 17.0 (16.4 without a norm), two 18.9 / 19.3 / 16.7; 2304 x
// (6912 + 9216) 16.7 / 15.8 / 14.7, 17.0 / 16.5 / 15.0; 2048 x (6144 + 8192) 14.7 / 14.4 / 13.5, 15.4 / 14.8 / 13.8; 640 strips of 2048 12.4 / 11.2 / 10.7.  (256: 18.1, 15.4,
// 13.4, 10.5; 400 18.8, 15.4, 13.7, 10.7.)
template <int SP>
__global__ __launch_bounds__(512, 4) void phi_in_kernel(GemmArgs a) {
  constexpr int NW = 8;
  __shared__ float red[2][NW - 1][64][4], sums[2][2][4];
  __shared__ __align__(16) bf16_t xs[2][256 * SP];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5, per_wave = (KS + NW - 1) / NW;
  const int j0 = wave * per_wave, j1 = min(KS, j0 + per_wave);
  const int r = wave >> 2, t = tid & 255, part = wave & 3;
  const bf16_t* row = a.x + (size_t)min(r, a.B - 1) * a.ldx;
  uint4 xv[2], nw[2], nb[2], wv[SP];
  int at[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) at[c] = r < a.B ? (t + 256 * c) * 8 : a.K;  // (wave-uniform: four waves have no row of one)
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (at[c] < a.K) xv[c] = ldg16(row + at[c]);
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (at[c] < a.K) {
      nw[c] = ldg16(a.norm_w + at[c]);
      nb[c] = ldg16(a.norm_b + at[c]);
    }
  EpiPre ep;
  auto ask = [&](int strip) {
    const uint4* wrow = a.wp + (size_t)strip * KS * 64 + lane;
#pragma unroll
    for (int c = 0; c < SP; ++c) wv[c] = ldg16_nt(wrow + (size_t)min(j0 + c, KS - 1) * 64);
    if (wave == 0) gemm_epilogue_fetch<EPI_PHI_IN>(a, m, strip, g, ep);
  };
  ask(blockIdx.x);
  __builtin_amdgcn_sched_barrier(0);
  float s = 0.f;
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (at[c] < a.K) {
      const uint32_t u[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) s += lo_bf(u[i]) + hi_bf(u[i]);
    }
  s = wave_sum(s);
  if (lane == 0) sums[0][r][part] = s;
  __syncthreads();
  const float mean = (((sums[0][r][0] + sums[0][r][1]) + sums[0][r][2]) + sums[0][r][3]) / (float)a.K;
  float q = 0.f;
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (at[c] < a.K) {
      const uint32_t u[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float a0 = lo_bf(u[i]) - mean, a1 = hi_bf(u[i]) - mean;
        q += a0 * a0 + a1 * a1;
      }
    }
  q = wave_sum(q);
  if (lane == 0) sums[1][r][part] = q;
  __syncthreads();
  const float var = (((sums[1][r][0] + sums[1][r][1]) + sums[1][r][2]) + sums[1][r][3]) / (float)a.K;
  const float rstd = 1.0f / sqrtf(var + a.eps);
#pragma unroll
  for (int c = 0; c < 2; ++c)
    if (at[c] < a.K) *reinterpret_cast<uint4*>(&xs[r][at[c]]) = lnorm8(xv[c], nw[c], nb[c], mean, rstd);
  __syncthreads();
  int into = 0;
  for (int strip = blockIdx.x; strip < a.nstrips; strip += gridDim.x) {
    uint4 w[SP];
#pragma unroll
    for (int c = 0; c < SP; ++c) w[c] = wv[c];
    const EpiPre e = ep;
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    if (strip + (int)gridDim.x < a.nstrips) ask(strip + gridDim.x);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const int k0 = 32 * (j0 + c) + 8 * g;
      const uint4 x = *reinterpret_cast<const uint4*>(&xs[min(m, 1)][min(k0, a.K - 8)]);
      const bool live = m < a.B && k0 < a.K;
      if (j0 + c < j1)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[c]), __builtin_bit_cast(bf16x8, live ? x : make_uint4(0, 0, 0, 0)), acc,
                                                      0, 0, 0);
    }
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) red[into][wave - 1][lane][i] = acc[i];
    }
    __syncthreads();  // (the sums of the strip after this one go elsewhere; those behind it, past its barrier)
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int w = 0; w < NW - 1; ++w) acc[i] += red[into][w][lane][i];
      }
      if (m < a.B) gemm_epilogue<EPI_PHI_IN, true>(a, m, strip, g, acc, e);
    }
    into ^= 1;
  }
}
// A wave's share is eight k-steps at least, and as many as it holds at most: wider rows and narrower ones are normed by a launch of their own, the strips by
// skinny_kernel, fewer of them a workgroup of sixteen waves each.
constexpr int PHI_IN_STEPS = 10;
static bool phi_in_norms(int rows, int d, int strips) { return rows <= 2 && d >= 2048 && d <= 256 * PHI_IN_STEPS && strips >= 400; }

// Phi's attention of single tokens beside the second product of its MLP, which does not wait for it: neither fills the chip - 352 teams of four waves,
// whose chain of round trips bounds them, and 160 strips - and one after the other they took the sum of their times.  The attention's go first: its
// chain is the longer one.  (Fewer of the product's loads in flight, 2 to 7 k-steps instead of 10, leave the times as they are.)
__global__ __launch_bounds__(1024) void phi_attn_linear_kernel(PhiAttnArgs t, GemmArgs a, int fours) {
  if ((int)blockIdx.x < fours) phi_attend<4, true>(t, blockIdx.x);
  else skinny<1, 0, EPI_BIAS, 16, 8>(a, blockIdx.x - fours);
}

// (chunks by fours of a head, merged by phi_dense_kernel)
__global__ __launch_bounds__(1024) void phi_parts_linear_kernel(PhiAttnArgs t, GemmArgs a, int fours) {
  if ((int)blockIdx.x < fours) phi_attend<4, true, true>(t, blockIdx.x);
  else skinny<1, 0, EPI_BIAS, 16, 8>(a, blockIdx.x - fours);
}
// The attention's output projection, which merges its chunks: sixteen waves a strip, each over its share of K (at most SP k-steps, parts of four heads) of
// up to ROWS rows.  Merged by the team that is last, a chunk's sums go to memory, a counter is asked, the sums come back and the row goes to memory and back:
// trips that take 2 us each while the weights of the product beside them stream (one row of 32 heads of 80 behind 700, beside 2560 x 10240: 17.1 us, without
// these trips 12.6).  The launch's end orders them for nothing; the sums come back with this product's weights, and a team's threads merge four features
// each.  What that costs is a CU's reads of everyone's sums, 2.3 us with sixteen chunks a head (126 KB), so four teams of a workgroup take chunks
// of one head and leave one sum: 0.6.  The order of the sums is the products' above.
template <int ROWS, int SP>
__global__ __launch_bounds__(1024) void phi_dense_kernel(PhiAttnArgs t, GemmArgs a) {
  constexpr int NW = 16, NCH = 4;
  __shared__ float red[NW - 1][64][4];
  __shared__ __align__(16) bf16_t xs[NW][ROWS][SP * 32];
  __shared__ __align__(16) float weight[NW][ROWS][4][NCH], part[NW][ROWS][4][NCH];
  const int strip = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5, per_wave = (KS + NW - 1) / NW;
  const int j0 = wave * per_wave, j1 = min(KS, j0 + per_wave);
  const int pos = t.pos_dev ? *t.pos_dev : t.pos;
  EpiPre ep;
  if (wave == 0) gemm_epilogue_fetch<EPI_BIAS_ADD2>(a, m, strip, g, ep);
  // lane: a chunk's {max, sum} of a row and one of the heads that the share lies in; four features, of every row and chunk (past the last: the last)
  const int D = t.D, last = (t.ns >> 2) - 1, h0 = min(32 * j0, a.K - 4) / D;
  const int prow = lane / (4 * NCH), phead = lane / NCH & 3, pc = lane & (NCH - 1);
  const float2 pair = *reinterpret_cast<const float2*>(phi_pairs(t, min(prow, a.B - 1), min(h0 + phead, t.H - 1)) + 2 * min(pc, last));
  const int f = min(32 * j0 + 4 * lane, a.K - 4), h = f / D;
  uint4 v[ROWS][NCH];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < NCH; ++c) v[r][c] = ldg16(phi_values(t, min(r, a.B - 1), h) + min(c, last) * D + (f - h * D));
  const uint4* wrow = a.wp + (size_t)strip * KS * 64 + lane;
  uint4 wv[SP];
#pragma unroll
  for (int c = 0; c < SP; ++c) wv[c] = ldg16_nt(wrow + (size_t)min(j0 + c, KS - 1) * 64);
  __builtin_amdgcn_sched_barrier(0);
  const int ns = (max(pos, 0) / phi_chunk(max(pos, 0), t.ns) >> 2) + 1;
  {
    const bool in = pc < ns;
    float M = in ? pair.x : PHI_LOWEST;
#pragma unroll
    for (int x = 1; x < NCH; x *= 2) M = fmaxf(M, __shfl_xor(M, x));
    const float wg = expf(pair.x - M);
    if (prow < ROWS) {
      weight[wave][prow][phead][pc] = in ? wg : -1.f;  // (negative: not counted, whatever lies there)
      part[wave][prow][phead][pc] = in ? wg * pair.y : 0.f;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    float num[4] = {0.f, 0.f, 0.f, 0.f}, den = 0.f;
    const float *wg = weight[wave][r][min(h - h0, 3)], *pt = part[wave][r][min(h - h0, 3)];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const float w = wg[c];
      const bool in = !(w < 0.f);
      const uint32_t u[4] = {v[r][c].x, v[r][c].y, v[r][c].z, v[r][c].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) num[i] += in ? w * __uint_as_float(u[i]) : 0.f;
      den += pt[c];
    }
    if (lane < 8 * SP) *reinterpret_cast<uint2*>(&xs[wave][r][4 * lane]) = make_uint2(pack_bf(num[0] / den, num[1] / den), pack_bf(num[2] / den, num[3] / den));
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < SP; ++c) {
    const bool live = m < a.B && 32 * (j0 + c) + 8 * g < a.K;
    uint4 x = *reinterpret_cast<const uint4*>(&xs[wave][min(m, ROWS - 1)][32 * c + 8 * g]);
    x = live ? x : make_uint4(0, 0, 0, 0);
    if (j0 + c < j1) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c]), __builtin_bit_cast(bf16x8, x), acc, 0, 0, 0);
  }
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave - 1][lane][i] = acc[i];
  }
  __syncthreads();
  if (wave) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int w = 0; w < NW - 1; ++w) acc[i] += red[w][lane][i];
  }
  if (m < a.B) gemm_epilogue<EPI_BIAS_ADD2, true>(a, m, strip, g, acc, ep);
}

// Rows without a norm, K up to 6144: a wave's share of K is at most CH k-steps, all of them requested before anything waits.  Above, rounds
// of six cost a round trip each; and a request costs what it costs whether its data are used, so CH is the share, rounded up to even.
// H = 2: a workgroup takes half a strip (eight columns, in both halves of the product's sixteen), where strips leave CUs idle.
// The sums are skinny_kernel's with as many waves.  us a call, from a graph with weights in HBM, skinny_kernel with four waves / this with H = 1
// / H = 2, at 1, 8, 16, 32 and 64 rows (four waves up to K 3072, then eight):
//   1024 x 512   3.16 3.42 3.54 3.57 3.63 / 2.68 2.87 3.07 3.06 3.06
//    768 x 768   2.81 3.27 3.64 3.70 3.75 / 2.73 3.25 3.63 3.65 3.64 / 2.93 3.30 3.68 3.75 4.61
//   1024 x 1024  3.77 4.15 4.40 4.38 4.38 / 3.10 3.33 3.69 3.69 3.71 / 3.19 3.35 3.69 3.73 4.90
//   2048 x 2048  5.31 5.82 6.35 6.35 8.20 / 4.05 4.43 5.21 5.18 7.80 / 4.11 4.31 5.01 7.21 12.1
//    768 x 3072  5.48 6.54 7.38 7.34 7.23 / 4.59 5.50 6.68 6.64 6.56 / 4.67 5.11 6.29 6.43 9.67
//   1024 x 4096  7.00 8.10 9.04 8.93 8.89 / 5.18 6.32 7.92 7.80 7.76 / 5.24 5.94 7.53 7.65 13.3
//   2048 x 5632  9.64 10.7 11.5 11.2 17.9 / 8.19 8.43 10.8 10.3 18.2 / 7.73 7.37 9.47 16.9 31.4
//   4096 x 2048  6.33 6.60 6.76 8.71 14.2 / 4.99 5.10 5.77 8.14 12.8;  4096 x 4096  8.90 9.72 10.0 14.5 24.6 / 7.55 7.64 8.94 14.7 26.7
// Sixteen waves are no faster (768 x 3072 4.59 5.68 7.04 6.87 6.75, 2048 x 5632 9.08 10.6 13.2 13.2 22.9).
template <int EPI, int H, int NW, int CH>
__global__ __launch_bounds__(NW * 64) void once_kernel(GemmArgs a) {
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int part = (local / a.ny) * 8 + xcd, strip = part / H, half = part % H;
  const int rbase = (local % a.ny) * 16;
  if (strip >= a.nstrips) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5;
  const int per_wave = (KS + NW - 1) / NW;
  const int j0 = wave * per_wave, j1 = min(KS, j0 + per_wave);
  const int b = rbase + m, q = H == 2 ? 2 * half + (g & 1) : g;  // q: which four of the strip's columns this lane finishes
  __shared__ f32x4 red[NW - 1][64];
  const bool pre_ok = ((a.N | a.ldo | a.ldr) & 3) == 0 && EPI == EPI_RESIDUAL;
  EpiPre ep;
  if (wave == 0 && pre_ok) gemm_epilogue_fetch<EPI>(a, b, strip, q, ep);
  const uint4* wrow = a.wp + (size_t)strip * KS * 64 + (H == 2 ? 16 * g + 8 * half + (m & 7) : lane);
  const bf16_t* xrow = a.x + (size_t)min(b, a.B - 1) * a.ldx;
  uint4 wv[CH], xv[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    wv[c] = ldg16_nt(wrow + (size_t)min(j0 + c, KS - 1) * 64);
    xv[c] = ldg16(xrow + min(32 * (j0 + c) + 8 * g, a.K - 8));
  }
  __builtin_amdgcn_sched_barrier(0);
  f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < CH; ++c) {
    const uint4 xn = 32 * (j0 + c) + 8 * g < a.K ? xv[c] : make_uint4(0, 0, 0, 0);
    if (j0 + c < j1) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c]), __builtin_bit_cast(bf16x8, xn), acc, 0, 0, 0);
  }
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int w = 0; w < NW - 1; ++w) acc += red[w][lane];
  if (g >= 4 / H || b >= a.B) return;
  if (pre_ok) gemm_epilogue<EPI, true>(a, b, strip, q, acc, ep);
  else gemm_epilogue<EPI>(a, b, strip, q, acc);
}

// Normed rows against 257 to 1024 strips, K <= 2048: S strips a workgroup, as many as make about one workgroup a CU of them.
// Above, every strip's workgroup norms the rows again (48 vector instructions a lane and k-step: 704 strips at 32 rows kept the
// chip busy for half of the launch) and its loads come in rounds.  Here NW waves split K so far that a wave's share is at
// most SP k-steps: rows, norm weights and the weights of all S strips are requested before anything waits, and a normed
// fragment is used S times.  The waves' sums meet in LDS and are added in the order of the waves, a wave to a fragment.
template <int BT, int EPI, int S, int NW, int SP>
__global__ __launch_bounds__(NW * 64) void group_kernel(GemmArgs a) {
  extern __shared__ __align__(16) unsigned char group_smem[];
  f32x4(*red)[S * BT][64] = reinterpret_cast<f32x4(*)[S * BT][64]>(group_smem);
  __shared__ float ssq[NW][BT * 16];
  const int strip0 = blockIdx.x * S, rbase = blockIdx.y * 16 * BT;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5;
  const int per_wave = (KS + NW - 1) / NW;
  const int j0 = wave * per_wave, j1 = min(KS, j0 + per_wave);

  uint4 xv[SP][BT], nw[SP], wv[SP][S];
#pragma unroll
  for (int c = 0; c < SP; ++c) {
    const int k0 = 32 * (j0 + c) + 8 * g;
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      const int b = rbase + m + 16 * t;
      const bool in = j0 + c < j1 && b < a.B && k0 < a.K;
      xv[c][t] = ldg16(a.x + (in ? (size_t)b * a.ldx + k0 : (size_t)0));
    }
  }
#pragma unroll
  for (int c = 0; c < SP; ++c) {
    const int k0 = 32 * (j0 + c) + 8 * g;
    nw[c] = ldg16(a.norm_w + (j0 + c < j1 && k0 < a.K ? k0 : 0));
  }
#pragma unroll
  for (int u = 0; u < S; ++u)
#pragma unroll
    for (int c = 0; c < SP; ++c)
      wv[c][u] = ldg16_nt(a.wp + ((size_t)min(strip0 + u, a.nstrips - 1) * KS + min(j0 + c, KS - 1)) * 64 + lane);
  const bool pre_ok = EPI == EPI_ROPE && ((a.N | a.ldo) & 3) == 0;
  EpiPre ep;
  if (pre_ok && wave < S * BT) gemm_epilogue_fetch<EPI>(a, rbase + m + 16 * (wave % BT), min(strip0 + wave / BT, a.nstrips - 1), g, ep);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    float part = 0.f;
#pragma unroll
    for (int c = 0; c < SP; ++c)
      if (j0 + c < j1 && rbase + m + 16 * t < a.B && 32 * (j0 + c) + 8 * g < a.K) part += sumsq8(xv[c][t]);
    part = lanes_sum<32, 32>(lanes_sum<16, 16>(part));
    if (g == 0) ssq[wave][16 * t + m] = part;
  }
  __syncthreads();
  // (uniform) what stands in for k-steps past the share: an infinite weight times zero would be a NaN.  A branch around it costs nothing,
  // but where the registers are full it spills ten more (11264 x 2048 at 32 rows: 16.1 us without, 18.3 with the branch, 16.2 with masks
  // alone; 16000 x 2048 at 1 row: 14.2, 14.2, 14.6).
  constexpr bool TIGHT = NW == 16 && S * BT * SP >= 24;
  if (TIGHT || j1 - j0 < SP) {
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const uint32_t in = j0 + c < j1 ? ~0u : 0u;
#pragma unroll
      for (int u = 0; u < S; ++u) wv[c][u] = make_uint4(wv[c][u].x & in, wv[c][u].y & in, wv[c][u].z & in, wv[c][u].w & in);
    }
  }
  f32x4 acc[S][BT];
#pragma unroll
  for (int t = 0; t < BT; ++t) {
    float tot = ssq[0][16 * t + m];
#pragma unroll
    for (int w = 1; w < NW; ++w) tot += ssq[w][16 * t + m];
    const float rinv = 1.0f / sqrtf(tot / (float)a.K + a.eps);
#pragma unroll
    for (int u = 0; u < S; ++u) acc[u][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < SP; ++c) {
      const bool in = j0 + c < j1 && rbase + m + 16 * t < a.B && 32 * (j0 + c) + 8 * g < a.K;
      const uint4 xn = in ? norm8(xv[c][t], nw[c], rinv) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int u = 0; u < S; ++u)
        acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c][u]), __builtin_bit_cast(bf16x8, xn),
                                                            acc[u][t], 0, 0, 0);
    }
  }
#pragma unroll
  for (int u = 0; u < S; ++u)
#pragma unroll
    for (int t = 0; t < BT; ++t) red[wave][u * BT + t][lane] = acc[u][t];
  __syncthreads();
  if (wave >= S * BT) return;
  const int strip = strip0 + wave / BT, b = rbase + m + 16 * (wave % BT);
  f32x4 sum = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) sum += red[w][wave][lane];
  if (strip >= a.nstrips || b >= a.B) return;
  if (pre_ok) gemm_epilogue<EPI, true>(a, b, strip, g, sum, ep);
  else gemm_epilogue<EPI>(a, b, strip, g, sum);
}

template <int BT, int EPI, int S, int NW, int SP>
int launch_group_s(const GemmArgs& a, hipStream_t st) {
  static_assert(S * BT <= NW, "a wave to a fragment");
  constexpr int LDS = NW * S * BT * 1024;
  if (LDS > 60 * 1024)
    (void)hipFuncSetAttribute((const void*)group_kernel<BT, EPI, S, NW, SP>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS);
  hipLaunchKernelGGL((group_kernel<BT, EPI, S, NW, SP>), dim3((a.nstrips + S - 1) / S, (a.B + 16 * BT - 1) / (16 * BT)), dim3(NW * 64), LDS, st, a);
  return ohara_launch_status();
}
template <int BT, int EPI, int NW, int SP>
int launch_group_nw(const GemmArgs& a, hipStream_t st) {
  switch ((a.nstrips + 255) / 256) {
    case 2: return launch_group_s<BT, EPI, 2, NW, SP>(a, st);
    case 3: return launch_group_s<BT, EPI, 3, NW, SP>(a, st);
    default: return launch_group_s<NW == 16 ? 1 : BT, EPI, 4, NW, SP>(a, st);  // (four strips and 32 rows at once do not fit sixteen waves' registers)
  }
}
// The waves' shares: three k-steps or four, and no request past them: 6144 x 768, 1, 16, 32 and 64 rows 4.63 4.85 6.61 9.60 us with four,
// 4.48 4.59 6.05 8.30 with three; 8192 x 1536 8.40 8.47 11.5 21.0 / 7.82 7.96 10.6 19.5.
template <int BT, int EPI>
int launch_group_bt(const GemmArgs& a, hipStream_t st) {
  if (a.K <= 1024) return a.K <= 768 ? launch_group_nw<BT, EPI, 8, 3>(a, st) : launch_group_nw<BT, EPI, 8, 4>(a, st);
  return a.K <= 1536 ? launch_group_nw<BT, EPI, 16, 3>(a, st) : launch_group_nw<BT, EPI, 16, 4>(a, st);
}
// us a call, a strip's workgroup each (four waves) / this kernel, 1, 16, 32 and 64 rows:
//   11264 x 2048  14.8 20.1 33.9 58 / 10.7 11.1 15.8 29.4      6144 x 768  5.25 6.2 7.6 11.4 / 4.48 4.6 6.05 8.3
//   8192 x 1024    6.1  6.8  9.5 15.4 / 5.4  5.4  7.6 12.9
// With fewer strips than CUs a group is one strip, and there it is no faster: 2304 x 768 3.7 4.3 5.7 7.2 / 3.8 4.2 5.6 7.8; 3072 x 2048
// with eight waves a strip 6.0 6.9 11.9 16.9 / 6.8 7.0 10.7 19.6.
bool group_applies(const GemmArgs& a, int epi, int strips) {
  return a.norm_w && (epi == EPI_STORE || epi == EPI_SWIGLU || epi == EPI_ROPE) && strips > 256 && strips <= 1024 && a.K <= 2048;
}
template <int EPI>
int launch_group(const GemmArgs& a, hipStream_t st) {  // past 32 rows, sixteen a workgroup where its K is short
  return a.B <= 16 || (a.B > 32 && a.K <= 1024) ? launch_group_bt<1, EPI>(a, st) : launch_group_bt<2, EPI>(a, st);
}

// Many strips (the vocabulary projection): the activations are the stationary operand.  Every
// workgroup normalises all rows once into LDS (up to 64 rows, zero-padded to
// 16*BT rows and 32*KS columns), then each of its 8 waves walks whole strips - full K, no
// cross-wave sum - reading the MFMA B operands from LDS, so the weights are read exactly once
// whatever the row count and the norm is computed once per workgroup, not once per strip.
constexpr int WIDE_WAVES = 8;
constexpr int WIDE_CH = 12;

template <int BT, bool NORM, int EPI>
__global__ __launch_bounds__(WIDE_WAVES * 64) void wide_kernel(GemmArgs a) {
  extern __shared__ __align__(16) unsigned char wide_smem[];
  bf16_t* xs = reinterpret_cast<bf16_t*>(wide_smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int KS = (a.K + 31) >> 5;
  const int ldxs = KS * 32 + 8;
  const int stride = gridDim.x * WIDE_WAVES;
  int strip = blockIdx.x * WIDE_WAVES + wave;
  // Two register buffers of WIDE_CH k-steps.  The first strip's are requested before the activations are staged, so the
  // weight stream starts with the kernel, but behind the request for the rows, where those fit registers: loads return in
  // order, so rows requested behind the weights wait for 24 KiB a wave before the norm can begin.  From a graph, weights in
  // HBM, 1, 16, 32 and 64 rows: 32768 x 768 12.3 13.0 14.8 19.3 us (rows behind the weights 13.3 14.0 15.9 21.6; a copy's
  // rate would take 9.9); 32000 x 2048, up to 32 rows, 26.4 26.6 28.0 (27.3 30.1 33.7, one row at a time; 25.9).
  uint4 wa[WIDE_CH], wb[WIDE_CH];
  // No branch around a load and nothing that touches the value: k-steps and strips outside the
  // matrix read a valid tile instead and are never multiplied (mul() skips k-steps >= KS, the strip
  // loop ends before a strip >= nstrips is used).  The compiler can then count the loads in flight
  // and wait for one buffer while the other fills.
  auto load = [&](uint4* w, int st, int j) {
    const uint4* wrow = a.wp + (size_t)(st < a.nstrips ? st : 0) * KS * 64 + lane;
#pragma unroll
    for (int c = 0; c < WIDE_CH; ++c) w[c] = ldg16_nt(wrow + (size_t)min(j + c, KS - 1) * 64);
  };
  auto stage = [&](auto pieces) {  // every row of this wave in 16-byte pieces of 512 columns
    constexpr int NP = decltype(pieces)::value, RPW = 16 * BT / WIDE_WAVES;
    uint4 v[RPW][NP], nwv[NP];
#pragma unroll
    for (int c = 0; c < NP; ++c) {
      const int k = lane * 8 + 512 * c;
      nwv[c] = (NORM && k < a.K) ? ldg16(a.norm_w + k) : make_uint4(0, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < RPW; ++r) {
        const int b = wave + WIDE_WAVES * r;
        v[r][c] = (b < a.B && k < a.K) ? ldg16(a.x + (size_t)b * a.ldx + k) : make_uint4(0, 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load(wa, strip, 0);
    load(wb, strip, WIDE_CH);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      const int b = wave + WIDE_WAVES * r;
      float rinv = 1.f;
      if (NORM) {
        float ss = sumsq8(v[r][0]);
#pragma unroll
        for (int c = 1; c < NP; ++c) ss += sumsq8(v[r][c]);
        rinv = 1.0f / sqrtf(wave_sum(ss) / (float)a.K + a.eps);
      }
#pragma unroll
      for (int c = 0; c < NP; ++c) {
        const int k = lane * 8 + 512 * c;
        if (k < KS * 32)
          *reinterpret_cast<uint4*>(xs + (size_t)b * ldxs + k) = NORM ? norm8(v[r][c], nwv[c], rinv) : v[r][c];
      }
    }
  };
  if (a.K <= 1024) {
    stage(std::integral_constant<int, 2>());
  } else if (BT <= 2 && a.K <= 2048) {
    stage(std::integral_constant<int, 4>());
  } else {
    load(wa, strip, 0);
    load(wb, strip, WIDE_CH);
    for (int b = wave; b < 16 * BT; b += WIDE_WAVES) {
      float rinv = 1.f;
      if (NORM && b < a.B) {
        float ss = 0.f;
        for (int k = lane * 8; k < a.K; k += 512) ss += sumsq8(ldg16(a.x + (size_t)b * a.ldx + k));
        rinv = 1.0f / sqrtf(wave_sum(ss) / (float)a.K + a.eps);
      }
      for (int k = lane * 8; k < KS * 32; k += 512) {
        uint4 v = make_uint4(0, 0, 0, 0);
        if (b < a.B && k < a.K) {
          v = ldg16(a.x + (size_t)b * a.ldx + k);
          if (NORM) v = norm8(v, ldg16(a.norm_w + k), rinv);
        }
        *reinterpret_cast<uint4*>(xs + (size_t)b * ldxs + k) = v;
      }
    }
  }
  __syncthreads();

  const bf16_t* xrow = xs + (size_t)m * ldxs + 8 * g;
  for (; strip < a.nstrips; strip += stride) {
    f32x4 acc[BT];
#pragma unroll
    for (int t = 0; t < BT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    auto mul = [&](const uint4* w, int j) {
#pragma unroll
      for (int c = 0; c < WIDE_CH; ++c) {
        if (j + c < KS) {
#pragma unroll
          for (int t = 0; t < BT; ++t) {
            const uint4 xv = *reinterpret_cast<const uint4*>(xrow + (size_t)(16 * t) * ldxs + 32 * (j + c));
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[c]),
                                                             __builtin_bit_cast(bf16x8, xv), acc[t], 0, 0, 0);
          }
        }
      }
    };
    // wa / wb hold k-steps [j, j + CH) and [j + CH, j + 2 CH) of this strip; each buffer is refilled
    // (from this strip, or from the start of the wave's next one) as soon as it has been multiplied
    for (int j = 0; j < KS; j += 2 * WIDE_CH) {
      const bool more = j + 2 * WIDE_CH < KS;
      mul(wa, j);
      if (more) load(wa, strip, j + 2 * WIDE_CH);
      else load(wa, strip + stride, 0);
      mul(wb, j + WIDE_CH);
      if (more) load(wb, strip, j + 3 * WIDE_CH);
      else load(wb, strip + stride, WIDE_CH);
    }
#pragma unroll
    for (int t = 0; t < BT; ++t) {
      const int b = m + 16 * t;
      if (b < a.B) gemm_epilogue<EPI>(a, b, strip, g, acc[t]);
    }
  }
}

template <int BT>
int launch_wide_bt(const GemmArgs& a, int epi, hipStream_t st) {
  const int KS = (a.K + 31) >> 5;
  const size_t smem = (size_t)16 * BT * (KS * 32 + 8) * sizeof(bf16_t);
  const int grid = (a.nstrips + WIDE_WAVES - 1) / WIDE_WAVES < 256 ? (a.nstrips + WIDE_WAVES - 1) / WIDE_WAVES : 256;
#define OHARA_WIDE(NORM_, EPI_)                                                                                   \
  do {                                                                                                            \
    if (smem > 64 * 1024)                                                                                         \
      (void)hipFuncSetAttribute((const void*)wide_kernel<BT, NORM_, EPI_>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                (int)smem);                                                                       \
    hipLaunchKernelGGL((wide_kernel<BT, NORM_, EPI_>), dim3(grid), dim3(WIDE_WAVES * 64), smem, st, a);           \
  } while (0)
  if (epi == EPI_STORE) {
    if (a.norm_w) OHARA_WIDE(true, EPI_STORE);
    else OHARA_WIDE(false, EPI_STORE);
  } else if (epi == EPI_SOFTCAP) {
    OHARA_WIDE(false, EPI_SOFTCAP);
  } else {
    return OHARA_EINVAL;
  }
#undef OHARA_WIDE
  return ohara_launch_status();
}

// The wide kernel serves plain and soft-capped stores of many strips whose rows fit LDS.
bool wide_applies(const GemmArgs& a, int epi, int strips) {
  const int KS = (a.K + 31) >> 5;
  const int bt = (a.B + 15) / 16;
  return (epi == EPI_STORE || epi == EPI_SOFTCAP) && strips >= 1024 && a.B <= 64 && (size_t)16 * bt * (KS * 32 + 8) * 2 <= 160 * 1024;
}

int launch_wide(const GemmArgs& a0, int epi, int strips, hipStream_t st) {
  GemmArgs a = a0;
  a.nstrips = strips;
  switch ((a.B + 15) / 16) {
    case 1: return launch_wide_bt<1>(a, epi, st);
    case 2: return launch_wide_bt<2>(a, epi, st);
    case 3: return launch_wide_bt<3>(a, epi, st);
    default: return launch_wide_bt<4>(a, epi, st);
  }
}

template <int EPI, int H, int NW, int CH>
int launch_once_as(const GemmArgs& a, hipStream_t st) {
  hipLaunchKernelGGL((once_kernel<EPI, H, NW, CH>), dim3((unsigned)((H * a.nstrips + 7) / 8 * 8 * a.ny)), dim3(NW * 64), 0, st, a);
  return ohara_launch_status();
}
template <int EPI, int H>
int launch_once_h(const GemmArgs& a, hipStream_t st) {
  const int KS = (a.K + 31) >> 5;
  if constexpr (H == 1) {  // (half strips start past K 1024)
    switch ((KS + 7) / 8 * 2) {
      case 2: return launch_once_as<EPI, H, 4, 2>(a, st);
      case 4: return launch_once_as<EPI, H, 4, 4>(a, st);
      case 6: return launch_once_as<EPI, H, 4, 6>(a, st);
      case 8: return launch_once_as<EPI, H, 4, 8>(a, st);
    }
  }
  if (KS <= 96) switch ((KS + 7) / 8 * 2) {  // four waves' shares, even
    case 10: return launch_once_as<EPI, H, 4, 10>(a, st);
    case 12: return launch_once_as<EPI, H, 4, 12>(a, st);
    case 14: return launch_once_as<EPI, H, 4, 14>(a, st);
    case 16: return launch_once_as<EPI, H, 4, 16>(a, st);
    case 18: return launch_once_as<EPI, H, 4, 18>(a, st);
    case 20: return launch_once_as<EPI, H, 4, 20>(a, st);
    case 22: return launch_once_as<EPI, H, 4, 22>(a, st);
    default: return launch_once_as<EPI, H, 4, 24>(a, st);
  }
  switch ((KS + 15) / 16 * 2) {
    case 14: return launch_once_as<EPI, H, 8, 14>(a, st);
    case 16: return launch_once_as<EPI, H, 8, 16>(a, st);
    case 18: return launch_once_as<EPI, H, 8, 18>(a, st);
    case 20: return launch_once_as<EPI, H, 8, 20>(a, st);
    case 22: return launch_once_as<EPI, H, 8, 22>(a, st);
    default: return launch_once_as<EPI, H, 8, 24>(a, st);
  }
}
// Past K 3072 while the workgroups are one to a CU (beyond, the eight waves' requests only queue: 4096 x 4096 above).
bool once_applies(const GemmArgs& a, int epi, int strips) {
  return !a.norm_w && (epi == EPI_STORE || epi == EPI_RESIDUAL) && (a.K <= 3072 || (a.K <= 6144 && strips * a.ny <= 256));
}
// Half a strip each while that is at most a workgroup to a CU; up to K 1024, and with few rows up to 4096, it gains nothing.
template <int EPI>
int launch_once(const GemmArgs& a, hipStream_t st) {
  const bool half = 2 * a.nstrips * a.ny <= 256 && a.K > 1024 && (a.B >= 8 || a.K > 4096);
  return half ? launch_once_h<EPI, 2>(a, st) : launch_once_h<EPI, 1>(a, st);
}

template <int BT, bool NORM>
int launch_epi(const GemmArgs& a, int epi, int strips, hipStream_t st) {
  dim3 grid((unsigned)((strips + 7) / 8 * 8 * a.ny)), block(256);
  // Linear-with-bias calls with a long K (2048 and up): 16 waves per workgroup.
  if (!NORM && ((epi >= EPI_BIAS && epi <= EPI_BIAS_ADD2) || epi == EPI_BIAS_XIELU) && a.K >= 2048) {
    if (strips * a.ny >= 400) {  // enough workgroups for four per CU: 8 waves each measured 5-9 % faster
      dim3 mid(512);
      switch (epi) {
        case EPI_BIAS: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS, 8>), grid, mid, 0, st, a); break;
        case EPI_BIAS_GELU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_GELU, 8>), grid, mid, 0, st, a); break;
        case EPI_BIAS_ADD2: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_ADD2, 8>), grid, mid, 0, st, a); break;
        case EPI_BIAS_XIELU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_XIELU, 8>), grid, mid, 0, st, a); break;
        default: return OHARA_EINVAL;
      }
      return ohara_launch_status();
    }
    dim3 big(1024);
    switch (epi) {
      case EPI_BIAS: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS, 16>), grid, big, 0, st, a); break;
      case EPI_BIAS_GELU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_GELU, 16>), grid, big, 0, st, a); break;
      case EPI_BIAS_ADD2: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_ADD2, 16>), grid, big, 0, st, a); break;
      case EPI_BIAS_XIELU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_XIELU, 16>), grid, big, 0, st, a); break;
      default: return OHARA_EINVAL;
    }
    return ohara_launch_status();
  }
  // Normed rows of 1025 to 2048 columns: eight waves, so that a wave's share of K is requested in one go (3072 x 2048, 1, 16, 32 and 64
  // rows: 9.0, 10.2, 13.9, 18.7 us with four, 6.0, 6.9, 11.9, 16.9 with eight), where the CUs have not more strips than that hides
  // anyway (33 and 64 rows, which wide_kernel cannot hold: 32000 x 2048 108, 155 us with four, 116, 161 with eight; 128256 x 2048 409, 596 and
  // 452, 627; 257 to 1024 strips are group_kernel's).
  if (NORM && a.K > 1024 && a.K <= 2048 && strips <= 256 && (epi == EPI_STORE || epi == EPI_ROPE)) {
    const bool six = a.K <= 1536;
    if (epi == EPI_STORE && six) hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_STORE, 8, 6>), grid, dim3(512), 0, st, a);
    else if (epi == EPI_STORE) hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_STORE, 8>), grid, dim3(512), 0, st, a);
    else if (six) hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_ROPE, 8, 6>), grid, dim3(512), 0, st, a);
    else hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_ROPE, 8>), grid, dim3(512), 0, st, a);
    return ohara_launch_status();
  }
  // Four waves' shares of at most six k-steps.  2304 x 768, 1, 16, 32 and 64 rows: 3.76 3.98 5.62 7.28 us with eight requested, 3.54 3.75 4.96
  // 6.29 with six (2304 x 1536 above, eight waves: 5.42 6.45 10.6 14.9 / 4.97 5.74 8.00 10.6).
  if (NORM && a.K <= 768 && (epi == EPI_STORE || epi == EPI_SWIGLU || epi == EPI_ROPE)) {
    if (epi == EPI_STORE) hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_STORE, 4, 6>), grid, block, 0, st, a);
    else if (epi == EPI_SWIGLU) hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_SWIGLU, 4, 6>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_ROPE, 4, 6>), grid, block, 0, st, a);
    return ohara_launch_status();
  }
  switch (epi) {
    case EPI_STORE: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_STORE>), grid, block, 0, st, a); break;
    case EPI_RESIDUAL: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_RESIDUAL>), grid, block, 0, st, a); break;
    case EPI_SWIGLU: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_SWIGLU>), grid, block, 0, st, a); break;
    case EPI_ROPE: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_ROPE>), grid, block, 0, st, a); break;
    case EPI_SOFTCAP: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_SOFTCAP>), grid, block, 0, st, a); break;  // never with a norm
    case EPI_GELU_LOOKUP: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_GELU_LOOKUP>), grid, block, 0, st, a); break;
    case EPI_BIAS_XIELU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_BIAS_XIELU>), grid, block, 0, st, a); break;
    case EPI_GLU: hipLaunchKernelGGL((skinny_kernel<BT, false, EPI_GLU>), grid, block, 0, st, a); break;
    case EPI_BIAS: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_BIAS>), grid, block, 0, st, a); break;
    case EPI_BIAS_GELU: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_BIAS_GELU>), grid, block, 0, st, a); break;
    case EPI_BIAS_ADD2: hipLaunchKernelGGL((skinny_kernel<BT, NORM, EPI_BIAS_ADD2>), grid, block, 0, st, a); break;
    default: return OHARA_EINVAL;
  }
  return ohara_launch_status();
}

// Up to 64 rows: every workgroup multiplies one strip by 16 rows; more rows are more workgroups
// per strip (the strip is then read once from HBM and again from L2), which keeps the per-wave
// register footprint and the norm work of a workgroup at the 16-row level.
int launch_chunk(const GemmArgs& a0, int epi, int strips, hipStream_t st) {
  GemmArgs a = a0;
  a.ny = (a.B + 15) / 16;
  a.nstrips = strips;
  if (a.ny > 4) return OHARA_ESIZE;
  if (epi == EPI_PHI_IN) {
    // optional LayerNorm prologue; wave count as for the Linear-with-bias calls
    dim3 grid((unsigned)((strips + 7) / 8 * 8 * a.ny));
#define OHARA_PHI_IN(NORM_)                                                                                              \
  do {                                                                                                                   \
    if (a.K < 2048) hipLaunchKernelGGL((skinny_kernel<1, NORM_, EPI_PHI_IN, 4>), grid, dim3(256), 0, st, a);             \
    else if (strips * a.ny >= 400) hipLaunchKernelGGL((skinny_kernel<1, NORM_, EPI_PHI_IN, 8>), grid, dim3(512), 0, st, a); \
    else hipLaunchKernelGGL((skinny_kernel<1, NORM_, EPI_PHI_IN, 16>), grid, dim3(1024), 0, st, a);                      \
  } while (0)
    if (a.norm_w) OHARA_PHI_IN(2);
    else OHARA_PHI_IN(0);
#undef OHARA_PHI_IN
    return ohara_launch_status();
  }
  if (group_applies(a, epi, strips)) {
    if (epi == EPI_STORE) return launch_group<EPI_STORE>(a, st);
    return epi == EPI_SWIGLU ? launch_group<EPI_SWIGLU>(a, st) : launch_group<EPI_ROPE>(a, st);
  }
  if (once_applies(a, epi, strips)) return epi == EPI_STORE ? launch_once<EPI_STORE>(a, st) : launch_once<EPI_RESIDUAL>(a, st);
  return a.norm_w ? launch_epi<1, true>(a, epi, strips, st) : launch_epi<1, false>(a, epi, strips, st);
}

// Rows beyond 64 are processed in chunks of 64 (each chunk streams the weights once).
int launch_skinny(const GemmArgs& a0, int epi, int packed_rows, hipStream_t st) {
  const int strips = packed_rows / 16;
  const int rows = a0.B;
  if (wide_applies(a0, epi, strips)) return launch_wide(a0, epi, strips, st);
  for (int r = 0; r < rows; r += 64) {
    GemmArgs a = a0;
    a.B = rows - r < 64 ? rows - r : 64;
    a.x = a0.x + (size_t)r * a0.ldx;
    if (epi == EPI_ROPE || epi == EPI_PHI_IN) {
      a.row0 = r;
    } else {
      a.out = a0.out + (size_t)r * a0.ldo;
      if (a0.resid) a.resid = a0.resid + (size_t)r * a0.ldr;
      if (a0.ids) a.ids = a0.ids + r;
      if (a0.resid2) a.resid2 = a0.resid2 + (size_t)r * a0.ldr2;
    }
    const int rc = launch_chunk(a, epi, strips, st);
    if (rc) return rc;
  }
  return OHARA_OK;
}

__global__ void pack_rows_kernel(const bf16_t* w, int n, int k, int ldw, const int32_t* perm, int n_padded,
                                 int KS, uint4* dst) {
  // one thread per (strip, kstep, lane)
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t total = (size_t)(n_padded / 16) * KS * 64;
  if (idx >= total) return;
  const int lane = idx & 63;
  const size_t sj = idx >> 6;
  const int j = (int)(sj % KS);
  const int s = (int)(sj / KS);
  const int m = lane & 15, g = lane >> 4;
  const int prow = 16 * s + m;
  const int src = perm ? perm[prow] : (prow < n ? prow : -1);
  const int k0 = 32 * j + 8 * g;
  uint16_t v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (src >= 0 && src < n && k0 + i < k) ? w[(size_t)src * ldw + k0 + i] : 0;
  dst[idx] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16));
}

// Eight columns of a row, the parts' sums added in their order.
template <int P>
__device__ __forceinline__ void merged8(const float* sums, int rows, int n, int row, int c, float (&f)[8]) {
  f32x4 lo[P], hi[P];
#pragma unroll
  for (int p = 0; p < P; ++p) {
    const float* at = sums + ((size_t)p * rows + row) * n + c;
    lo[p] = *reinterpret_cast<const f32x4*>(at);
    hi[p] = *reinterpret_cast<const f32x4*>(at + 4);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[i] = lo[0][i];
    f[4 + i] = hi[0][i];
#pragma unroll
    for (int p = 1; p < P; ++p) {
      f[i] += lo[p][i];
      f[4 + i] += hi[p][i];
    }
  }
}

// resid += the product (EPI_RESIDUAL's rounding), a row a workgroup, and its RMSNorm (ohara/modules/norm.py:16-21) where the next
// projection wants it.  n % 16 == 0, n <= 4096: at most two columns of eight a thread.
template <int P>
__global__ __launch_bounds__(256) void merge_norm_kernel(const float* sums, int rows, int n, bf16_t* resid, const bf16_t* norm_w, bf16_t* xn, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x, step = 8 * blockDim.x;
  bf16_t* x = resid + (size_t)row * n;
  uint4 v[2], w[2];
  float ss = 0.f;
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = 8 * threadIdx.x + t * step;
    if (c >= n) continue;
    float f[8];
    const uint4 r = ldg16(x + c);
    if (norm_w) w[t] = ldg16(norm_w + c);
    merged8<P>(sums, rows, n, row, c, f);
    const uint32_t u[4] = {r.x, r.y, r.z, r.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      o[i] = pack_bf(lo_bf(u[i]) + rbf(f[2 * i]), hi_bf(u[i]) + rbf(f[2 * i + 1]));
      ss = __builtin_fmaf(lo_bf(o[i]), lo_bf(o[i]), ss);
      ss = __builtin_fmaf(hi_bf(o[i]), hi_bf(o[i]), ss);
    }
    v[t] = make_uint4(o[0], o[1], o[2], o[3]);
    *reinterpret_cast<uint4*>(x + c) = v[t];
  }
  if (!norm_w) return;
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = red[0];
  for (int i = 1; i < (int)(blockDim.x >> 6); ++i) ss += red[i];
  const float rinv = 1.0f / sqrtf(ss / (float)n + eps);
  auto two = [&](uint32_t xx, uint32_t ww) { return pack_bf(rbf(lo_bf(xx) * rinv) * lo_bf(ww), rbf(hi_bf(xx) * rinv) * hi_bf(ww)); };
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int c = 8 * threadIdx.x + t * step;
    if (c < n) *reinterpret_cast<uint4*>(xn + (size_t)row * n + c) = make_uint4(two(v[t].x, w[t].x), two(v[t].y, w[t].y), two(v[t].z, w[t].z), two(v[t].w, w[t].w));
  }
}

// EPI_BIAS_ADD2 of the merged product.
template <int P>
__global__ __launch_bounds__(256) void merge_add2_kernel(GemmArgs a, const float* sums) {
  const int row = blockIdx.x;
  for (int c = 8 * threadIdx.x; c < a.N; c += 2048) {
    float f[8];
    const uint4 b = ldg16(a.bias + c), r1 = ldg16(a.resid + (size_t)row * a.ldr + c), r2 = ldg16(a.resid2 + (size_t)row * a.ldr2 + c);
    merged8<P>(sums, a.B, a.N, row, c, f);
    const uint32_t bu[4] = {b.x, b.y, b.z, b.w}, u1[4] = {r1.x, r1.y, r1.z, r1.w}, u2[4] = {r2.x, r2.y, r2.z, r2.w};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = pack_bf(rbf(lo_bf(u1[i]) + rbf(f[2 * i] + lo_bf(bu[i]))) + lo_bf(u2[i]), rbf(hi_bf(u1[i]) + rbf(f[2 * i + 1] + hi_bf(bu[i]))) + hi_bf(u2[i]));
    *reinterpret_cast<uint4*>(a.out + (size_t)row * a.ldo + c) = make_uint4(o[0], o[1], o[2], o[3]);
  }
}

}  // namespace

// Chunks of the attention beside the product in one launch; 0: two launches.  One where the product's workgroups are sixteen waves by themselves.  Such
// a workgroup has a CU to itself, and so has each four teams of the attention, on the CUs that are left: eight chunks of them at least, or all.
// Launches of their own spread the teams over all CUs, and what bounds them is what a CU takes in; so one launch costs what a CU takes in more of the
// keys and values, and gives the product's time.  The line is through 520 calls, of 512 x 2048 to 2560 x 10240 with 8 to 32 heads of 64, 80 and
// 128, 1 to 16 rows, behind 0 to 2040: 0.07 us dearer on average than the quicker of the two, 2.9 at worst (`pos >= 1750` before: 1.3 and 45, and
// in 126 of them dearer than this attention and product had been by themselves).  us, two launches / this: 2560 x 10240, 32 heads of 80, one row
// behind 40 16.6 / 11.9, 700 22.3 / 17.5, 2040 25.1 / 24.8; 2048 x 8192, 32 of 64, four rows behind 200 20.6 / 16.6, 1500 33.3 / 41.4; sixteen
// behind 1500 95 / 130; 1024 x 4096, 16 of 64, one row behind 40 10.7 / 9.9, 700 16.1 / 16.4; 512 x 2048, 8 of 64 behind 100 9.5 / 11.9.
static int phi_beside(int batch, int h, int dh, int n_split, int pos, int n, int k) {
  const int strips = (n + 15) / 16, heads = batch * h;
  const int chunks = strips < 256 ? std::min(n_split, (256 - (strips + 7) / 8 * 8) * 4 / std::max(heads, 1)) : 0;
  if (batch > 16 || k < 2048 || chunks < std::min(n_split, 8)) return 0;
  auto walk = [&](int ns) { return ns > 1 ? std::min(phi_chunk(pos, ns), pos + 1) : pos + 1; };  // positions of a team
  const int alone = walk(n_split), teams = heads * (pos / alone + 1);
  const float more = (4.f * walk(chunks) - std::max(1.f, teams * (1.f / 256)) * alone) * dh * 4.f;  // bytes a CU takes in
  return more <= 6e-3f * n * k + 20e3f ? chunks : 0;
}
bool ohara_launch_phi_attn_linear(PhiAttnArgs t, GemmArgs a, hipStream_t st, int* rc) {
  t.ns = phi_eights(t) ? phi_beside(a.B, t.H, t.D, t.ns, std::min(std::max(t.pos, 0), t.t_max - 1), a.N, a.K) : 0;
  if (!t.ns) return false;
  a.ny = 1; a.nstrips = (a.N + 15) / 16;
  const int fours = (t.B * t.H * t.ns + 31) / 32 * 8;  // (whole eights: a strip's XCD is its workgroup's number)
  hipLaunchKernelGGL(phi_attn_linear_kernel, dim3((unsigned)(fours + (a.nstrips + 7) / 8 * 8)), dim3(1024), 0, st, t, a, fours);
  *rc = ohara_launch_status();
  return true;
}

// Chunks of the attention whose fours the projection merges; 0: the calls above.  All teams and strips are on the chip at once, a workgroup to a CU, so
// one or two rows, and no more fours than the strips leave CUs.  A context of one chunk is the calls' above where they are one launch (its sums need no
// merge: the projection's costs 0.4 us), and of 256 where the product is the longer part anyway.  A team's positions bound the launch past the product's
// time, two launches spread them over all CUs: the line is through 360 calls, 2048 to 3584 wide with heads of 64 to 128, products of twice and four times the
// width, one and two rows behind 20 to 4000.  us with the projection, the calls above / this: 2560 x 10240, 32 heads of 80, one row behind 40 16.5 / 16.9, 200
// 20.3 / 17.2, 700 22.5 / 18.0, 2040 29.5 / 25.0, two rows behind 40 21.7 / 17.8, 700 29.2 / 24.4, 1200 32.0 / 30.6, 2000 35 / 49; 2048 x 8192, 32 of 64, one behind
// 700 22.2 / 16.9; 3584 x 14336, 28 of 128, one behind 400 34.5 / 26.2, 1400 37.3 / 37.1; 2048 x 4096, 16 of 128, two rows behind 3000 27.5 / 29.1.
static int phi_merged(int batch, int h, int dh, int rot, int n_split, int pos, int n, int k) {
  const int strips = (n + 15) / 16, heads = batch * h, depth = h * dh, share = ((depth + 31) / 32 + 15) / 16 * 32;
  if (batch > 2 || depth < 2048 || share > 256 || k < 2048 || strips >= 256 || (rot >> 1 & 7)) return 0;
  for (int first = 0; first < depth; first += share)  // a share's heads
    if ((std::min(first + share, depth) - 1) / dh - first / dh > 3) return 0;
  const int chunks = std::min(n_split, 16) / 4 * 4 < 4 ? 0 : 4 * std::min(std::min(n_split, 16) / 4, (256 - (strips + 7) / 8 * 8) / heads);
  if (!chunks || std::min(phi_chunk(pos, chunks), pos + 1) > 128 + k / 64 || (int64_t)heads * dh * (pos + 1) > 10500000) return 0;
  return pos >= ((int64_t)n * k <= 30000000 ? 64 : 256) || !phi_beside(batch, h, dh, n_split, pos, n, k) ? chunks : 0;
}
int ohara_launch_phi_attn_out(PhiAttnArgs t, GemmArgs a, GemmArgs out, hipStream_t st) {
  t.ns = phi_eights(t) ? phi_merged(a.B, t.H, t.D, t.rot, t.ns, std::min(std::max(t.pos, 0), t.t_max - 1), a.N, a.K) : 0;
  if (!t.ns) return OHARA_ESIZE;
  const int strips = (a.N + 15) / 16, fours = (a.B * t.H * (t.ns >> 2) + 7) / 8 * 8;  // (whole eights: a strip's XCD is its workgroup's number)
  a.ny = 1; a.nstrips = strips;
  hipLaunchKernelGGL(phi_parts_linear_kernel, dim3((unsigned)(fours + (strips + 7) / 8 * 8)), dim3(1024), 0, st, t, a, fours);
  const int rc = ohara_launch_status();
  if (rc) return rc;
  const bool five = (out.K + 31) / 32 <= 5 * 16;
  auto kernel = a.B == 1 ? (five ? phi_dense_kernel<1, 5> : phi_dense_kernel<1, 8>) : five ? phi_dense_kernel<2, 5> : phi_dense_kernel<2, 8>;
  hipLaunchKernelGGL(kernel, dim3((unsigned)strips), dim3(1024), 0, st, t, out);
  return ohara_launch_status();
}

extern "C" {

int ohara_phi_attn_out_chunks(int batch, int h, int dh, int rot, int n_split, int pos, int n, int k) {
  if (batch < 1 || h < 1 || dh < 8 || dh > 128 || (dh & 7) || rot < 2 || (rot & 1) || rot > dh || n_split < 1 || n_split > 64 || pos < 0 || n < 1 || k < 1)
    return OHARA_EINVAL;
  return (int64_t)batch * h * dh > INT32_MAX ? 0 : phi_merged(batch, h, dh, rot, n_split, pos, n, k);
}

int ohara_pack_rows_bf16(const uint16_t* w, int n, int k, int ldw, const int32_t* perm, int n_padded,
                         uint16_t* dst, int64_t* bytes, void* stream) {
  if (n < 1 || k < 1 || (n_padded < n && perm == nullptr)) return OHARA_EINVAL;
  if (n_padded % 16) return OHARA_EINVAL;
  const int KS = (k + 31) / 32;
  const int64_t total = (int64_t)(n_padded / 16) * KS * 64;
  if (bytes) *bytes = total * 16;
  if (!dst) return OHARA_OK;
  if (!w || ldw < k) return OHARA_EINVAL;
  const int threads = 256;
  const int64_t blocks = (total + threads - 1) / threads;
  hipLaunchKernelGGL(pack_rows_kernel, dim3((unsigned)blocks), dim3(threads), 0, (hipStream_t)stream, w, n, k, ldw,
                     perm, n_padded, KS, reinterpret_cast<uint4*>(dst));
  return ohara_launch_status();
}

int ohara_projection_norm_ahead(int rows, int k, int packed_rows) { return rows > 0 && k > 0 && packed_rows > 0 && ohara_norm_ahead(rows, k, packed_rows); }

int ohara_phi_attn_linear_chunks(int batch, int h, int dh, int n_split, int pos, int n, int k) {
  if (batch < 1 || h < 1 || dh < 8 || dh > 128 || n_split < 1 || n_split > 64 || pos < 0 || n < 1 || k < 1 || (int64_t)batch * h > INT32_MAX) return OHARA_EINVAL;
  return phi_beside(batch, h, dh, n_split, pos, n, k);
}

int ohara_swiglu_perm(int f, int32_t* perm_host) {
  if (f < 1 || !perm_host) return OHARA_EINVAL;
  const int fp = (f + 7) / 8 * 8;
  for (int s = 0; s < fp / 8; ++s)
    for (int g = 0; g < 4; ++g)
      for (int i = 0; i < 4; ++i) {
        const int fcol = 8 * s + 2 * g + (i & 1);
        const int src = (i < 2) ? fcol : f + fcol;
        perm_host[16 * s + 4 * g + i] = fcol < f ? src : -1;
      }
  return OHARA_OK;
}

int ohara_linear_bias_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, int rows,
                           int epilogue, const uint16_t* add1, int ld1, const uint16_t* add2, int ld2, uint16_t* out,
                           int ldo, void* stream) {
  if (!x || !wp || !bias || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;  // 16-byte activation loads
  if ((n & 3) || (ldo & 3) || ldo < n) return OHARA_EINVAL;   // 8-byte bias loads and stores
  int epi;
  switch (epilogue) {
    case OHARA_LIN_BIAS: epi = EPI_BIAS; break;
    case OHARA_LIN_BIAS_GELU: epi = EPI_BIAS_GELU; break;
    case OHARA_LIN_BIAS_ADD2: epi = EPI_BIAS_ADD2; break;
    default: return OHARA_EINVAL;
  }
  if (epi == EPI_BIAS_ADD2 && (!add1 || !add2 || (ld1 & 3) || (ld2 & 3) || ld1 < n || ld2 < n)) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx;
  a.B = rows; a.N = n; a.K = k;
  a.out = out; a.ldo = ldo; a.bias = bias;
  a.resid = add1; a.ldr = ld1; a.resid2 = add2; a.ldr2 = ld2;
  const int packed_rows = (n + 15) / 16 * 16;
  if (ohara_tiles_win(rows, k, packed_rows)) return ohara_launch_gemm_tile(a, epi, packed_rows, (hipStream_t)stream);
  return launch_skinny(a, epi, packed_rows, (hipStream_t)stream);
}

// ---- products in parts of the depth (ohara_depth_parts), merged by rows ---------------------------------------------------------
// The merge of a residual is the norm behind it too: 1 us more than that norm's launch, and as long as that where the depth is under 2048 (two
// parts: 128 x 768 3.0 / 3.2); the other one is a launch of its own, 3.  us with the norm, whole / in two parts of at least 384: 768 x 768, 64, 128,
// 192 rows 5.4 6.8 7.2 / 5.0 5.5 6.3; 1024 x 1024, 96 and 128 rows 7.3 7.4 / 5.9 6.0; 1536 x 1536, 128, 192 rows 8.9 10 / 7.8 8.8, 384 rows 11.9 / 12.1.
// Under 640 columns: the merge as beyond 2048, and parts of 512 at least (33 to 500 rows, 512 x 1280 8.4 / 6.5, 512 x 1792 9.4 / 7.4, 256 x 1536 9.0 /
// 6.9 at 96 rows).  That leaves the products of a model of at most 512 columns whose MLP is 1024 wide whole at any rows, which is what gives its prompts the same
// bits alone and side by side (there is no room for parts there); it costs them 1 us a product (512 x 1024, 128 rows 6.8 / 5.7).  Wider or
// deeper models' prompts differ between the two by the order of fp32 sums, and by their number of rows.  (Up to 32 rows a strip's workgroup over the whole
// depth is the faster one.)
static int residual_parts(int rows, int n, int k) {
  if (rows <= 32 || (n & 15) || n > 4096 || (n < 640 && k < 1024)) return 1;
  return ohara_depth_parts(rows, n, k, n >= 640 && k < 2048 ? 0.1f : 1.f);
}
static int bias_parts(int rows, int n, int k) { return rows > 32 && (n & 15) == 0 ? ohara_depth_parts(rows, n, k, 3.f) : 1; }
static int64_t parts_bytes(int parts, int rows, int n) { return parts > 1 ? (int64_t)parts * rows * n * (int64_t)sizeof(float) : 0; }

int64_t ohara_gemm_residual_norm_bytes(int rows, int n, int k) {
  if (rows < 1 || n < 1 || k < 1) return OHARA_EINVAL;
  return parts_bytes(residual_parts(rows, n, k), rows, n);
}

int ohara_gemm_residual_norm_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, int rows, uint16_t* resid, const uint16_t* norm_w,
                                  float eps, uint16_t* xn, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !wp || !resid || n < 1 || k < 1 || rows < 1 || (norm_w && !xn)) return OHARA_EINVAL;
  const int parts = residual_parts(rows, n, k);
  const bool aligned = !(((uintptr_t)x | (uintptr_t)resid | (uintptr_t)norm_w | (uintptr_t)xn | (uintptr_t)workspace) & 15) && !(ldx & 7) &&
                       ldx >= k && ldx <= OHARA_PARTS_LDX;
  if (parts > 1 && aligned && workspace && workspace_bytes >= parts_bytes(parts, rows, n)) {
    GemmArgs a{};
    a.wp = reinterpret_cast<const uint4*>(wp);
    a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k;
    float* sums = (float*)workspace;
    const int rc = ohara_launch_gemm_parts(a, n, parts, sums, (hipStream_t)stream);
    if (rc) return rc;
    const dim3 grid(rows), block(std::min(256, (n / 8 + 63) / 64 * 64));
#define OHARA_MERGE(P) hipLaunchKernelGGL(merge_norm_kernel<P>, grid, block, 0, (hipStream_t)stream, sums, rows, n, resid, norm_w, xn, eps)
    if (parts == 2) OHARA_MERGE(2);
    else if (parts == 4) OHARA_MERGE(4);
    else OHARA_MERGE(8);
#undef OHARA_MERGE
    return ohara_launch_status();
  }
  const int rc = ohara_gemm_skinny_bf16(x, ldx, wp, n, k, nullptr, eps, rows, OHARA_EPI_RESIDUAL, resid, n, resid, n, stream);
  return rc || !norm_w ? rc : ohara_rmsnorm_bf16(resid, norm_w, xn, rows, n, eps, stream);
}

int64_t ohara_linear_bias_add2_bytes(int rows, int n, int k) {
  if (rows < 1 || n < 1 || k < 1) return OHARA_EINVAL;
  return parts_bytes(bias_parts(rows, n, k), rows, n);
}

int ohara_linear_bias_add2_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, int rows, const uint16_t* add1,
                                int ld1, const uint16_t* add2, int ld2, uint16_t* out, int ldo, void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !wp || !bias || !add1 || !add2 || !out || n < 1 || k < 1 || rows < 1 || ldx < k || ld1 < n || ld2 < n || ldo < n) return OHARA_EINVAL;
  const int parts = bias_parts(rows, n, k);
  const bool aligned = !(((uintptr_t)x | (uintptr_t)bias | (uintptr_t)add1 | (uintptr_t)add2 | (uintptr_t)out | (uintptr_t)workspace) & 15) &&
                       !((ldx | ld1 | ld2 | ldo) & 7) && ldx <= OHARA_PARTS_LDX;
  if (parts == 1 || !aligned || !workspace || workspace_bytes < parts_bytes(parts, rows, n))
    return ohara_linear_bias_bf16(x, ldx, wp, n, k, bias, rows, OHARA_LIN_BIAS_ADD2, add1, ld1, add2, ld2, out, ldo, stream);
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k;
  a.bias = bias; a.resid = add1; a.ldr = ld1; a.resid2 = add2; a.ldr2 = ld2; a.out = out; a.ldo = ldo;
  float* sums = (float*)workspace;
  const int rc = ohara_launch_gemm_parts(a, n, parts, sums, (hipStream_t)stream);
  if (rc) return rc;
#define OHARA_MERGE(P) hipLaunchKernelGGL(merge_add2_kernel<P>, dim3(rows), dim3(256), 0, (hipStream_t)stream, a, sums)
  if (parts == 2) OHARA_MERGE(2);
  else if (parts == 4) OHARA_MERGE(4);
  else OHARA_MERGE(8);
#undef OHARA_MERGE
  return ohara_launch_status();
}

int ohara_phi_block_in_bf16(const uint16_t* x, int ldx, const uint16_t* ln_w, const uint16_t* ln_b, float eps,
                            const uint16_t* wp, const uint16_t* bias, int d, int ff, int batch, int seq_len, int pos,
                            const int32_t* pos_dev, uint16_t* q, int ldq, uint16_t* kcache, uint16_t* vcache, int t_max,
                            uint16_t* act, int ldact, void* stream) {
  if (!x || !wp || !bias || !q || !kcache || !vcache || !act || (ln_w && !ln_b)) return OHARA_EINVAL;
  if (d < 8 || ff < 4 || batch < 1 || seq_len < 1 || t_max < 1) return OHARA_EINVAL;
  if ((d & 15) || (ff & 3) || (ldx & 7) || ldx < d || (ldq & 3) || ldq < d || (ldact & 3) || ldact < ff) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  if (pos_dev && seq_len != 1) return OHARA_EINVAL;
  if ((int64_t)batch * seq_len > INT32_MAX) return OHARA_ESIZE;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.norm_w = ln_w; a.norm_b = ln_b; a.eps = eps;
  a.B = batch * seq_len; a.N = 3 * d + ff; a.K = d;
  a.out = q; a.ldo = ldq; a.out2 = act; a.ldo2 = ldact; a.split_n = 3 * d; a.bias = bias;
  a.S = seq_len; a.Tmax = t_max; a.pos = pos; a.pos_dev = pos_dev; a.kcache = kcache; a.vcache = vcache;
  const int packed_rows = (a.N + 15) / 16 * 16;
  if (ln_w && phi_in_norms(a.B, d, packed_rows / 16) && !(((uintptr_t)ln_w | (uintptr_t)ln_b | (uintptr_t)x) & 15)) {
    a.nstrips = packed_rows / 16;
    hipLaunchKernelGGL(phi_in_kernel<PHI_IN_STEPS>, dim3((unsigned)std::min(a.nstrips, 512)), dim3(512), 0, (hipStream_t)stream, a);
    return ohara_launch_status();
  }
  if (!ln_w && ohara_tiles_win(a.B, a.K, packed_rows)) return ohara_launch_gemm_tile(a, EPI_PHI_IN, packed_rows, (hipStream_t)stream);  // prefill
  return launch_skinny(a, EPI_PHI_IN, packed_rows, (hipStream_t)stream);
}

int ohara_phi_block_norms(int rows, int d, int ff) { return rows > 0 && d > 0 && ff > 0 && ff < (1 << 28) && phi_in_norms(rows, d, (3 * d + ff + 15) / 16); }

int ohara_gemm_softcap_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, float cap, int rows,
                            uint16_t* out, int ldo, void* stream) {
  if (!x || !wp || !out || n < 1 || k < 1 || rows < 1 || !(cap > 0.f)) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k || ldo < n) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo; a.cap = cap;
  if (rows > 64) return ohara_launch_gemm_tile(a, EPI_SOFTCAP, (n + 15) / 16 * 16, (hipStream_t)stream);
  return launch_skinny(a, EPI_SOFTCAP, (n + 15) / 16 * 16, (hipStream_t)stream);
}

int ohara_gemm_glu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, float limit, float alpha, float offset,
                        int rows, uint16_t* out, int ldo, void* stream) {
  if (!x || !wp || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k || ldo < n || ((n | ldo) & 1)) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo; a.glu = OharaGlu{limit, alpha, offset, 0};
  const int packed_rows = 2 * ((n + 7) / 8 * 8);
  if (rows > 64) return ohara_launch_gemm_tile(a, EPI_GLU, packed_rows, (hipStream_t)stream);
  return launch_skinny(a, EPI_GLU, packed_rows, (hipStream_t)stream);
}

int ohara_gemm_xielu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* bias, float above, float below,
                          int rows, uint16_t* out, int ldo, void* stream) {
  if (!x || !wp || !bias || !out || n < 1 || k < 1 || rows < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k || (n & 3) || (ldo & 3) || ldo < n) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo; a.bias = bias; a.above = above; a.below = below;
  if (rows > 64) return ohara_launch_gemm_tile(a, EPI_BIAS_XIELU, (n + 15) / 16 * 16, (hipStream_t)stream);
  return launch_skinny(a, EPI_BIAS_XIELU, (n + 15) / 16 * 16, (hipStream_t)stream);
}

int ohara_gemm_gelu_lookup_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* table, int ldt,
                                const int64_t* ids, int vocab, int rows, uint16_t* out, int ldo, void* stream) {
  if (!x || !wp || !table || !ids || !out || n < 1 || k < 1 || rows < 1 || vocab < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k || ldo < n || ldt < n || ((n | ldo | ldt) & 3)) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.B = rows; a.N = n; a.K = k; a.out = out; a.ldo = ldo;
  a.table = table; a.ldt = ldt; a.ids = ids; a.vocab = vocab;
  if (rows > 64) return ohara_launch_gemm_tile(a, EPI_GELU_LOOKUP, (n + 15) / 16 * 16, (hipStream_t)stream);
  return launch_skinny(a, EPI_GELU_LOOKUP, (n + 15) / 16 * 16, (hipStream_t)stream);
}

int ohara_gemm_skinny_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int n, int k, const uint16_t* norm_w,
                           float eps, int batch, int epilogue, const uint16_t* resid, int ldr, uint16_t* out,
                           int ldo, void* stream) {
  if (!x || !wp || !out || n < 1 || k < 1 || batch < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;  // 16-byte activation loads
  if (epilogue == OHARA_EPI_RESIDUAL && (!resid || ldr < n)) return OHARA_EINVAL;
  if (epilogue < OHARA_EPI_STORE || epilogue > OHARA_EPI_SWIGLU) return OHARA_EINVAL;
  if (ldo < n) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps;
  a.B = batch; a.N = n; a.K = k;
  a.out = out; a.ldo = ldo; a.resid = resid; a.ldr = ldr;
  int packed_rows;
  if (epilogue == OHARA_EPI_SWIGLU) packed_rows = 2 * ((n + 7) / 8 * 8);
  else packed_rows = (n + 15) / 16 * 16;
  // (a residual, 17, 33 and 64 rows, strips / tiles: 2048 x 2048 5.6 7.6 7.9 / 6.9 6.9 7.0; 2048 x 5632 11.1 18.7 18.1 / 18.5 18.4 18.6 us)
  if (!norm_w && (epilogue == OHARA_EPI_RESIDUAL ? batch > 64 : ohara_tiles_win(batch, k, packed_rows)))
    return ohara_launch_gemm_tile(a, epilogue, packed_rows, (hipStream_t)stream);
  return launch_skinny(a, epilogue, packed_rows, (hipStream_t)stream);
}

static int qkv_rope_impl(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w,
                         float eps, int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                         const uint16_t* sin, int pos, const int32_t* pos_dev, int pos_stride, uint16_t* q_out,
                         uint16_t* kcache, uint16_t* vcache, int t_max, int stage, void* stream) {
  if (!x || !wp || !cos || !sin || !q_out || !kcache || !vcache) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || h_kv < 1 || h % h_kv || dh < 4 || (dh & 3) || t_max < 1)
    return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  if ((int64_t)batch * seq_len > INT32_MAX) return OHARA_ESIZE;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps;
  a.B = batch * seq_len; a.N = (h + 2 * h_kv) * dh; a.K = k;
  a.S = seq_len; a.row0 = 0;
  a.out = q_out; a.ldo = h * dh;
  a.H = h; a.Hkv = h_kv; a.Dh = dh; a.Tmax = t_max; a.pos = pos; a.pos_dev = pos_dev; a.pos_stride = pos_stride;
  a.cos = cos; a.sin = sin; a.kcache = kcache; a.vcache = vcache; a.stage = stage;
  const int packed_rows = (a.N + 15) / 16 * 16;
  if (!norm_w && ohara_tiles_win(a.B, k, packed_rows)) return ohara_launch_gemm_tile(a, EPI_ROPE, packed_rows, (hipStream_t)stream);
  return launch_skinny(a, EPI_ROPE, packed_rows, (hipStream_t)stream);
}

int ohara_qkv_rope_append_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w,
                               float eps, int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                               const uint16_t* sin, int pos, const int32_t* pos_dev, uint16_t* q_out,
                               uint16_t* kcache, uint16_t* vcache, int t_max, void* stream) {
  return qkv_rope_impl(x, ldx, wp, k, norm_w, eps, batch, seq_len, h, h_kv, dh, cos, sin, pos, pos_dev, 0, q_out, kcache,
                       vcache, t_max, 0, stream);
}

int ohara_qkv_rope_append_ragged_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w,
                                      float eps, int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos,
                                      const uint16_t* sin, const int32_t* seq_pos, uint16_t* q_out, uint16_t* kcache,
                                      uint16_t* vcache, int t_max, void* stream) {
  if (!seq_pos) return OHARA_EINVAL;
  return qkv_rope_impl(x, ldx, wp, k, norm_w, eps, batch, seq_len, h, h_kv, dh, cos, sin, 0, seq_pos, 1, q_out, kcache,
                       vcache, t_max, 0, stream);
}

int ohara_qkv_rope_append_rows_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, int rows, int h, int h_kv, int dh,
                                    const uint16_t* cos, const uint16_t* sin, const int32_t* at, uint16_t* q_out, uint16_t* kcache,
                                    uint16_t* vcache, int t_max, void* stream) {
  if (!x || !wp || !cos || !sin || !at || !q_out || !kcache || !vcache) return OHARA_EINVAL;
  if (rows < 1 || h < 1 || h_kv < 1 || h % h_kv || dh < 4 || (dh & 3) || t_max < 1) return OHARA_EINVAL;
  if ((k & 7) || (ldx & 7) || ldx < k) return OHARA_EINVAL;
  GemmArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp);
  a.x = x; a.ldx = ldx;
  a.B = rows; a.N = (h + 2 * h_kv) * dh; a.K = k; a.S = 1;
  a.out = q_out; a.ldo = h * dh;
  a.H = h; a.Hkv = h_kv; a.Dh = dh; a.Tmax = t_max; a.rows = at; a.nrows = rows;
  a.cos = cos; a.sin = sin; a.kcache = kcache; a.vcache = vcache;
  return ohara_launch_gemm_tile(a, EPI_ROPE, (a.N + 15) / 16 * 16, (hipStream_t)stream);
}

int ohara_qkv_rope_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w, float eps,
                        int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos, const uint16_t* sin,
                        int pos, const int32_t* pos_dev, int t_max, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
                        void* stream) {
  return qkv_rope_impl(x, ldx, wp, k, norm_w, eps, batch, seq_len, h, h_kv, dh, cos, sin, pos, pos_dev, 0, q_out, k_out,
                       v_out, t_max, 1, stream);
}

int ohara_qkv_rope_ragged_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int k, const uint16_t* norm_w, float eps,
                               int batch, int seq_len, int h, int h_kv, int dh, const uint16_t* cos, const uint16_t* sin,
                               const int32_t* seq_pos, int t_max, uint16_t* q_out, uint16_t* k_out, uint16_t* v_out,
                               void* stream) {
  if (!seq_pos) return OHARA_EINVAL;
  return qkv_rope_impl(x, ldx, wp, k, norm_w, eps, batch, seq_len, h, h_kv, dh, cos, sin, 0, seq_pos, 1, q_out, k_out,
                       v_out, t_max, 1, stream);
}

}  // extern "C"
