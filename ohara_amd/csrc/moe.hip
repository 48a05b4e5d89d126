// Grouped mixture-of-experts feed-forward for decode (eval mode of GroupedMoE,
// ohara/modules/moe_grouped.py:122-228; same routing as the loop variant ohara/modules/moe.py:65-127).
//
//   route    logits = float(bf16 router Linear) (:126); experts = first k of top-(k+1) of
//            logits + router_bias (:129-133) or plain top-k (:135), ties to the lowest id;
//            weights = softmax over the k selected UNBIASED logits (:140-142) or sigmoid,
//            optionally normalised (:144-146); cast to bf16 (:217)
//   sort     (token, slot) pairs grouped by expert, token order kept inside an expert (the
//            stable argsort + bincount + cumsum of :165-168), as a counting sort in LDS
//   experts  per expert e and its pairs: hidden = bf16(silu(bf16(x W_gate[e]))) * bf16(x W_up[e]),
//            y = bf16(bf16(hidden W_down[e]) * weight) (:175-181) - the expert weights are
//            streamed once per 16-token column tile through the same packed MFMA tiles as the
//            dense projections (at ~8 tokens per expert this is a weight stream, not a GEMM)
//   combine  out[token] = sum over its experts in ascending expert id, each add rounded to bf16
//            (index_add_ in the activation dtype, :184), + shared expert (:206-207,219-220),
//            + residual (ohara/models/llama.py:200)
//
// The second half is a layer of another kind without a counterpart in the reference: fp32 router over experts and identity
// outputs with groups, clamped gated units, fp32 weights.  It shares the sort and the expert kernel; its sum over the
// chosen experts is part of the residual update (OharaMixture, residual_norm.hip).
#include "lds_tile.h"
#include "mfma_frag.h"

namespace {

// ---- routing ---------------------------------------------------------------------------------
// The selection and the weights of one token by one wave: lane l holds experts l, l + 64, ... (raw: the unbiased
// logits, sel: what the top-k looks at, -inf past E); lanes below k end up with one selected expert and its weight.
template <int MAXPL>
__device__ __forceinline__ void route_core(float (&sel)[MAXPL], const float (&raw)[MAXPL], int E, int k, int sigmoid,
                                           int normalize, int lane, int& my_id, float& wt) {
  // Winner j is kept by lane j.
  float my_raw = 0.f;
  my_id = 0;
  if constexpr (MAXPL == 1) {
    // An expert a lane: its rank is how many come before it, counted over the 64 keys, and the lanes swap places by rank.  (64 times
    // four instructions where k arg-max butterflies are k times six dependent steps; with the product's
    // reads below, 64 experts, 8 chosen, d 1024: 24 tokens 12.7 -> 10.6 us, one 10.9 -> 8.4)
    const float v = sel[0] + 0.f;  // (-0 is 0)
    const uint32_t bits = __float_as_uint(v);
    uint32_t key = bits ^ (bits >> 31 ? 0xffffffffu : 0x80000000u);  // ascending as v is
    if (v != v) key = 2;  // NaN: behind every number
    if (lane >= E) key = 1;
    int rank = 0;
#pragma unroll
    for (int j = 0; j < 64; ++j) rank += (uint32_t)__builtin_amdgcn_readlane((int)key, j) > key - (j < lane ? 1u : 0u);  // (ties: the lower id)
    my_id = __builtin_amdgcn_ds_permute(rank * 4, lane);
    my_raw = __uint_as_float((uint32_t)__builtin_amdgcn_ds_permute(rank * 4, (int)__float_as_uint(raw[0])));
  } else {
    // the arg-max butterfly runs on DPP moves and row swaps
    for (int j = 0; j < k; ++j) {
      // lane-local best (lowest id on ties), then across the wave
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) {
        const int e = i * 64 + lane;
        if (e < E && (sel[i] > bv || (sel[i] == bv && e < bi))) {
          bv = sel[i];
          bi = e;
        }
      }
      lane_xor_argmax<32>(bv, bi);
      lane_xor_argmax<16>(bv, bi);
      lane_xor_argmax<8>(bv, bi);
      lane_xor_argmax<4>(bv, bi);
      lane_xor_argmax<2>(bv, bi);
      lane_xor_argmax<1>(bv, bi);
      // fetch the unbiased logit of the winner and retire it
      float r = 0.f;
#pragma unroll
      for (int i = 0; i < MAXPL; ++i)
        if (i * 64 + lane == bi) {
          r = raw[i];
          sel[i] = -INFINITY;
        }
      r = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(r), bi & 63));
      if (lane == j) {
        my_raw = r;
        my_id = bi;
      }
    }
  }
  // weights: every lane below k holds one; the sums run in slot order, as a loop over the slots would
  const bool has = lane < k;
  if (!sigmoid) {
    const float m = wave_max(has ? my_raw : -INFINITY);
    const float e = has ? expf(my_raw - m) : 0.f;
    float z = 0.f;
    for (int j = 0; j < k; ++j) z += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(e), j));
    wt = e / z;
  } else {
    const float sg = has ? 1.0f / (1.0f + expf(-my_raw)) : 0.f;
    float z = 0.f;
    for (int j = 0; j < k; ++j) z += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(sg), j));
    wt = normalize ? sg / fmaxf(z, 1e-9f) : sg;
  }
}

// one wave per token; E <= 64 * MAXPL experts (MAXPL experts per lane), k <= 16
template <int MAXPL>
__global__ __launch_bounds__(256) void moe_route_kernel(const bf16_t* logits, int ldl, const bf16_t* bias, int N, int E,
                                                        int k, int biased, int sigmoid, int normalize, int32_t* idx,
                                                        bf16_t* w) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.x * 4 + wave;
  if (n >= N) return;
  float sel[MAXPL], raw[MAXPL];
#pragma unroll
  for (int i = 0; i < MAXPL; ++i) {
    const int e = i * 64 + lane;
    if (e < E) {
      raw[i] = bf2f(logits[(size_t)n * ldl + e]);
      sel[i] = biased ? raw[i] + bf2f(bias[e]) : raw[i];
    } else {
      raw[i] = 0.f;
      sel[i] = -INFINITY;
    }
  }
  int my_id;
  float wt;
  route_core<MAXPL>(sel, raw, E, k, sigmoid, normalize, lane, my_id, wt);
  if (lane < k) {
    idx[(size_t)n * k + lane] = my_id;
    w[(size_t)n * k + lane] = f2bf(wt);
  }
}

// ---- counting sort of the (token, slot) pairs by expert -----------------------------------------
// offs[e] .. offs[e+1]: pairs of expert e, in token order; pair_of[sorted position] = n*k + j;
// pos_of[n*k + j] = sorted position.
//
// At most 64 experts and 1024 pairs (decode), one workgroup: a pair's rank among the earlier pairs of
// its expert is a ballot match inside its wave (six ballots for the six bits of an expert id) plus the
// counts of the waves before it, instead of a scan over all earlier pairs; the offsets are one wave's scan.
// COH: idx is read past the caches (other workgroups wrote it in this launch).  wcnt: pairs of expert e in wave w, then the first
// sorted position of that wave's pairs of e.
template <bool COH>
__device__ __forceinline__ void sort_small_1024(const int32_t* idx, int NK, int E, int32_t* offs, int32_t* pair_of, int32_t* pos_of,
                                                int (*wcnt)[64]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  wcnt[wave][lane] = 0;
  const int e = tid < NK ? (COH ? (int)ld_coh4(idx + tid) : idx[tid]) : -1;
  unsigned long long same = __ballot(e >= 0);
#pragma unroll
  for (int bit = 0; bit < 6; ++bit) {
    const unsigned long long b = __ballot((e >> bit) & 1);
    same &= ((e >> bit) & 1) ? b : ~b;
  }
  const int rank = __popcll(same & ((1ull << lane) - 1ull));
  __syncthreads();
  if (e >= 0 && (same >> lane) == 1ull) wcnt[wave][e] = __popcll(same);  // the last lane of the wave with this expert
  __syncthreads();
  if (wave == 0) {
    int tot = 0, c[16];
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      c[w] = wcnt[w][lane];
      tot += c[w];
    }
    const int incl = wave_incl_scan_i(lane < E ? tot : 0);
    int run = incl - (lane < E ? tot : 0);
    if (lane < E) offs[lane] = run;
    if (lane == 63) offs[E] = incl;  // lanes at and past E added nothing
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      wcnt[w][lane] = run;
      run += c[w];
    }
  }
  __syncthreads();
  if (e >= 0) {
    const int o = wcnt[wave][e] + rank;
    pair_of[o] = tid;
    pos_of[tid] = o;
  }
}
__global__ __launch_bounds__(1024) void moe_sort_small_kernel(const int32_t* idx, int NK, int E, int32_t* offs,
                                                              int32_t* pair_of, int32_t* pos_of) {
  __shared__ int wcnt[16][64];
  sort_small_1024<false>(idx, NK, E, offs, pair_of, pos_of, wcnt);
}

// ---- norm + router + selection + sort in one launch (decode: at most 64 experts and 1024 pairs) -------
// What precedes the experts is four small steps on the same rows - RMSNorm (ohara/modules/norm.py:16-21), the router
// Linear, the selection, the sort of the pairs - and as four launches they cost four launch latencies for a few
// microseconds of work.  Here a workgroup takes four tokens, one per wave: the wave norms its row (into LDS for the
// router product and out to memory for the experts), wave s multiplies the four rows with strip s of the router's
// packed weights (16 experts, the whole contraction in one wave; the products are rounded to bf16 as the Linear's
// output is), every wave selects for its token, and the workgroup that finishes last sorts the pairs of all tokens.
struct RouteFusedArgs {
  const bf16_t* x;        // (N, d) rows before the norm
  int ldx;
  const bf16_t* norm_w;
  float eps;
  const uint4* wp;        // the router's packed rows: [strip][KS][64]
  const bf16_t* bias;
  int N, d, E, k, biased, sigmoid, normalize;
  bf16_t* xn;             // (N, d) normalised rows
  int ldxn;
  bf16_t* logits;         // optional (N, E) router outputs
  int ldl;
  int32_t* idx;           // (N, k)
  bf16_t* w;              // (N, k)
  int32_t* offs;
  int32_t* pair_of;
  int32_t* pos_of;
  int* counter;           // one word, zero between calls
};

// moe_sort_small_kernel's sort by 256 threads: a thread takes pairs tid + 256 r; a "wave" of that kernel is a run of 64
// consecutive pairs, four of which a wave here handles one after the other.  idx is read past the caches (other
// workgroups wrote it in this launch).
__device__ __forceinline__ void sort_small_256(const int32_t* idx, int NK, int E, int32_t* offs, int32_t* pair_of,
                                               int32_t* pos_of, int (*wcnt)[64]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int e[4], rank[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) wcnt[wave + 4 * r][lane] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int p = tid + 256 * r;
    e[r] = p < NK ? (int)ld_coh4(idx + p) : -1;
    unsigned long long same = __ballot(e[r] >= 0);
#pragma unroll
    for (int bit = 0; bit < 6; ++bit) {
      const unsigned long long b = __ballot((e[r] >> bit) & 1);
      same &= ((e[r] >> bit) & 1) ? b : ~b;
    }
    rank[r] = __popcll(same & ((1ull << lane) - 1ull));
    if (e[r] >= 0 && (same >> lane) == 1ull) wcnt[wave + 4 * r][e[r]] = __popcll(same);  // the run's last pair of this expert
  }
  __syncthreads();
  if (wave == 0) {
    int tot = 0, c[16];
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      c[w] = wcnt[w][lane];
      tot += c[w];
    }
    const int incl = wave_incl_scan_i(lane < E ? tot : 0);
    int run = incl - (lane < E ? tot : 0);
    if (lane < E) offs[lane] = run;
    if (lane == 63) offs[E] = incl;  // lanes at and past E added nothing
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      wcnt[w][lane] = run;
      run += c[w];
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (e[r] >= 0) {
      const int p = tid + 256 * r;
      const int o = wcnt[wave + 4 * r][e[r]] + rank[r];
      pair_of[o] = p;
      pos_of[p] = o;
    }
}

__global__ __launch_bounds__(256) void moe_route_fused_kernel(RouteFusedArgs a) {
  extern __shared__ __align__(16) unsigned char route_smem[];
  __shared__ float slog[4][64];
  __shared__ int wcnt[16][64];
  __shared__ int is_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int KS = (a.d + 31) >> 5;
  const int ldxs = KS * 32 + 8;
  bf16_t* xs = reinterpret_cast<bf16_t*>(route_smem);  // four normalised rows
  const int t0 = blockIdx.x * 4;
  const uint4* wrow = a.wp + (size_t)min(wave, ((a.E + 15) >> 4) - 1) * KS * 64 + lane;  // (2.: strip `wave` of the router)
  uint4 wv[32];
  // 1. RMSNorm, a row per wave (the row stays in registers between the sum and the scaling):
  //    y = bf16(bf16(x * rinv) * w), rinv = 1 / sqrt(mean(x^2) + eps)
  {
    const int n = t0 + wave;
    const bf16_t* xr = a.x + (size_t)min(n, a.N - 1) * a.ldx;
    uint4 xv[8], gv[8];  // (d <= 4096)
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int i = (c * 64 + lane) * 8;
      xv[c] = i < a.d ? ldg16(xr + i) : make_uint4(0, 0, 0, 0);
      gv[c] = i < a.d ? ldg16(a.norm_w + i) : make_uint4(0, 0, 0, 0);
    }
    // the router's weights are asked for before anything waits, behind the row (24 tokens, 64 experts, d 1024: 14.4 -> 13.6 us)
#pragma unroll
    for (int c = 0; c < 32; ++c) wv[c] = ldg16_nt(wrow + (size_t)min(c, KS - 1) * 64);
    __builtin_amdgcn_sched_barrier(0);
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const uint32_t u[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float lo = lo_bf(u[q]), hi = hi_bf(u[q]);
        ss += lo * lo + hi * hi;
      }
    }
    ss = wave_sum(ss);
    const float rinv = 1.0f / sqrtf(ss / (float)a.d + a.eps);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      const int i = (c * 64 + lane) * 8;
      if (i < KS * 32) {  // (the columns between d and the next multiple of 32 are zero for the product)
        const uint32_t u[4] = {xv[c].x, xv[c].y, xv[c].z, xv[c].w}, gw[4] = {gv[c].x, gv[c].y, gv[c].z, gv[c].w};
        uint32_t y[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          y[q] = pack_bf(rbf(lo_bf(u[q]) * rinv) * lo_bf(gw[q]), rbf(hi_bf(u[q]) * rinv) * hi_bf(gw[q]));
        const uint4 o = make_uint4(y[0], y[1], y[2], y[3]);
        if (n < a.N && i < a.d) *reinterpret_cast<uint4*>(a.xn + (size_t)n * a.ldxn + i) = o;
        *reinterpret_cast<uint4*>(xs + (size_t)wave * ldxs + i) = o;
      }
    }
  }
  __syncthreads();
  // 2. the router product: wave s takes strip s (experts 16 s ..) over the whole contraction, the four tokens in
  //    columns 0..3 (the other columns repeat them and are dropped), 32 k-steps of weights in flight
  {
    const int m = lane & 15, g = lane >> 4;
    const int strips = (a.E + 15) >> 4;
    if (wave < strips) {
      const bf16_t* xrow = xs + (size_t)(m & 3) * ldxs + 8 * g;
      f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
      for (int jb = 0; jb < KS; jb += 32) {
        if (jb) {
#pragma unroll
          for (int c = 0; c < 32; ++c) wv[c] = ldg16_nt(wrow + (size_t)min(jb + c, KS - 1) * 64);
        }
#pragma unroll
        for (int cb = 0; cb < 32; cb += 8) {  // eight steps' reads together (a branch a step waited for each)
          if (jb + cb + 8 <= KS) {
            uint4 xv[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) xv[c] = *reinterpret_cast<const uint4*>(xrow + 32 * (jb + cb + c));
#pragma unroll
            for (int c = 0; c < 8; ++c)
              acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[cb + c]), __builtin_bit_cast(bf16x8, xv[c]),
                                                            acc, 0, 0, 0);
          } else {
#pragma unroll
            for (int c = 0; c < 7; ++c) {
              if (jb + cb + c < KS) {
                const uint4 xv = *reinterpret_cast<const uint4*>(xrow + 32 * (jb + cb + c));
                acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[cb + c]), __builtin_bit_cast(bf16x8, xv),
                                                              acc, 0, 0, 0);
              }
            }
          }
        }
      }
      if (m < 4) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int e = 16 * wave + 4 * g + i;
          const float y = rbf(acc[i]);
          slog[m][e] = y;
          if (a.logits && e < a.E && t0 + m < a.N) a.logits[(size_t)(t0 + m) * a.ldl + e] = f2bf(y);
        }
      }
    }
  }
  __syncthreads();
  // 3. the selection: a token per wave, lane = expert
  {
    const int n = t0 + wave;
    if (n < a.N) {  // (wave-uniform)
      float raw[1], sel[1];
      raw[0] = lane < a.E ? slog[wave][lane] : 0.f;
      sel[0] = lane < a.E ? (a.biased ? raw[0] + bf2f(a.bias[lane]) : raw[0]) : -INFINITY;
      int my_id;
      float wt;
      route_core<1>(sel, raw, a.E, a.k, a.sigmoid, a.normalize, lane, my_id, wt);
      if (lane < a.k) {
        st_coh4(a.idx + (size_t)n * a.k + lane, (uint32_t)my_id);  // (read by the workgroup that sorts)
        a.w[(size_t)n * a.k + lane] = f2bf(wt);
      }
    }
  }
  // 4. the workgroup that finishes last sorts all pairs
  wait_own_stores();
  __syncthreads();
  if (tid == 0) {
    const int old = __hip_atomic_fetch_add(a.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = old == (int)gridDim.x - 1;
    if (is_last) __hip_atomic_store(a.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next call
  }
  __syncthreads();
  if (is_last) sort_small_256(a.idx, a.N * a.k, a.E, a.offs, a.pair_of, a.pos_of, wcnt);
}

// ---- expert projections --------------------------------------------------------------------------
enum { X_SWIGLU = 0, X_DOWN = 1, X_GLU = 2, X_RAW = 3 };  // X_GLU: clamped unit; X_RAW: X_DOWN without weights

struct ExpertArgs {
  const uint4* wp;        // [E][strips][KS][64] packed rows of every expert
  size_t expert_stride;   // uint4 per expert
  const bf16_t* x;        // X_SWIGLU: (N, K) activations, gathered by token; X_DOWN: (NK, K) by sorted position
  int ldx;
  const int32_t* offs;    // (E+1)
  const int32_t* pair_of; // (NK)
  const bf16_t* w;        // (NK) routing weights, pair order (X_DOWN)
  int k;                  // experts per token
  int N_out, K;           // output width (X_SWIGLU: hidden F; X_DOWN: d) and contraction length
  bf16_t* out;            // (NK, N_out) by sorted position
  int ldo;
  // The shared expert (moe_grouped.py:206-207, 219-220) as more rows of the grid, blockIdx.y >= E, 16 tokens a row:
  // every token is its "pair" (row n of x_sh -> row n of out_sh), its weights have their own widths, and its output
  // is not scaled.
  int E, N_sh;            // experts; tokens of the shared expert (0: none)
  const uint4* wp_sh;
  const bf16_t* x_sh;     // X_SWIGLU: (N, K) the tokens' rows; X_DOWN: (N, K_sh) the shared expert's activations
  int ldx_sh;
  int N_out_sh, K_sh;
  bf16_t* out_sh;
  int ldo_sh;
  OharaGlu glu, glu_sh;   // X_GLU
  const float* pair_w;    // X_GLU: factor of a pair's input (null: none)
};

// CH: k-steps a wave has in flight at once (the host takes 4 when a wave's share of K is that short).
// Every load of a batch is issued whatever its index - clamped into the strip and the row, zeroed
// afterwards where it lies beyond the wave's share - so the batch is one run of loads without branches.
template <int EPI, int CH>
__global__ __launch_bounds__(256) void moe_expert_kernel(ExpertArgs a) {
  constexpr bool GATED = EPI == X_SWIGLU || EPI == X_GLU;
  const int strip = blockIdx.x, e = blockIdx.y;
  const bool sh = e >= a.E;  // (workgroup-uniform) a row of the shared expert: 16 tokens each
  const int p0 = sh ? (e - a.E) * 16 : a.offs[e], p1 = sh ? min(a.N_sh, p0 + 16) : a.offs[e + 1];
  if (p0 >= p1) return;
  const int N_out = sh ? a.N_out_sh : a.N_out, K = sh ? a.K_sh : a.K;
  if (strip * 16 >= (GATED ? 2 * ((N_out + 7) / 8 * 8) : N_out)) return;  // (the grid is as wide as the widest)
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m = lane & 15, g = lane >> 4;
  const int KS = (K + 31) >> 5;
  const int per = (KS + 3) >> 2;
  const int j0 = wave * per, j1 = min(KS, j0 + per);
  __shared__ float red[3][64][4];
  const uint4* wrow = (sh ? a.wp_sh : a.wp + (size_t)e * a.expert_stride) + (size_t)strip * KS * 64 + lane;
  bf16_t* const outp = sh ? a.out_sh : a.out;
  const int ldo = sh ? a.ldo_sh : a.ldo;
  for (int pt = p0; pt < p1; pt += 16) {  // 16-token column tiles of this expert
    const int pos = pt + m;
    const bool has = pos < p1;
    const int posc = min(pos, p1 - 1);  // a token of this expert: lanes past the end compute a column nobody stores
    const int pair = sh || EPI == X_RAW ? 0 : a.pair_of[posc];
    const bf16_t* xrow = sh ? a.x_sh + (size_t)posc * a.ldx_sh
                            : a.x + (size_t)(GATED ? pair / a.k : posc) * a.ldx;
    float wt = 1.0f;  // (the shared expert's output is not scaled: a bf16 value times one is itself)
    if (EPI == X_GLU && !sh && a.pair_w) wt = a.pair_w[pair];
    if (EPI == X_DOWN && !sh) wt = bf2f(a.w[pair]);  // asked for here, used in the epilogue
    f32x4 acc = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int jb = j0; jb < j1; jb += CH) {
      uint4 wv[CH], xv[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int j = min(jb + c, j1 - 1);
        wv[c] = ldg16_nt(wrow + (size_t)j * 64);
        xv[c] = ldg16(xrow + min(32 * j + 8 * g, K - 8));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const bool live = jb + c < j1 && 32 * (jb + c) + 8 * g < K;
        if (!live) xv[c] = make_uint4(0, 0, 0, 0);  // the packed weights are zero beyond K; the row's values are not
        if (jb + c >= j1) wv[c] = make_uint4(0, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[c]), __builtin_bit_cast(bf16x8, xv[c]),
                                                      acc, 0, 0, 0);
      }
    }
    if (wave > 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) red[wave - 1][lane][i] = acc[i];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[i] = ((acc[i] + red[0][lane][i]) + red[1][lane][i]) + red[2][lane][i];
      if (has && EPI == X_GLU) {
        const OharaGlu u = sh ? a.glu_sh : a.glu;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] *= wt;
        const int f = strip * 8 + 2 * g;
        bf16_t* o = outp + (size_t)pos * ldo + f;
        if (f < N_out) o[0] = f2bf(clamped_glu(acc[0], acc[2], u.limit, u.alpha, u.offset));
        if (f + 1 < N_out) o[1] = f2bf(clamped_glu(acc[1], acc[3], u.limit, u.alpha, u.offset));
      } else if (has) {
        const float y0 = rbf(acc[0]), y1 = rbf(acc[1]), y2 = rbf(acc[2]), y3 = rbf(acc[3]);
        if (EPI == X_SWIGLU) {
          const int f = strip * 8 + 2 * g;
          bf16_t* o = outp + (size_t)pos * ldo + f;
          if (f < N_out) o[0] = f2bf(rbf(silu_f(y0)) * y2);
          if (f + 1 < N_out) o[1] = f2bf(rbf(silu_f(y1)) * y3);
        } else {
          const int r0 = strip * 16 + 4 * g;
          const float v[4] = {y0 * wt, y1 * wt, y2 * wt, y3 * wt};
          bf16_t* o = outp + (size_t)pos * ldo + r0;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (r0 + i < N_out) o[i] = f2bf(v[i]);
        }
      }
    }
    __syncthreads();
  }
}

// ---- fp32 router, groups, identity outputs -------------------------------------------------------
template <typename T>
struct RouterArgs {
  const T* x;
  const T* w;
  const float* correction;
  int ldx, ldw, N, K, E, top, groups, keep;  // E: outputs (experts and identities)
  int32_t* idx;
  float* wgt;
  int32_t* offs;   // sort: the workgroup that finishes last sorts the pairs of all tokens (E <= 64, at most 1024 pairs)
  int32_t* pair_of;
  int32_t* pos_of;
  int* counter;
  int flags;
  int sort;
};

constexpr int RT = 16;  // tokens of a workgroup, waves of a workgroup
constexpr int RED_LD = 260;  // floats of one wave's share of a strip (256), apart in LDS banks

// The products of 16 tokens with up to NS strips of 16 router rows at a time, K split over the sixteen waves (a single token's launch
// is one round of loads); then a token per wave, lane l looking at outputs l, l + 64, ...
template <typename T, int MAXPL, int NS>
__global__ __launch_bounds__(1024) void moe_router_kernel(RouterArgs<T> a) {
  extern __shared__ __align__(16) float zs[];  // [RT][E], then every wave's sums [RT][NS][RED_LD]
  __shared__ int wcnt[16][64];
  __shared__ int is_last;
  float* red = zs + RT * a.E;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * RT, KS = (a.K + 31) >> 5;
  const T* xr = a.x + (size_t)min(t0 + m, a.N - 1) * a.ldx + 8 * g;
  for (int e0 = 0; e0 < a.E; e0 += 16 * NS) {
    f32x4 acc[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const T* wr[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) wr[s] = a.w + (size_t)min(e0 + 16 * s + m, a.E - 1) * a.ldw + 8 * g;
    constexpr int CH = (sizeof(T) == 2 ? 4 : 2) / (NS == 4 ? 2 : 1);  // steps whose loads are issued together
    for (int jb = wave; jb < KS; jb += RT * CH) {
      Frag<T> xf[CH], wf[CH][NS];
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const int j = jb + RT * c;
        const bool in = 32 * j + 8 * g < a.K;  // K is a multiple of 8
        if (in) frag_load(xf[c], xr + 32 * j);
        else frag_zero(xf[c]);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          if (in) frag_load(wf[c][s], wr[s] + 32 * j);
          else frag_zero(wf[c][s]);
        }
      }
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[s] = mma(wf[c][s], xf[c], acc[s]);
    }
    if (e0) __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) *reinterpret_cast<f32x4*>(red + (wave * NS + s) * RED_LD + 4 * lane) = acc[s];
    __syncthreads();
    for (int i = tid; i < NS * 256; i += 1024) {  // strip i / 256, row and token i % 256
      const int s = i >> 8, r = (i >> 4) & 15, t = i & 15, e = e0 + 16 * s + r;
      float z = 0.f;
#pragma unroll
      for (int w = 0; w < RT; ++w) z += red[(w * NS + s) * RED_LD + 4 * (16 * (r >> 2) + t) + (r & 3)];
      if (e < a.E) zs[t * a.E + e] = z;
    }
  }
  __syncthreads();
  const int per = a.E / a.groups;
  const int n = t0 + wave;
  if (n < a.N) {  // the same for the whole wave, whose row of zs is its own from here on
    float* z = zs + wave * a.E;
    float s[MAXPL], ch[MAXPL], mx = -INFINITY, sum = 0.f;
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
      const int e = 64 * i + lane;
      s[i] = e < a.E ? z[e] : -INFINITY;
      mx = fmaxf(mx, s[i]);
    }
    if (a.flags & OHARA_ROUTER_SIGMOID) {
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) {
        ch[i] = s[i];  // the scores' order, also where they round to 1
        s[i] = 1.0f / (1.0f + expf(-s[i]));
      }
    } else {
      mx = wave_max(mx);
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) {
        s[i] = 64 * i + lane < a.E ? expf(s[i] - mx) : 0.f;
        sum += s[i];
      }
      sum = wave_sum(sum);
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) ch[i] = s[i] /= sum;
    }
#pragma unroll
    for (int i = 0; i < MAXPL; ++i) {
      const int e = 64 * i + lane;
      ch[i] = e < a.E ? (a.correction ? s[i] + a.correction[e] : ch[i]) : -INFINITY;
      if (!(ch[i] == ch[i])) ch[i] = -INFINITY;  // a padding row may hold anything: every row still picks distinct outputs
    }
    if (a.groups > 1) {
#pragma unroll
      for (int i = 0; i < MAXPL; ++i)
        if (64 * i + lane < a.E) z[64 * i + lane] = ch[i];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      float best = -INFINITY;  // of group `lane`
      if (lane < a.groups)
        for (int e = lane * per; e < (lane + 1) * per; ++e) best = fmaxf(best, z[e]);
      int rank = 0;
      for (int o = 0; o < a.groups; ++o) {
        const float v = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(best), o));
        rank += v > best || (v == best && o < lane) ? 1 : 0;
      }
      const unsigned long long open = __ballot(lane < a.groups && rank < a.keep);
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) {
        const int e = 64 * i + lane;
        if (e < a.E && !((open >> (e / per)) & 1ull)) ch[i] = -INFINITY;
      }
    }
    // the best `top`, winner j kept by lane j
    uint32_t taken = 0;
    int my_id = 0;
    float my_s = 0.f;
    for (int j = 0; j < a.top; ++j) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < MAXPL; ++i) {
        const int e = 64 * i + lane;
        if (e < a.E && !((taken >> i) & 1u) && (ch[i] > bv || bi == 0x7fffffff)) {
          bv = ch[i];
          bi = e;
        }
      }
      lane_xor_argmax<32>(bv, bi);
      lane_xor_argmax<16>(bv, bi);
      lane_xor_argmax<8>(bv, bi);
      lane_xor_argmax<4>(bv, bi);
      lane_xor_argmax<2>(bv, bi);
      lane_xor_argmax<1>(bv, bi);
      float r = 0.f;
#pragma unroll
      for (int i = 0; i < MAXPL; ++i)
        if (64 * i + lane == bi) {
          r = s[i];
          taken |= 1u << i;
        }
      r = __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(r), bi & 63));
      if (lane == j) {
        my_s = r;
        my_id = bi;
      }
    }
    float tot = 0.f;
    for (int j = 0; j < a.top; ++j) tot += __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(my_s), j));
    if (lane < a.top) {
      st_coh4(a.idx + (size_t)n * a.top + lane, (uint32_t)my_id);  // (read by the workgroup that sorts)
      a.wgt[(size_t)n * a.top + lane] = (a.flags & OHARA_ROUTER_PLAIN) ? my_s : my_s / (tot + 1e-20f);
    }
  }
  if (!a.sort) return;
  wait_own_stores();
  __syncthreads();
  if (tid == 0) {
    const int old = __hip_atomic_fetch_add(a.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = old == (int)gridDim.x - 1;
    if (is_last) __hip_atomic_store(a.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next call
  }
  __syncthreads();
  if (is_last) sort_small_1024<true>(a.idx, a.N * a.top, a.E, a.offs, a.pair_of, a.pos_of, wcnt);
}

// The sort for many pairs on many workgroups: every block of 1024 pairs places its own.  The counts that it needs - all pairs of an
// expert, and those in blocks before it - come from a launch that counted each block (HIST), or, without memory for
// them, from the block's own walk over all ids (30720 pairs: 11 us in all, where one workgroup that walked the blocks one
// after the other took 700).
__global__ __launch_bounds__(1024) void moe_count_kernel(const int32_t* idx, int NK, int E, int32_t* hist) {
  __shared__ int cnt[1024];
  const int tid = threadIdx.x, p = blockIdx.x * 1024 + tid;
  cnt[tid] = 0;
  __syncthreads();
  if (p < NK) atomicAdd(&cnt[idx[p]], 1);
  __syncthreads();
  if (tid < E) hist[(size_t)blockIdx.x * E + tid] = cnt[tid];
}
// A pair's rank among the earlier pairs of its expert: a ballot match inside its wave, and the counts of the waves before it.
template <bool HIST>
__global__ __launch_bounds__(1024) void moe_place_kernel(const int32_t* idx, int NK, int E, const int32_t* hist, int32_t* offs,
                                                         int32_t* pair_of, int32_t* pos_of) {
  extern __shared__ int wcnt[];  // [16][E]: pairs of an expert in a wave, then the sorted position of that wave's first
  __shared__ int wsum[16], tot[HIST ? 1 : 1024], bef[HIST ? 1 : 1024];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, blk = blockIdx.x, nb = gridDim.x;
  const int p = blk * 1024 + tid, e = p < NK ? idx[p] : -1;
  for (int i = tid; i < 16 * E; i += 1024) wcnt[i] = 0;
  int total = 0, before = 0;
  if (!HIST) {
    tot[tid] = bef[tid] = 0;
    __syncthreads();
    for (int p0 = tid; p0 < NK; p0 += 4096) {  // four ids in flight
      int id[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) id[u] = idx[min(p0 + 1024 * u, NK - 1)];
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (p0 + 1024 * u < NK) {
          atomicAdd(&tot[id[u]], 1);
          if (p0 + 1024 * u < blk * 1024) atomicAdd(&bef[id[u]], 1);
        }
    }
    __syncthreads();
    if (tid < E) {
      total = tot[tid];
      before = bef[tid];
    }
  } else if (tid < E) {
    for (int b0 = 0; b0 < nb; b0 += 8) {  // eight blocks' counts in flight
      int c[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] = hist[(size_t)min(b0 + u, nb - 1) * E + tid];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        total += b0 + u < nb ? c[u] : 0;
        before += b0 + u < blk ? c[u] : 0;
      }
    }
  }
  const int incl = wave_incl_scan_i(total);
  if (lane == 63) wsum[wave] = incl;
  unsigned long long same = __ballot(e >= 0);
  for (int bit = 0; (E - 1) >> bit; ++bit) {
    const unsigned long long b = __ballot((e >> bit) & 1);
    same &= ((e >> bit) & 1) ? b : ~b;
  }
  const int rank = __popcll(same & ((1ull << lane) - 1ull));
  __syncthreads();
  if (e >= 0 && (same >> lane) == 1ull) wcnt[wave * E + e] = __popcll(same);  // the last lane of the wave with this expert
  __syncthreads();
  int run = incl - total;
  for (int w = 0; w < wave; ++w) run += wsum[w];
  if (tid < E) {
    if (blk == 0) {
      offs[tid] = run;
      if (tid == E - 1) offs[E] = run + total;
    }
    run += before;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      const int c = wcnt[w * E + tid];
      wcnt[w * E + tid] = run;
      run += c;
    }
  }
  __syncthreads();
  if (e >= 0) {
    const int o = wcnt[wave * E + e] + rank;
    pair_of[o] = p;
    pos_of[p] = o;
  }
}

// ---- many pairs: tiles of pairs of one expert x packed weight rows -------------------------------------
// tile_product (lds_tile.h) over rows gathered by pair (gated: the token's row) or by sorted position.  An XCD gets a contiguous
// run of tiles, the weight tiles of one tile of pairs side by side, so an expert's weights and rows stay in its L2.
struct ExpertTileArgs {
  const uint4* wp;
  size_t expert_stride;   // uint4 per expert
  const bf16_t* x;
  int ldx;
  const int32_t* offs;
  const int32_t* pair_of;
  int top, E, N_out, K;
  bf16_t* out;
  int ldo;
  OharaGlu glu;
  const float* pair_w;    // X_GLU: factor of a pair's input (null: none)
  const bf16_t* w;        // X_DOWN: routing weights, pair order
};

template <int EPI, class C>
__global__ __launch_bounds__(C::NW * 64, 2) void moe_tile_kernel(ExpertTileArgs a, int NT, int nstrips) {
  constexpr bool GATED = EPI == X_SWIGLU || EPI == X_GLU;
  constexpr int TM = C::TM, FM = C::FM, FN = C::FN;
  extern __shared__ __align__(16) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // tiles of pairs there are (the grid is as large as there could be), and which of them is this workgroup's
  auto scan = [&](int e0, int& c) {
    c = e0 + lane < a.E ? (a.offs[e0 + lane + 1] - a.offs[e0 + lane] + TM - 1) / TM : 0;
    return wave_incl_scan_i(c);
  };
  int total = 0, c;
  for (int e0 = 0; e0 < a.E; e0 += 64) total += __builtin_amdgcn_readlane(scan(e0, c), 63);
  const int T = total * NT;
  const int xcd = blockIdx.x & 7, q = blockIdx.x >> 3, base = T >> 3, rem = T & 7;
  if (q >= base + (xcd < rem ? 1 : 0)) return;
  const int pid = xcd * base + min(xcd, rem) + q;
  int tile = pid / NT, e = 0;
  const int tn = pid - tile * NT;
  for (int e0 = 0; e0 < a.E; e0 += 64) {
    const int incl = scan(e0, c);
    const unsigned long long past = __ballot(incl > tile);
    if (past) {
      const int l = __ffsll((long long)past) - 1;
      tile -= __builtin_amdgcn_readlane(incl - c, l);
      e = e0 + l;
      break;
    }
    tile -= __builtin_amdgcn_readlane(incl, 63);
  }
  e = __builtin_amdgcn_readfirstlane(e);
  const int row0 = a.offs[e] + tile * TM, rows = min(TM, a.offs[e + 1] - row0), strip0 = tn * C::TS;
  XOffsets<C, true> x;
#pragma unroll
  for (int i = 0; i < C::XPW; ++i) {
    const int r = row0 + min(x.row(i, wave, lane), rows - 1);
    x.set(i, wave, lane, (uint32_t)(GATED ? a.pair_of[r] / a.top : r) * (uint32_t)a.ldx);
  }
  f32x4 acc[FN][FM];
  tile_product<C, true>(acc, reinterpret_cast<const char*>(a.x), x, a.wp + (size_t)e * a.expert_stride, strip0, nstrips, a.K, wave, lane, smem);
  const int r0 = wave / C::WN * FM * 16, sbase = strip0 + wave % C::WN * FN;
  // Strips' columns lie side by side in a row of the output; exchanged among the lanes of a row they are stored 16 bytes a lane.
  if (FN % 2 == 0 && ((a.N_out | a.ldo) & 7) == 0 && ((uintptr_t)a.out & 15) == 0) {
#pragma unroll
    for (int t = 0; t < FM; ++t) {
      const int r = r0 + t * 16 + m, rc = row0 + min(r, rows - 1);
      bf16_t* o = a.out + (size_t)rc * a.ldo;
      float w = 1.f;
      if (EPI == X_GLU && a.pair_w) w = a.pair_w[a.pair_of[rc]];
      if (EPI == X_DOWN) w = bf2f(a.w[a.pair_of[rc]]);
      if constexpr (GATED) {
        uint32_t y[FN];  // two columns of strip u
        if constexpr (EPI == X_GLU) {
#pragma unroll
          for (int u = 0; u < FN; ++u) {
            const f32x4 c4 = acc[u][t];
            y[u] = pack_bf(clamped_glu(c4[0] * w, c4[2] * w, a.glu.limit, a.glu.alpha, a.glu.offset),
                           clamped_glu(c4[1] * w, c4[3] * w, a.glu.limit, a.glu.alpha, a.glu.offset));
          }
        } else {
          float low = acc[0][t][0];
#pragma unroll
          for (int u = 0; u < FN; ++u) low = fminf(low, fminf(acc[u][t][0], acc[u][t][1]));
          if (__any(low < -86.5f)) {  // (-87 after rounding)
#pragma unroll
            for (int u = 0; u < FN; ++u)
              y[u] = pack_bf(rbf(silu_f(rbf(acc[u][t][0]))) * rbf(acc[u][t][2]), rbf(silu_f(rbf(acc[u][t][1]))) * rbf(acc[u][t][3]));
          } else {
#pragma unroll
            for (int u = 0; u < FN; ++u)
              y[u] = pack_bf(rbf(silu_from_m87(rbf(acc[u][t][0]))) * rbf(acc[u][t][2]),
                             rbf(silu_from_m87(rbf(acc[u][t][1]))) * rbf(acc[u][t][3]));
          }
        }
        const int left = r < rows ? a.N_out - sbase * 8 : 0;  // columns this row still has
        if constexpr (FN == 4) {
          const u32x2 p = __builtin_amdgcn_permlane32_swap(y[0], y[2], false, false), q = __builtin_amdgcn_permlane32_swap(y[1], y[3], false, false);
          const u32x2 c = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false), d = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
          if (8 * g < left) *reinterpret_cast<uint4*>(o + sbase * 8 + 8 * g) = make_uint4(c[0], c[1], d[0], d[1]);
        } else {
#pragma unroll
          for (int u = 0; u < FN; u += 2) {
            const u32x2 c = __builtin_amdgcn_permlane16_swap(y[u], y[u + 1], false, false);
            const int at = 8 * u + 8 * (g & 1) + 4 * (g >> 1);
            if (at < left) *reinterpret_cast<uint2*>(o + sbase * 8 + at) = make_uint2(c[0], c[1]);
          }
        }
      } else {
        auto column4 = [&](f32x4 c4) {
          if (EPI == X_DOWN) return make_uint2(pack_bf(rbf(c4[0]) * w, rbf(c4[1]) * w), pack_bf(rbf(c4[2]) * w, rbf(c4[3]) * w));
          return make_uint2(pack_bf(c4[0], c4[1]), pack_bf(c4[2], c4[3]));
        };
#pragma unroll
        for (int u = 0; u < FN; u += 2) {
          const uint2 l = column4(acc[u][t]), h = column4(acc[u + 1][t]);
          const u32x2 c = __builtin_amdgcn_permlane16_swap(l.x, h.x, false, false), d = __builtin_amdgcn_permlane16_swap(l.y, h.y, false, false);
          const int col = (sbase + u + (g & 1)) * 16 + 8 * (g >> 1);
          if (r < rows && col < a.N_out) *reinterpret_cast<uint4*>(o + col) = make_uint4(c[0], d[0], c[1], d[1]);
        }
      }
    }
    return;
  }
#pragma unroll
  for (int t = 0; t < FM; ++t) {
    const int r = r0 + t * 16 + m;
    if (r >= rows) continue;
    bf16_t* o = a.out + (size_t)(row0 + r) * a.ldo;
    float w = 1.f;
    if (EPI == X_GLU && a.pair_w) w = a.pair_w[a.pair_of[row0 + r]];
    if (EPI == X_DOWN) w = bf2f(a.w[a.pair_of[row0 + r]]);
#pragma unroll
    for (int u = 0; u < FN; ++u) {
      const int strip = sbase + u;
      if (strip >= nstrips) continue;
      f32x4 c4 = acc[u][t];
      if (GATED) {
        const int f = strip * 8 + 2 * g;
        float v0, v1;
        if (EPI == X_GLU) {
#pragma unroll
          for (int i = 0; i < 4; ++i) c4[i] *= w;
          v0 = clamped_glu(c4[0], c4[2], a.glu.limit, a.glu.alpha, a.glu.offset);
          v1 = clamped_glu(c4[1], c4[3], a.glu.limit, a.glu.alpha, a.glu.offset);
        } else {
          v0 = rbf(silu_f(rbf(c4[0]))) * rbf(c4[2]);
          v1 = rbf(silu_f(rbf(c4[1]))) * rbf(c4[3]);
        }
        if (f + 1 < a.N_out && !(a.ldo & 1)) {
          *reinterpret_cast<uint32_t*>(o + f) = pack_bf(v0, v1);
        } else {
          if (f < a.N_out) o[f] = f2bf(v0);
          if (f + 1 < a.N_out) o[f + 1] = f2bf(v1);
        }
      } else {
        const int f = strip * 16 + 4 * g;
        float v[4] = {c4[0], c4[1], c4[2], c4[3]};
        if (EPI == X_DOWN) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = rbf(v[i]) * w;
        }
        if (f + 3 < a.N_out && !(a.ldo & 3)) {
          *reinterpret_cast<uint2*>(o + f) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (f + i < a.N_out) o[f + i] = f2bf(v[i]);
        }
      }
    }
  }
}

typedef Tile<2, 4, 2, 2, 2, 3, 1> E64;   //  64 pairs x 128 packed rows
typedef Tile<2, 4, 4, 2, 2, 2, 0> E128;  // 128 x 128
typedef HalvesTile<2, 4, 8, 4, 1, 3, 4> E256;  // 256 x 256, waves in two halves

template <int EPI, class C>
int launch_expert_tiles(const ExpertTileArgs& t, int n_pairs, int strips, hipStream_t st) {
  const int64_t NT = (strips + C::TS - 1) / C::TS, blocks = ((int64_t)n_pairs / C::TM + t.E) * NT;
  if (blocks > INT32_MAX - 8) return OHARA_ESIZE;
  if (C::LDS > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)moe_tile_kernel<EPI, C>, hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS);
  hipLaunchKernelGGL((moe_tile_kernel<EPI, C>), dim3((unsigned)(blocks + 7) / 8 * 8), dim3(C::NW * 64), C::LDS, st, t, (int)NT, strips);
  return ohara_launch_status();
}

// us for gate/up + down of 64 experts (1024 x 512) at so many pairs an expert, streaming the weights per 16 pairs / tiles of
// 64 pairs / of 128:
//     8    24 + 14    23 + 13    23 + 14        64   132 + 81    33 + 23    26 + 17
//    16    40 + 25    23 + 14    23 + 14       256   504 + 296   66 + 44    57 + 41
//    48   100 + 62    24 + 15    25 + 17       512   978 + 580  121 + 78    92 + 65
// (tiles of 32 are behind everywhere: 27 + 18 at 32).  What bounds the tiles: the experts' weights (201 MB) up to 48 pairs, the
// products' operands through LDS beyond.
constexpr int TILE_PAIRS = 12;    // pairs an expert, on average, from which tiles beat streaming the weights
constexpr int LARGE_PAIRS = 56;   // and from which tiles of 128 do those of 64
// Tiles of 256 take a product in less time (a model's dense products: 12 to 20 % less), but what an expert's pairs leave of the last one is
// multiplied too.  us a forward of 16 layers, tiles of 128 / 256, at so many pairs an expert: 100 2234 / 2327, 128 2537 / 2386, 160 2698 / 2529,
// 200 2911 / 2711, 220 3131 / 3249, 300 3563 / 3719, 375 4089 / 4028, 450 4577 / 4680, 600 5391 / 5224, 712 6532 / 6610, 800 6932 / 6691,
// 1000 8421 / 7901; so: where most experts' pairs are one such tile, more than half full, and from three on.  (128 x 256 in halves: 480 pairs
// 4491 / 4636.)
inline bool huge_tiles(int64_t pairs, int E, int K) {
  return K >= 64 && ((pairs >= 112 * (int64_t)E && pairs <= 208 * (int64_t)E) || pairs >= 768 * (int64_t)E);
}

// false: the rows are not on 16 bytes or not within 4 GiB of each other.
template <int EPI>
bool expert_tiles(const ExpertTileArgs& t, int rows, int n_pairs, int strips, hipStream_t st, int* rc) {
  if (((uintptr_t)t.x & 15) || (t.ldx & 7) || (uint64_t)rows * t.ldx * 2 > UINT32_MAX) return false;
  *rc = huge_tiles(n_pairs, t.E, t.K) ? launch_expert_tiles<EPI, E256>(t, n_pairs, strips, st)
        : n_pairs >= (int64_t)LARGE_PAIRS * t.E ? launch_expert_tiles<EPI, E128>(t, n_pairs, strips, st)
                                                : launch_expert_tiles<EPI, E64>(t, n_pairs, strips, st);
  return true;
}


template <typename T>
int launch_router(RouterArgs<T> a, int32_t* hist, hipStream_t st) {
  if (!a.x || !a.w || !a.idx || !a.wgt || !a.offs || !a.pair_of || !a.pos_of || !a.counter) return OHARA_EINVAL;
  if (a.N < 1 || a.K < 8 || (a.K & 7) || a.ldx < a.K || a.ldw < a.K || ((a.ldx | a.ldw) & 7) || a.E < 1) return OHARA_EINVAL;
  if (a.top < 1 || a.top > a.E || a.groups < 1 || a.E % a.groups || a.keep < 1 || a.keep > a.groups) return OHARA_EINVAL;
  if (a.keep * (a.E / a.groups) < a.top) return OHARA_EINVAL;
  if (a.E > 1024 || a.top > 64 || a.groups > 64 || (int64_t)a.N * a.top > (1 << 30)) return OHARA_ESIZE;
  const int NK = a.N * a.top;
  a.sort = a.E <= 64 && NK <= 1024;
  if (!a.sort && !hist) return OHARA_EINVAL;
  const dim3 grid((unsigned)((a.N + RT - 1) / RT)), block(64 * RT);
  auto go = [&](auto kernel, int ns) {
    const size_t smem = (size_t)RT * (a.E + ns * RED_LD) * sizeof(float);
    if (smem > 32 * 1024) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    hipLaunchKernelGGL(kernel, grid, block, smem, st, a);
  };
  if (a.E <= 16) go(moe_router_kernel<T, 1, 1>, 1);
  else if (a.E <= 32) go(moe_router_kernel<T, 1, 2>, 2);
  else if (a.E <= 64) go(moe_router_kernel<T, 1, 4>, 4);
  else if (a.E <= 256) go(moe_router_kernel<T, 4, 4>, 4);
  else go(moe_router_kernel<T, 16, 4>, 4);
  if (!a.sort) {
    const dim3 blocks((unsigned)((NK + 1023) / 1024));
    hipLaunchKernelGGL(moe_count_kernel, blocks, dim3(1024), 0, st, a.idx, NK, a.E, hist);
    const size_t lds = (size_t)16 * a.E * sizeof(int);
    if (lds > 60 * 1024) (void)hipFuncSetAttribute((const void*)moe_place_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(moe_place_kernel<true>, blocks, dim3(1024), lds, st, a.idx, NK, a.E, hist, a.offs, a.pair_of, a.pos_of);
  }
  return ohara_launch_status();
}

template <int EPI>
int launch_experts(ExpertArgs a, int n_pairs, int n_sh, hipStream_t st) {
  constexpr bool GATED = EPI == X_GLU || EPI == X_SWIGLU;
  auto strips_of = [](int n) { return GATED ? 2 * ((n + 7) / 8 * 8) / 16 : (n + 15) / 16; };
  int strips = strips_of(a.N_out);
  if (n_pairs >= (int64_t)TILE_PAIRS * a.E && !n_sh) {
    const ExpertTileArgs t{a.wp, a.expert_stride, a.x, a.ldx, a.offs, a.pair_of, a.k, a.E, a.N_out, a.K, a.out, a.ldo, a.glu, a.pair_w, a.w};
    int rc;
    if (expert_tiles<EPI>(t, GATED ? n_pairs / a.k : n_pairs, n_pairs, strips, st, &rc)) return rc;
  }
  int rows = a.E, ks = (a.K + 31) / 32;
  if (n_sh) {
    const int s2 = strips_of(a.N_out_sh), k2 = (a.K_sh + 31) / 32;
    strips = strips > s2 ? strips : s2;
    ks = ks > k2 ? ks : k2;
    rows += (n_sh + 15) / 16;
  }
  if (rows > 65535) return OHARA_ESIZE;
  const dim3 grid((unsigned)strips, (unsigned)rows);
  if (ks <= 16) hipLaunchKernelGGL((moe_expert_kernel<EPI, 4>), grid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((moe_expert_kernel<EPI, 8>), grid, dim3(256), 0, st, a);
  return ohara_launch_status();
}

// ---- combine ---------------------------------------------------------------------------------------
// out[n] = resid[n] + ( (sum over the token's experts, ascending id, bf16 adds) + shared[n] )
__global__ __launch_bounds__(256) void moe_combine_kernel(const bf16_t* y, int ldy, const int32_t* idx, const int32_t* pos_of,
                                                          int k, const bf16_t* shared, int lds_, const bf16_t* resid, int ldr,
                                                          bf16_t* out, int ldo, int d) {
  const int n = blockIdx.x;
  __shared__ int order[16];
  if (threadIdx.x < 64) {
    // slots of this token in ascending expert id (k <= 16 distinct experts): lane j ranks its own slot
    const int lane = threadIdx.x;
    const int mine = lane < k ? idx[(size_t)n * k + lane] : 0x7fffffff;
    const int pos = lane < k ? pos_of[(size_t)n * k + lane] : 0;
    int rank = 0;
    for (int j = 0; j < k; ++j) {
      const int other = __shfl(mine, j, WAVE);
      rank += (other < mine || (other == mine && j < lane)) ? 1 : 0;
    }
    if (lane < k) order[rank] = pos;
  }
  __syncthreads();
  const bool vec = ((d | ldy | ldo | lds_ | ldr) & 3) == 0;
  if (vec) {  // four columns per thread, 8-byte loads; the adds stay one bf16 add per expert, in order
    for (int c = threadIdx.x * 4; c < d; c += 1024) {
      uint2 yv[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) yv[j] = j < k ? ldg8(y + (size_t)order[j] * ldy + c) : make_uint2(0, 0);
      const uint2 sv = shared ? ldg8(shared + (size_t)n * lds_ + c) : make_uint2(0, 0);
      const uint2 rv = resid ? ldg8(resid + (size_t)n * ldr + c) : make_uint2(0, 0);
      float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 16; ++j)
        if (j < k) {
          acc[0] = rbf(acc[0] + lo_bf(yv[j].x)); acc[1] = rbf(acc[1] + hi_bf(yv[j].x));
          acc[2] = rbf(acc[2] + lo_bf(yv[j].y)); acc[3] = rbf(acc[3] + hi_bf(yv[j].y));
        }
      if (shared) {
        acc[0] = rbf(acc[0] + lo_bf(sv.x)); acc[1] = rbf(acc[1] + hi_bf(sv.x));
        acc[2] = rbf(acc[2] + lo_bf(sv.y)); acc[3] = rbf(acc[3] + hi_bf(sv.y));
      }
      if (resid) {
        acc[0] = rbf(lo_bf(rv.x) + acc[0]); acc[1] = rbf(hi_bf(rv.x) + acc[1]);
        acc[2] = rbf(lo_bf(rv.y) + acc[2]); acc[3] = rbf(hi_bf(rv.y) + acc[3]);
      }
      stg8(out + (size_t)n * ldo + c, make_uint2(pack_bf(acc[0], acc[1]), pack_bf(acc[2], acc[3])));
    }
    return;
  }
  for (int c = threadIdx.x; c < d; c += 256) {
    float acc = 0.f;
    for (int j = 0; j < k; ++j) acc = rbf(acc + bf2f(y[(size_t)order[j] * ldy + c]));
    if (shared) acc = rbf(acc + bf2f(shared[(size_t)n * lds_ + c]));
    if (resid) acc = rbf(bf2f(resid[(size_t)n * ldr + c]) + acc);
    out[(size_t)n * ldo + c] = f2bf(acc);
  }
}

}  // namespace

extern "C" {

int ohara_moe_route_topk(const uint16_t* router_logits, int ldl, const uint16_t* router_bias, int n_tokens, int n_experts,
                         int k, int biased_topk, int gate_sigmoid, int normalize, int32_t* expert_idx,
                         uint16_t* expert_w, void* stream) {
  if (!router_logits || !expert_idx || !expert_w || n_tokens < 1 || n_experts < 1 || k < 1) return OHARA_EINVAL;
  if (k > 16 || n_experts > 1024 || k > n_experts || ldl < n_experts) return OHARA_ESIZE;
  if (biased_topk && !router_bias) return OHARA_EINVAL;
  const dim3 grid((n_tokens + 3) / 4), block(256);
#define OHARA_ROUTE(PL_)                                                                                            \
  hipLaunchKernelGGL(moe_route_kernel<PL_>, grid, block, 0, (hipStream_t)stream, router_logits, ldl, router_bias, \
                     n_tokens, n_experts, k, biased_topk, gate_sigmoid, normalize, expert_idx, expert_w)
  if (n_experts <= 64) OHARA_ROUTE(1);
  else if (n_experts <= 256) OHARA_ROUTE(4);
  else OHARA_ROUTE(16);
#undef OHARA_ROUTE
  return ohara_launch_status();
}

int ohara_moe_route_fused(const uint16_t* x, int ldx, const uint16_t* norm_w, float eps, const uint16_t* router_wp,
                          const uint16_t* router_bias, int n_tokens, int d, int n_experts, int k, int biased_topk,
                          int gate_sigmoid, int normalize, uint16_t* x_norm, int ld_x_norm, uint16_t* router_logits, int ldl,
                          int32_t* expert_idx, uint16_t* expert_w, int32_t* offsets, int32_t* pair_of, int32_t* pos_of,
                          int32_t* counter, void* stream) {
  if (!x || !norm_w || !router_wp || !x_norm || !expert_idx || !expert_w || !offsets || !pair_of || !pos_of || !counter)
    return OHARA_EINVAL;
  if (n_tokens < 1 || d < 8 || (d & 7) || (ldx & 7) || (ld_x_norm & 7) || k < 1 || n_experts < 1) return OHARA_EINVAL;
  if (n_experts > 64 || k > 16 || k > n_experts || (int64_t)n_tokens * k > 1024 || d > 4096) return OHARA_ESIZE;
  if (biased_topk && !router_bias) return OHARA_EINVAL;
  if (router_logits && ldl < n_experts) return OHARA_EINVAL;
  RouteFusedArgs a{};
  a.x = x; a.ldx = ldx; a.norm_w = norm_w; a.eps = eps; a.wp = reinterpret_cast<const uint4*>(router_wp); a.bias = router_bias;
  a.N = n_tokens; a.d = d; a.E = n_experts; a.k = k; a.biased = biased_topk; a.sigmoid = gate_sigmoid; a.normalize = normalize;
  a.xn = x_norm; a.ldxn = ld_x_norm; a.logits = router_logits; a.ldl = ldl; a.idx = expert_idx; a.w = expert_w;
  a.offs = offsets; a.pair_of = pair_of; a.pos_of = pos_of; a.counter = counter;
  const size_t smem = (size_t)4 * (((d + 31) / 32) * 32 + 8) * sizeof(bf16_t);
  hipLaunchKernelGGL(moe_route_fused_kernel, dim3((n_tokens + 3) / 4), dim3(256), smem, (hipStream_t)stream, a);
  return ohara_launch_status();
}

int ohara_moe_sort_pairs(const int32_t* expert_idx, int n_pairs, int n_experts, int32_t* offsets, int32_t* pair_of,
                         int32_t* pos_of, void* stream) {
  if (!expert_idx || !offsets || !pair_of || !pos_of || n_pairs < 1 || n_experts < 1) return OHARA_EINVAL;
  if (n_pairs > 65536 || n_experts > 1024) return OHARA_ESIZE;
  if (n_experts <= 64 && n_pairs <= 1024)
    hipLaunchKernelGGL(moe_sort_small_kernel, dim3(1), dim3(1024), 0, (hipStream_t)stream, expert_idx, n_pairs, n_experts,
                       offsets, pair_of, pos_of);
  else {
    const size_t lds = (size_t)16 * n_experts * sizeof(int);
    if (lds > 48 * 1024) (void)hipFuncSetAttribute((const void*)moe_place_kernel<false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL(moe_place_kernel<false>, dim3((n_pairs + 1023) / 1024), dim3(1024), lds, (hipStream_t)stream, expert_idx, n_pairs,
                       n_experts, nullptr, offsets, pair_of, pos_of);
  }
  return ohara_launch_status();
}

int ohara_moe_experts_gate_up_shared(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                                     int n_experts, int hidden, int d, int k, const int32_t* offsets,
                                     const int32_t* pair_of, uint16_t* act, int ld_act, const uint16_t* wp_shared,
                                     int shared_hidden, int n_tokens, uint16_t* act_shared, int ld_act_shared,
                                     void* stream) {
  if (!x || !wp_gate_up || !offsets || !pair_of || !act || hidden < 1 || d < 1 || (d & 7) || (ldx & 7)) return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp_gate_up); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = x; a.ldx = ldx; a.offs = offsets; a.pair_of = pair_of; a.k = k; a.N_out = hidden; a.K = d;
  a.out = act; a.ldo = ld_act; a.E = n_experts;
  int strips = 2 * ((hidden + 7) / 8 * 8) / 16;
  int rows = n_experts;
  if (wp_shared) {  // the shared expert: a row of the grid per 16 tokens
    if (!act_shared || n_tokens < 1 || shared_hidden < 1 || ld_act_shared < shared_hidden) return OHARA_EINVAL;
    a.N_sh = n_tokens; a.wp_sh = reinterpret_cast<const uint4*>(wp_shared); a.x_sh = x; a.ldx_sh = ldx;
    a.N_out_sh = shared_hidden; a.K_sh = d; a.out_sh = act_shared; a.ldo_sh = ld_act_shared;
    const int s2 = 2 * ((shared_hidden + 7) / 8 * 8) / 16;
    strips = strips > s2 ? strips : s2;
    rows += (n_tokens + 15) / 16;
  }
  if ((d + 31) / 32 <= 16)
    hipLaunchKernelGGL((moe_expert_kernel<X_SWIGLU, 4>), dim3(strips, rows), dim3(256), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL((moe_expert_kernel<X_SWIGLU, 8>), dim3(strips, rows), dim3(256), 0, (hipStream_t)stream, a);
  return ohara_launch_status();
}

int ohara_moe_experts_gate_up(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                              int n_experts, int hidden, int d, int k, const int32_t* offsets, const int32_t* pair_of,
                              uint16_t* act, int ld_act, void* stream) {
  return ohara_moe_experts_gate_up_shared(x, ldx, wp_gate_up, expert_stride_bytes, n_experts, hidden, d, k, offsets, pair_of,
                                          act, ld_act, nullptr, 0, 0, nullptr, 0, stream);
}

int ohara_moe_experts_down_shared(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes,
                                  int n_experts, int d, int hidden, int k, const int32_t* offsets, const int32_t* pair_of,
                                  const uint16_t* expert_w, uint16_t* y, int ldy, const uint16_t* wp_shared,
                                  int shared_hidden, int n_tokens, const uint16_t* act_shared, int ld_act_shared,
                                  uint16_t* y_shared, int ldy_shared, void* stream) {
  if (!act || !wp_down || !offsets || !pair_of || !expert_w || !y || hidden < 1 || d < 1 || (hidden & 7) || (ld_act & 7))
    return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp_down); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = act; a.ldx = ld_act; a.offs = offsets; a.pair_of = pair_of; a.w = expert_w; a.k = k; a.N_out = d; a.K = hidden;
  a.out = y; a.ldo = ldy; a.E = n_experts;
  int rows = n_experts, ks = (hidden + 31) / 32;
  if (wp_shared) {  // the shared expert: a row of the grid per 16 tokens
    if (!act_shared || !y_shared || n_tokens < 1 || shared_hidden < 1 || (shared_hidden & 7) || (ld_act_shared & 7))
      return OHARA_EINVAL;
    a.N_sh = n_tokens; a.wp_sh = reinterpret_cast<const uint4*>(wp_shared); a.x_sh = act_shared; a.ldx_sh = ld_act_shared;
    a.N_out_sh = d; a.K_sh = shared_hidden; a.out_sh = y_shared; a.ldo_sh = ldy_shared;
    const int ks2 = (shared_hidden + 31) / 32;
    ks = ks > ks2 ? ks : ks2;
    rows += (n_tokens + 15) / 16;
  }
  if (ks <= 16)
    hipLaunchKernelGGL((moe_expert_kernel<X_DOWN, 4>), dim3((d + 15) / 16, rows), dim3(256), 0, (hipStream_t)stream, a);
  else
    hipLaunchKernelGGL((moe_expert_kernel<X_DOWN, 8>), dim3((d + 15) / 16, rows), dim3(256), 0, (hipStream_t)stream, a);
  return ohara_launch_status();
}

int ohara_moe_experts_down(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes,
                           int n_experts, int d, int hidden, int k, const int32_t* offsets, const int32_t* pair_of,
                           const uint16_t* expert_w, uint16_t* y, int ldy, void* stream) {
  return ohara_moe_experts_down_shared(act, ld_act, wp_down, expert_stride_bytes, n_experts, d, hidden, k, offsets, pair_of,
                                       expert_w, y, ldy, nullptr, 0, 0, nullptr, 0, nullptr, 0, stream);
}

int ohara_moe_experts_gate_up_many(const uint16_t* x, int ldx, const uint16_t* wp_gate_up, int64_t expert_stride_bytes,
                                   int n_experts, int hidden, int d, int k, int n_pairs, const int32_t* offsets,
                                   const int32_t* pair_of, uint16_t* act, int ld_act, void* stream) {
  if (!x || !wp_gate_up || !offsets || !pair_of || !act || n_experts < 1 || k < 1 || n_pairs < 1) return OHARA_EINVAL;
  if (hidden < 1 || d < 8 || ((d | ldx) & 7) || ldx < d || ld_act < hidden) return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp_gate_up); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = x; a.ldx = ldx; a.offs = offsets; a.pair_of = pair_of; a.k = k; a.N_out = hidden; a.K = d;
  a.out = act; a.ldo = ld_act; a.E = n_experts;
  return launch_experts<X_SWIGLU>(a, n_pairs, 0, (hipStream_t)stream);
}

int ohara_moe_experts_down_many(const uint16_t* act, int ld_act, const uint16_t* wp_down, int64_t expert_stride_bytes, int n_experts,
                                int d, int hidden, int k, int n_pairs, const int32_t* offsets, const int32_t* pair_of,
                                const uint16_t* expert_w, uint16_t* y, int ldy, void* stream) {
  if (!act || !wp_down || !offsets || !pair_of || !expert_w || !y || n_experts < 1 || k < 1 || n_pairs < 1) return OHARA_EINVAL;
  if (hidden < 8 || d < 1 || ((hidden | ld_act) & 7) || ld_act < hidden || ldy < d) return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp_down); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = act; a.ldx = ld_act; a.offs = offsets; a.pair_of = pair_of; a.w = expert_w; a.k = k; a.N_out = d; a.K = hidden;
  a.out = y; a.ldo = ldy; a.E = n_experts;
  return launch_experts<X_DOWN>(a, n_pairs, 0, (hipStream_t)stream);
}

int ohara_moe_combine(const uint16_t* y, int ldy, const int32_t* expert_idx, const int32_t* pos_of, int n_tokens, int k,
                      const uint16_t* shared, int ld_shared, const uint16_t* resid, int ldr, uint16_t* out, int ldo, int d,
                      void* stream) {
  if (!y || !expert_idx || !pos_of || !out || n_tokens < 1 || k < 1 || k > 16 || d < 1) return OHARA_EINVAL;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(n_tokens), dim3(256), 0, (hipStream_t)stream, y, ldy, expert_idx, pos_of, k,
                     shared, ld_shared, resid, ldr, out, ldo, d);
  return ohara_launch_status();
}

int ohara_moe_router_bf16(const uint16_t* x, int ldx, const uint16_t* w, int ldw, const float* correction, int rows, int k, int n_out,
                          int top, int groups, int keep, int flags, int32_t* idx, float* wgt, int32_t* offs, int32_t* pair_of,
                          int32_t* pos_of, int32_t* hist, int32_t* counter, void* stream) {
  return launch_router<bf16_t>(RouterArgs<bf16_t>{x, w, correction, ldx, ldw, rows, k, n_out, top, groups, keep, idx, wgt, offs,
                                                  pair_of, pos_of, counter, flags, 0}, hist, (hipStream_t)stream);
}
int ohara_moe_router_f32(const float* x, int ldx, const float* w, int ldw, const float* correction, int rows, int k, int n_out,
                         int top, int groups, int keep, int flags, int32_t* idx, float* wgt, int32_t* offs, int32_t* pair_of,
                         int32_t* pos_of, int32_t* hist, int32_t* counter, void* stream) {
  return launch_router<float>(RouterArgs<float>{x, w, correction, ldx, ldw, rows, k, n_out, top, groups, keep, idx, wgt, offs,
                                                pair_of, pos_of, counter, flags, 0}, hist, (hipStream_t)stream);
}

int ohara_moe_glu_bf16(const uint16_t* x, int ldx, const uint16_t* wp, int64_t expert_stride_bytes, int n_experts, int hidden, int d,
                       int top, int n_pairs, const int32_t* offs, const int32_t* pair_of, const float* pair_w, const OharaGlu* glu, uint16_t* act,
                       int ld_act, const uint16_t* wp_shared, int hidden_shared, int n_tokens, const OharaGlu* glu_shared,
                       uint16_t* act_shared, int ld_act_shared, void* stream) {
  if (!x || !wp || !offs || !pair_of || !glu || !act || n_experts < 1 || top < 1 || n_pairs < 1) return OHARA_EINVAL;
  if (d < 8 || hidden < 8 || ((d | hidden | ldx | ld_act) & 7) || ldx < d || ld_act < hidden) return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = x; a.ldx = ldx; a.offs = offs; a.pair_of = pair_of; a.k = top; a.N_out = hidden; a.K = d;
  a.out = act; a.ldo = ld_act; a.E = n_experts; a.glu = *glu; a.pair_w = pair_w;
  int n_sh = 0;
  if (wp_shared) {
    if (!act_shared || !glu_shared || n_tokens < 1 || hidden_shared < 8 || (hidden_shared & 7) || ld_act_shared < hidden_shared)
      return OHARA_EINVAL;
    a.N_sh = n_sh = n_tokens; a.wp_sh = reinterpret_cast<const uint4*>(wp_shared); a.x_sh = x; a.ldx_sh = ldx;
    a.N_out_sh = hidden_shared; a.K_sh = d; a.out_sh = act_shared; a.ldo_sh = ld_act_shared; a.glu_sh = *glu_shared;
  }
  return launch_experts<X_GLU>(a, n_pairs, n_sh, (hipStream_t)stream);
}

int ohara_moe_down_bf16(const uint16_t* act, int ld_act, const uint16_t* wp, int64_t expert_stride_bytes, int n_experts, int d,
                        int hidden, int n_pairs, const int32_t* offs, uint16_t* y, int ldy, const uint16_t* wp_shared,
                        int hidden_shared, int n_tokens, const uint16_t* act_shared, int ld_act_shared, uint16_t* y_shared,
                        int ldy_shared, void* stream) {
  if (!act || !wp || !offs || !y || n_experts < 1 || n_pairs < 1) return OHARA_EINVAL;
  if (d < 8 || hidden < 8 || ((d | hidden | ld_act) & 7) || (ldy & 3) || ld_act < hidden || ldy < d) return OHARA_EINVAL;
  ExpertArgs a{};
  a.wp = reinterpret_cast<const uint4*>(wp); a.expert_stride = (size_t)expert_stride_bytes / 16;
  a.x = act; a.ldx = ld_act; a.offs = offs; a.k = 1; a.N_out = d; a.K = hidden; a.out = y; a.ldo = ldy; a.E = n_experts;
  int n_sh = 0;
  if (wp_shared) {
    if (!act_shared || !y_shared || n_tokens < 1 || hidden_shared < 8 || ((hidden_shared | ld_act_shared) & 7) ||
        ld_act_shared < hidden_shared || ldy_shared < d)
      return OHARA_EINVAL;
    a.N_sh = n_sh = n_tokens; a.wp_sh = reinterpret_cast<const uint4*>(wp_shared); a.x_sh = act_shared; a.ldx_sh = ld_act_shared;
    a.N_out_sh = d; a.K_sh = hidden_shared; a.out_sh = y_shared; a.ldo_sh = ldy_shared;
  }
  return launch_experts<X_RAW>(a, n_pairs, n_sh, (hipStream_t)stream);
}

}  // extern "C"
