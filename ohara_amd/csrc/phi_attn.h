// Phi's attention of single tokens over the cache (ohara/models/phi.py:98-117, rotary.py:131-184), as a kernel of its own (phi.hip) and beside a product's
// workgroups (gemm_skinny.hip).
#pragma once
#include "gemm_epilogue.h"

// ---- attention ---------------------------------------------------------------------------
// Four waves - a team - per (sequence, head, new token) and context chunk; a workgroup is a team or several.  Sixteen lanes own one cached
// position at a time (lane l the eight features 8l .. 8l+7) and fetch two positions per round before
// using either (four measured slower: 178 registers halve the occupancy), so a team walks 32
// positions per round with an online softmax per 16-lane group;
// the groups are merged through LDS at the end.  With several chunks (decode: few queries, long
// context) every chunk leaves {weighted sum, max, sum} and the team that finishes last combines
// them in chunk order.
// What bounds it: for few rows a chain of round trips - the query and its angles, two rounds of positions, the chunks' sums to memory, their
// counter, and back; for many the arithmetic of a position, sixteen lanes' weights and two exponentials.  So the first round's positions are asked for
// with the query, a chunk holds 64 positions at least (32: behind 40 7.7 instead of 5.4, 700 11.5 instead of 10.7), the live chunks are dealt over all
// XCDs, and a feature that is not rotated has its weight as the addend of one that is.  32 heads of 80, us before / now: one row behind 40 10.0 / 5.4,
// 200 10.4 / 9.0, 700 11.9 / 10.7, 2040 15.3 / 14.1; 16 rows behind 700 38.2 / 36.1, 2040 93.2 / 83.8.  (Three positions in flight: 700 10.9.)
//
// The reference rotates every cached key again at each step (phi.py:104).  With the rotated query
// qr and c, s the cosine / sine of key position t the score is
//   sum_i (k1_i c_i - k2_i s_i) qr1_i + (k1_i s_i + k2_i c_i) qr2_i + sum_rest k_j q_j
//     = sum_i k1_i (c_i qr1_i + s_i qr2_i) + k2_i (c_i qr2_i - s_i qr1_i) + sum_rest k_j q_j,
// i.e. a dot product of the raw key row with a per-position weight vector built from two per-lane
// constants A, B: w_j = c A_j + s B_j.  All of it in fp32, as the reference (phi.py:98-100).
struct PhiAttnArgs {
  const bf16_t* q;
  int ldq;
  const bf16_t* kc;
  const bf16_t* vc;
  const float* cos;  // (t_max, rot/2) fp32
  const float* sin;
  bf16_t* out;       // (rows, H*D)
  int B, S, H, D, rot, t_max, pos;
  const int32_t* pos_dev;
  int ns;         // context chunks at most (decode)
  float* ws;      // ns > 1: per (row, head, chunk) D + 2 floats {weighted sum[D], max, sum}
  int* counters;  // ns > 1: per (row, head) chunks finished; zero between calls
};

// What the calls below are refused for, and the arguments.
inline int phi_attn_args(PhiAttnArgs& a, const uint16_t* q, int ldq, const uint16_t* kcache, const uint16_t* vcache, const float* cos, const float* sin,
                         int rot, int batch, int seq_len, int h, int dh, int t_max, int pos, const int32_t* pos_dev, int n_split, void* workspace,
                         uint16_t* out) {
  if (!q || !kcache || !vcache || !cos || !sin || !out) return OHARA_EINVAL;
  if (batch < 1 || seq_len < 1 || h < 1 || t_max < 1) return OHARA_EINVAL;
  if (dh < 8 || dh > 128 || (dh & 7)) return OHARA_ESIZE;
  if (rot < 2 || (rot & 1) || rot > dh) return OHARA_EINVAL;  // rotary.py:118-121
  if (ldq < h * dh) return OHARA_EINVAL;
  if (!pos_dev && (pos < 0 || pos + seq_len > t_max)) return OHARA_EINVAL;
  if (pos_dev && seq_len != 1) return OHARA_EINVAL;
  if (n_split < 1 || n_split > 64 || (n_split > 1 && (!workspace || seq_len != 1))) return OHARA_EINVAL;
  if ((int64_t)batch * seq_len * h * n_split > INT32_MAX) return OHARA_ESIZE;
  const size_t counters = (((size_t)batch * h * sizeof(int)) + 255) & ~(size_t)255;
  a = PhiAttnArgs{q, ldq, kcache, vcache, cos, sin, out, batch, seq_len, h, dh, rot, t_max, pos, pos_dev, n_split,
                  reinterpret_cast<float*>(reinterpret_cast<char*>(workspace) + counters), reinterpret_cast<int*>(workspace)};
  return OHARA_OK;
}

// A lane's eight features lie in one half of the rotated ones, or behind them, and their angles on 16 bytes.
inline bool phi_eights(const PhiAttnArgs& a) { return ((a.rot >> 1) & 7) == 0 && (((uintptr_t)a.cos | (uintptr_t)a.sin) & 15) == 0; }

// Positions of a chunk where there are ns of them, the query at `pos`: whole rounds, of 64 at least.
__host__ __device__ inline int phi_chunk(int pos, int ns) {
  const int per = (pos + ns) / ns;
  return ((per < 64 ? 64 : per) + 15) & ~15;
}

// gemm_skinny.hip: the attention beside y = x W^T + bias in one launch, where that is the quicker way (else false, and nothing is launched).
bool ohara_launch_phi_attn_linear(PhiAttnArgs t, GemmArgs a, hipStream_t st, int* rc);
// The attention's chunks left in t.ws, beside the product or before it; then out = merged W^T + bias, added as EPI_BIAS_ADD2 adds.
int ohara_launch_phi_attn_out(PhiAttnArgs t, GemmArgs a, GemmArgs out, hipStream_t st);

namespace {

// Where a maximum of scores begins, the lowest finite number: a score of minus infinity then has the weight zero, as what came before a finite score has, and
// nothing has to be left out where sums are merged - what saw no position adds zeros, a score that is not a number its NaN.  (From minus infinity on, a group
// of lanes whose scores are all NaN, which a maximum ignores, looks like one that saw no position.)  The merges' products are rounded by themselves, in all kernels.
constexpr float PHI_LOWEST = -__FLT_MAX__;

// Where the sums of four chunks go that the next launch merges (phi_dense_kernel): values on 16 bytes, then {max, sum}.  a.ns is a multiple of four.
__device__ __forceinline__ float* phi_values(const PhiAttnArgs& a, int row, int h) { return a.ws + ((size_t)row * a.H + h) * (a.ns >> 2) * a.D; }
__device__ __forceinline__ float* phi_pairs(const PhiAttnArgs& a, int row, int h) {
  return a.ws + (size_t)a.B * a.H * (a.ns >> 2) * a.D + ((size_t)row * a.H + h) * (a.ns >> 2) * 2;
}

// `block`: the workgroup's place among those that do this.  PARTS: one token a sequence; a workgroup's teams take four chunks
// in turn of one head, and leave their sums together.
template <int TEAMS, bool EIGHTS, bool PARTS = false>
__device__ __forceinline__ void phi_attend(const PhiAttnArgs& a, int block) {
  constexpr int R = 2;  // positions a lane group has in flight
  __shared__ float qr_[TEAMS][128];
  __shared__ float gm_[TEAMS][16], gl_[TEAMS][16];
  __shared__ float gacc_[TEAMS][16][128];
  __shared__ float teams_m[TEAMS], teams_l[TEAMS];
  const int team = TEAMS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), tid = TEAMS == 1 ? threadIdx.x : threadIdx.x & 255;
  const int lane = tid & 63, wave = tid >> 6;
  float(&qr)[128] = qr_[team];
  float(&gm)[16] = gm_[team];
  float(&gl)[16] = gl_[team];
  float(&gacc)[16][128] = gacc_[team];
  const int grp = wave * 4 + (lane >> 4), l = lane & 15;
  const int D = a.D, half = a.rot >> 1;
  // The cache is position-major: the heads of one position lie side by side, 2 * D bytes each, so the rows of
  // neighbouring heads share 128-byte lines.  Workgroups are handed to the eight XCDs in turn, each with an L2 of
  // its own: taken as launched, neighbouring heads would land on different XCDs and every L2 would fetch the
  // shared lines again.  So the launch order is re-read: XCD x works through the x-th eighth of the (chunk,
  // sequence, head) list, heads fastest.  (Any bijection is correct; this one needs a number of live teams
  // that is eight times whole workgroups, otherwise the order stays as launched.)
  const int pos = a.pos_dev ? *a.pos_dev : a.pos;
  int per = 0, ns = 1;  // positions of a chunk; chunks (they belong to calls of one token a sequence)
  if (a.ns > 1) {
    per = phi_chunk(max(pos, 0), a.ns);
    ns = max(pos, 0) / per + 1;
  }
  static_assert(!PARTS || TEAMS == 4, "");
  constexpr int APART = PARTS ? 1 : TEAMS;  // ids of a workgroup
  const int rows = a.B * a.S * a.H, n = rows * (PARTS ? (ns + 3) >> 2 : ns);
  int id = block * APART + (PARTS ? 0 : team);
  bool there = id < n;  // (the other teams of a workgroup come along to its barriers)
  if ((n & (8 * APART - 1)) == 0) {
    const int share = n >> 3, mine = (block >> 3) * APART + (PARTS ? 0 : team);
    there = mine < share;
    id = (block & 7) * share + mine;
  }
  id = there ? id : 0;
  int by = id / rows;
  int w = id - by * rows;
  if (PARTS) {
    if (!there) return;  // (the whole workgroup)
    by = 4 * by + team;
    there = by < ns;
  }
  const int s = w % a.S; w /= a.S;
  const int h = w % a.H;
  const int seq = w / a.H;
  const int row = seq * a.S + s;
  const int pq = pos + s;  // position of this query; keys 0 .. pq are visible
  const bool live = there && pq >= 0 && pq < a.t_max;
  if (TEAMS == 1 && !live) return;
  const int t_lo = live ? by * per : 0, t_hi = !live ? -1 : ns > 1 ? min(pq, t_lo + per - 1) : pq;  // this team's positions

  const int e0 = 8 * l;
  const bool own = e0 < D;
  // Lanes beyond the head (own == false) read the head's first features instead: their weights A / Bc are
  // zero, so what they read only has to be mapped memory.
  const int e0c = own ? e0 : 0;
  const size_t hd = (size_t)a.H * D;
  const bf16_t* kb = a.kc + (size_t)seq * a.t_max * hd + (size_t)h * D + e0c;
  const bf16_t* vb = a.vc + (size_t)seq * a.t_max * hd + (size_t)h * D + e0c;
  const bool rotates = own && e0 < a.rot;
  const int fc = rotates ? (e0 < half ? e0 : e0 - half) : 0;  // EIGHTS: the first of this lane's angles
  uint4 kv[R], vv[R];
  float cs[R][8], sn[R][8];
  // every load of a round is issued whatever its position (clamped to the chunk's last one): one run
  // of loads without branches; a position past the end is skipped when the round is consumed
  auto fetch = [&](int t) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int tt = max(min(t + 16 * r, t_hi), 0);
      kv[r] = ldg16(kb + (size_t)tt * hd);
      vv[r] = ldg16(vb + (size_t)tt * hd);
      if (EIGHTS) {
        // the lane's eight angles are eight adjacent table entries (asking for those of rotated features only takes as long)
        const float* cp = a.cos + (size_t)tt * half + fc;
        const float* sp = a.sin + (size_t)tt * half + fc;
        const uint4 c0 = ldg16(cp), c1 = ldg16(cp + 4), s0 = ldg16(sp), s1 = ldg16(sp + 4);
        const uint32_t cu[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const uint32_t su[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          cs[r][u] = __uint_as_float(cu[u]);
          sn[r][u] = __uint_as_float(su[u]);
        }
      } else {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int j = e0 + u;
          // (pieces of 4 bytes: asked for only where there is a position, 32 rows of 32 heads of 80, 40 rotated, behind 0 10.1 -> 7.6 us, 5 10.3 -> 7.8)
          const bool rot_u = own && j < a.rot && t + 16 * r <= t_hi;
          const int f = j < half ? j : j - half;
          cs[r][u] = rot_u ? a.cos[(size_t)tt * half + f] : 1.0f;
          sn[r][u] = rot_u ? a.sin[(size_t)tt * half + f] : 0.0f;
        }
      }
    }
  };
  // the query's row and angles, then the first round: they come back in order
  float q0 = 0.f, q1 = 0.f, qc = 1.f, qs = 0.f;
  if (tid < D) {
    const bf16_t* qrow = a.q + (size_t)row * a.ldq + h * D;
    const int i = tid < half ? tid : tid - half;
    q0 = bf2f(qrow[tid]);
    if (tid < a.rot) {
      const size_t at = (size_t)min(max(pq, 0), a.t_max - 1) * half + i;
      q1 = bf2f(qrow[tid < half ? tid + half : i]);
      qc = a.cos[at];
      qs = a.sin[at];
    }
  }
  fetch(t_lo + grp);
  __builtin_amdgcn_sched_barrier(0);
  if (tid < D) qr[tid] = tid < half ? q0 * qc - q1 * qs : tid < a.rot ? q1 * qs + q0 * qc : q0;
  __syncthreads();

  float A[8], Bc[8], fixed[8];  // a feature's weight is cos A + sin B + fixed: the last where EIGHTS are not rotated
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const int j = e0 + u;
    A[u] = own && !(EIGHTS && !rotates) ? qr[j] : 0.f;
    Bc[u] = own && j < half ? qr[j + half] : own && j < a.rot ? -qr[j - half] : 0.f;
    fixed[u] = own && EIGHTS && !rotates ? qr[j] : 0.f;
  }
  const float scale = sqrtf(1.0f / (float)D);

  float m = PHI_LOWEST, lsum = 0.f, acc[8];
#pragma unroll
  for (int u = 0; u < 8; ++u) acc[u] = 0.f;
  for (int t = t_lo + grp; t <= t_hi;) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (t + 16 * r > t_hi) break;  // uniform within the 16-lane group
      const uint32_t ku[4] = {kv[r].x, kv[r].y, kv[r].z, kv[r].w};
      float part = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float w0 = EIGHTS ? __builtin_fmaf(sn[r][2 * i], Bc[2 * i], __builtin_fmaf(cs[r][2 * i], A[2 * i], fixed[2 * i]))
                                : cs[r][2 * i] * A[2 * i] + sn[r][2 * i] * Bc[2 * i];
        const float w1 = EIGHTS ? __builtin_fmaf(sn[r][2 * i + 1], Bc[2 * i + 1], __builtin_fmaf(cs[r][2 * i + 1], A[2 * i + 1], fixed[2 * i + 1]))
                                : cs[r][2 * i + 1] * A[2 * i + 1] + sn[r][2 * i + 1] * Bc[2 * i + 1];
        part += lo_bf(ku[i]) * w0;
        part += hi_bf(ku[i]) * w1;
      }
      part = lane_xor_sum<8>(lane_xor_sum<4>(lane_xor_sum<2>(lane_xor_sum<1>(part))));
      const float sc = part * scale;
      const float mn = fmaxf(m, sc);
      // hardware exponential: its error (about 1e-6 relative) is far below the bf16 rounding of the output
      const float corr = __expf(m - mn), p = __expf(sc - mn);
      lsum = lsum * corr + p;
      const uint32_t vu[4] = {vv[r].x, vv[r].y, vv[r].z, vv[r].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc[2 * i] = acc[2 * i] * corr + p * lo_bf(vu[i]);
        acc[2 * i + 1] = acc[2 * i + 1] * corr + p * hi_bf(vu[i]);
      }
      m = mn;
    }
    t += 16 * R;
    if (t <= t_hi) fetch(t);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (l == 0) {
    gm[grp] = m;
    gl[grp] = lsum;
  }
  if (own) {
#pragma unroll
    for (int u = 0; u < 8; ++u) gacc[grp][e0 + u] = acc[u];
  }
  __syncthreads();
  if ((PARTS || live) && tid < D) {
    float M = PHI_LOWEST, gv[16];
#pragma unroll
    for (int g = 0; g < 16; ++g) gv[g] = gacc[g][tid];
#pragma unroll
    for (int g = 0; g < 16; ++g) M = fmaxf(M, gm[g]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int g = 0; g < 16; ++g) {  // (no branch: every read would be waited for behind it; with the merge's below, whose values are asked for
                                    // with the maxima: 32 heads of 80 behind 700 13.1 -> 11.2 us)
#pragma clang fp contract(off)
      const float wg = expf(gm[g] - M);
      num += wg * gv[g];
      den += wg * gl[g];
    }
    if (PARTS) {
      gacc[0][tid] = num;  // (this thread's column)
      if (tid == 0) {
        teams_m[team] = M;
        teams_l[team] = den;
      }
    } else if (ns > 1) {
      // write-through stores: the workgroup that merges may sit on another XCD
      float* o = a.ws + (((size_t)row * a.H + h) * a.ns + by) * (D + 2);
      st_coh4(o + tid, __float_as_uint(num));
      if (tid == 0) {
        st_coh4(o + D, __float_as_uint(M));
        st_coh4(o + D + 1, __float_as_uint(den));
      }
    } else {
      a.out[(size_t)row * hd + (size_t)h * D + tid] = f2bf(num / den);
    }
  }
  if (PARTS) {
    __syncthreads();
    if (team || tid >= D) return;
    float M = PHI_LOWEST, num = 0.f, den = 0.f;
#pragma unroll
    for (int i = 0; i < TEAMS; ++i) M = fmaxf(M, teams_m[i]);
#pragma unroll
    for (int i = 0; i < TEAMS; ++i) {
#pragma clang fp contract(off)
      const float wg = expf(teams_m[i] - M);
      num += wg * gacc_[i][0][tid];
      den += wg * teams_l[i];
    }
    phi_values(a, row, h)[(by >> 2) * D + tid] = num;
    if (tid == 0) *reinterpret_cast<float2*>(phi_pairs(a, row, h) + 2 * (by >> 2)) = make_float2(M, den);
    return;
  }
  if (TEAMS == 1 ? ns == 1 : a.ns == 1) return;

  // The team that finishes last merges the chunks of its (row, head), in chunk order.  Every
  // wave waits for its own write-through stores before the workgroup barrier; the counter is a
  // relaxed device-scope atomic; the merge reads with cache-bypassing loads.
  __shared__ int last_[TEAMS];
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  wait_own_stores();
  __syncthreads();
  int* counter = a.counters + (size_t)row * a.H + h;
  if (tid == 0) last_[team] = 0;
  if (tid == 0 && live && ns > 1) {
    const int old = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last_[team] = old == ns - 1;
    if (old == ns - 1) __hip_atomic_store(counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next call
  }
  __syncthreads();
  const bool last = last_[team];
  if (TEAMS == 1 && !last) return;
  const float* p = a.ws + ((size_t)row * a.H + h) * a.ns * (D + 2);
  // at most 64: one round of loads for all (max, sum) pairs and the first sixteen chunks' values
  float av[16];
  if (last && tid < D) {
#pragma unroll
    for (int i = 0; i < 16; ++i) av[i] = __uint_as_float(ld_coh4(p + (size_t)min(i, ns - 1) * (D + 2) + tid));
  }
  if (last && tid < ns) {
    // qr and gacc are free again: chunk maxima and sums go there
    qr[tid] = __uint_as_float(ld_coh4(p + (size_t)tid * (D + 2) + D));
    gacc[0][tid] = __uint_as_float(ld_coh4(p + (size_t)tid * (D + 2) + D + 1));
  }
  __syncthreads();
  if (last && tid < D) {
    float M = PHI_LOWEST;
    for (int c = 0; c < ns; ++c) M = fmaxf(M, qr[c]);
    float num = 0.f, den = 0.f;
    for (int c0 = 0; c0 < ns; c0 += 16) {  // sixteen chunks' values in flight, every load unconditional
      if (c0) {
#pragma unroll
        for (int i = 0; i < 16; ++i) av[i] = __uint_as_float(ld_coh4(p + (size_t)min(c0 + i, ns - 1) * (D + 2) + tid));
        __builtin_amdgcn_sched_barrier(0);
      }
      float mc[16], lc[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        mc[i] = qr[min(c0 + i, ns - 1)];
        lc[i] = gacc[0][min(c0 + i, ns - 1)];
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
#pragma clang fp contract(off)
        const bool in = c0 + i < ns;
        const float wg = expf(mc[i] - M);
        num += in ? wg * av[i] : 0.f;
        den += in ? wg * lc[i] : 0.f;
      }
    }
    a.out[(size_t)row * hd + (size_t)h * D + tid] = f2bf(num / den);
  }
}

}  // namespace
